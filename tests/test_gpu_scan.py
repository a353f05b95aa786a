"""The scans at the edges of their tiles (2,048 counts) and of the two ways of
summing the tiles, and the offsets of a view's rays."""
import ctypes

import pytest
import torch

from nsvf_amd._lib import lib

pytestmark = pytest.mark.gpu
_p = lambda x: ctypes.c_void_p(x.data_ptr())
SIZES = [1, 2047, 2048, 2049, 300_000, 4096 * 2048, 4096 * 2048 + 1]


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("alias", [False, True])
def test_scan(device, n, alias):
    g = torch.Generator().manual_seed(n)
    a = torch.randint(0, 100, (n,), generator=g, dtype=torch.int32).to(device)
    want = torch.cumsum(a, 0, dtype=torch.int32)
    src = a.clone()
    out = src if alias else torch.full_like(a, -1)
    ws = torch.empty(int(lib().nsvf_scan_workspace_ints(n)), dtype=torch.int32, device=device)
    total = torch.full((1,), -1, dtype=torch.int32, device=device)
    assert lib().nsvf_scan_exclusive_i32(_p(src), _p(out), n, _p(ws), _p(total), None) == 0
    torch.cuda.synchronize()
    assert torch.equal(out, want - a) and int(total) == int(want[-1])


@pytest.mark.parametrize("R", [0] + SIZES[:5] + [600_001])
def test_render_offsets(device, R):
    g = torch.Generator().manual_seed(R)
    flag = (torch.rand(R, generator=g) < 0.4).int().to(device)
    bound = torch.randint(0, 200, (R,), generator=g, dtype=torch.int32).to(device) * flag
    rank, lst, off, zero = (torch.full((R,), -1, dtype=torch.int32, device=device)
                            for _ in range(4))
    scal = torch.full((9,), -1, dtype=torch.int32, device=device)
    ws = torch.empty(int(lib().nsvf_render_offsets_workspace_ints(R)) + 1, dtype=torch.int32,
                     device=device)
    assert lib().nsvf_render_offsets(_p(flag), _p(bound), R, _p(rank), _p(lst), _p(off), _p(zero),
                                     _p(scal), 8, _p(ws), None) == 0
    torch.cuda.synchronize()
    n = int(flag.sum())
    assert scal.tolist() == [n, int(bound.sum())] + [0] * 6 + [-1]
    assert torch.equal(rank, (torch.cumsum(flag, 0) - flag).int())
    assert torch.equal(off, (torch.cumsum(bound, 0) - bound).int())
    assert torch.equal(lst[:n], flag.nonzero()[:, 0].int()) and bool((lst[n:] == -1).all())
    assert not bool(zero.any())
