"""The offsets of calls beyond the tiles that a block adds up by itself (8.4
million rays), and the limit of the scans (33.5 million)."""
import ctypes

import pytest
import torch

from nsvf_amd._lib import lib

pytestmark = pytest.mark.gpu
_p = lambda x: ctypes.c_void_p(x.data_ptr())
DIRECT, MOST = 4096 * 2048, 16384 * 2048


def _call(device, R):
    g = torch.Generator(device=device).manual_seed(R)
    flag = (torch.rand(R, generator=g, device=device) < 0.4).int()
    bound = torch.randint(0, 100, (R,), generator=g, dtype=torch.int32, device=device) * flag
    rank, lst, off, zero = (torch.full((R,), -1, dtype=torch.int32, device=device)
                            for _ in range(4))
    scal = torch.full((9,), -1, dtype=torch.int32, device=device)
    ws = torch.empty(int(lib().nsvf_render_offsets_workspace_ints(R)), dtype=torch.int32,
                     device=device)
    rc = lib().nsvf_render_offsets(_p(flag), _p(bound), R, _p(rank), _p(lst), _p(off), _p(zero),
                                   _p(scal), 8, _p(ws), None)
    torch.cuda.synchronize()
    return rc, flag, bound, rank, lst, off, zero, scal


@pytest.mark.parametrize("R", [DIRECT, DIRECT + 1, 10_000_003, MOST])
def test_offsets(device, R):
    rc, flag, bound, rank, lst, off, zero, scal = _call(device, R)
    assert rc == 0
    n = int(flag.sum())
    assert scal.tolist() == [n, int(bound.sum())] + [0] * 6 + [-1]
    assert torch.equal(rank, torch.cumsum(flag, 0, dtype=torch.int32) - flag)
    assert torch.equal(off, torch.cumsum(bound, 0, dtype=torch.int32) - bound)
    assert torch.equal(lst[:n], flag.nonzero()[:, 0].int()) and bool((lst[n:] == -1).all())
    assert not bool(zero.any())


def test_too_many_rays(device):
    assert _call(device, MOST + 1)[0] != 0
    assert b"too many rays" in lib().nsvf_last_error()
