"""The training step's packing, point and background kernels against the torch
operations that they stand for."""
import numpy as np
import pytest
import torch

from _cases import shell, shell_rays
from nsvf_amd.render import BG_COLOR, BG_DEPTH, DeviceScene, Renderer
from nsvf_amd.train import (StreamComposite, _CompositeOver, _pack_split, pack_mlp_train_x3,
                            pack_mlp_x3)
from nsvf_amd._lib import check, lib
from nsvf_amd.train import _p, _stream

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("strided", [False, True])
def test_split_pack(device, strided):
    g = torch.Generator().manual_seed(2)
    shapes = [(128, 32), (128, 128), (128, 128), (4, 128)]
    ws = [torch.randn(s, generator=g) for s in shapes]
    ws[0][3, 5], ws[1][0, 0], ws[2][1, 1] = 1e-41, -0.0, 3e38
    bs = [torch.randn(s[0], generator=g) for s in shapes]
    to = lambda t: (t.t().contiguous().to(device).t() if strided and t.dim() == 2 else t.to(device))
    frags, back, bias, count = _pack_split([to(w) for w in ws], [to(b) for b in bs], 77, True)
    want, want_bias = pack_mlp_x3(ws, bs)
    assert torch.equal(frags.cpu(), want) and torch.equal(bias.cpu(), want_bias)
    assert torch.equal(back.cpu(), pack_mlp_train_x3(ws)) and int(count) == 77


def _stream_of(device):
    rs, rd = (torch.from_numpy(x).to(device) for x in shell_rays(width=40))
    dsc = DeviceScene(shell(), device)
    g = Renderer(device, precision="fp32", hierarchical=False).coarse_stream(dsc, rs, rd).owned()
    return rs, rd, g


def test_stream_points(device):
    rs, rd, g = _stream_of(device)
    M = g.samples.shape[0]
    assert M % 256 and bool((g.samples[:, 0] == -1).any())
    s_idx = torch.empty(M, dtype=torch.int32, device=device)
    xyz = torch.empty((M, 3), device=device)
    check(lib().nsvf_stream_points(_p(g.samples), M, _p(rs), _p(rd), rs.shape[0], _p(s_idx),
                                   _p(xyz), _stream(device)), "stream_points")
    ray, depth = g.samples[:, 3].long(), g.samples[:, 1].view(torch.float32)
    assert torch.equal(s_idx, g.samples[:, 0])
    assert torch.equal(xyz, rs[ray] + rd[ray] * depth[:, None])


@pytest.mark.parametrize("used", ["rgb", "depth", "missed", "all"])
def test_composite_over(device, used):
    """Same outputs; the gradients' background term is summed by the kernel,
    so its three products may round in another order: 4 ulp of the largest."""
    rs, rd, g = _stream_of(device)
    assert 0 < g.n_hit < g.rays
    gen = torch.Generator().manual_seed(3)
    f = torch.randn((g.slots, 4), generator=gen).to(device)
    up = [torch.randn(s, generator=gen).to(device) for s in ((g.rays, 3), (g.rays,), (g.rays,))]
    a, b = (f.clone().requires_grad_(True) for _ in range(2))
    got = _CompositeOver.apply(a, g)
    rgb, dep, missed = StreamComposite.apply(b, g)
    bg = torch.tensor(BG_COLOR, device=device)
    want = (rgb + missed[:, None] * bg, dep + missed * BG_DEPTH, missed)
    loss = [0, 0]
    for i, name in enumerate(("rgb", "depth", "missed")):
        assert torch.equal(got[i], want[i]), name
        if used in (name, "all"):
            loss = [loss[0] + (got[i] * up[i]).sum(), loss[1] + (want[i] * up[i]).sum()]
    loss[0].backward()
    loss[1].backward()
    assert float((a.grad - b.grad).abs().max()) <= 4 * 2.0 ** -23 * float(b.grad.abs().max())
