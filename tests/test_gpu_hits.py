"""The traversal's two kernels, a walk per ray (small calls) and a walk per 64
rays, give the same rows: one large call against the same rays in pieces."""
import ctypes

import numpy as np
import pytest
import torch

from _cases import shell
from nsvf_amd import scene as S
from nsvf_amd._lib import lib
from nsvf_amd.render import DeviceScene

pytestmark = pytest.mark.gpu


def hits(dsc, rs, rd, n_max, width=0, order=None):
    R, dev = rs.shape[0], rs.device
    row = torch.full((R, n_max, 4), -7, dtype=torch.int32, device=dev)
    cnt, flag, bound = (torch.full((R,), -7, dtype=torch.int32, device=dev) for _ in range(3))
    tot = torch.full((R,), -7.0, device=dev)
    p = lambda x: ctypes.c_void_p(x.data_ptr())
    tail = (p(dsc.tree_records), dsc.num_nodes, dsc.tree_depth, n_max, 0.01, p(row), p(cnt),
            p(tot), p(flag), p(bound), None)
    if order is None:
        rc = lib().nsvf_render_hits(p(rs), p(rd), R, width, *tail)
    else:
        rc = lib().nsvf_render_hits_ordered(p(rs), p(rd), R, p(order), *tail)
    assert rc == 0
    torch.cuda.synchronize()
    return row, cnt, tot.view(torch.int32), flag, bound


@pytest.mark.parametrize("n_max", [60, 7, 1])
@pytest.mark.parametrize("kind", ["image", "order", "mixed"])
def test_one_call_equals_its_pieces(device, kind, n_max):
    dsc = DeviceScene(shell(), device)
    L = lib()
    w = 456
    rs, rd = (torch.from_numpy(x).to(device) for x in S.camera_rays(w, w, S.sphere_camera(2.5, 7)))
    if kind == "mixed":   # rays of every direction, along axes, from inside the scene
        g = torch.Generator().manual_seed(3)
        rd = torch.randn(rs.shape, generator=g).to(device)
        rd[::5, 0], rd[::7, 1] = 0.0, -0.0
        rd = rd / rd.norm(dim=1, keepdim=True)
        rs = (torch.rand(rs.shape, generator=g).to(device) * 2 - 1) * 1.2
    R = rs.shape[0]
    assert not L.nsvf_render_hits_alone(R) and L.nsvf_render_hits_alone(9999)
    order = None
    if kind == "order":
        order = torch.randperm(R, generator=torch.Generator().manual_seed(4)).int().to(device)
    one = hits(dsc, rs, rd, n_max, w if kind == "image" else 0, order)
    cuts = list(range(0, R, 49_999)) + [R - 3, R]
    parts = [hits(dsc, rs[a:b].contiguous(), rd[a:b].contiguous(), n_max)
             for a, b in zip(cuts, cuts[1:])]
    parts = [torch.cat(x) for x in zip(*parts)]
    cnt = one[1]
    assert int(cnt.max()) > min(n_max, 12) - 1
    live = torch.arange(n_max, device=device)[None] < cnt[:, None]
    for a, b in zip(one[1:], parts[1:]):
        assert torch.equal(a, b)
    assert torch.equal(one[0][live], parts[0][live])
