"""The traversal's two kernels, a walk per ray (small calls) and a walk per 64
rays, give the same rows: one large call against the same rays in pieces."""
import ctypes

import numpy as np
import pytest
import torch

from _cases import shell
from nsvf_amd import _ext, geometry
from nsvf_amd import scene as S
from nsvf_amd import scene_io as IO
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


@pytest.mark.parametrize("n_max", [65, 100, 200])
def test_long_rows_are_stably_sorted(device, n_max):
    """A dense cube (rows of up to 160 hits; many fill, many hold equal entry
    depths): the svo op's rows, stably sorted by entry depth."""
    n, vs = 40, 2.0 ** -4
    g = (np.arange(n) - (n - 1) / 2) * vs
    pts = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3).astype(np.float32)
    sc = IO.scene_from_points(pts, vs, embed_dim=32)
    dsc = DeviceScene(sc, device)
    rng = np.random.default_rng(5)
    R = 300
    d = rng.normal(size=(R, 3)).astype(np.float32)
    d[:150] = np.sign(d[:150])                       # along the diagonals: ties
    d[50:150] += 0.05 * rng.random((100, 3))
    d[280:, 0] = 0.0
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    rd = torch.from_numpy(d.astype(np.float32)).to(device)
    rs = (-3 * rd).contiguous()
    cen, ch = geometry.build_easy_octree(torch.from_numpy(np.ascontiguousarray(sc.points)),
                                         torch.tensor(np.float32(vs)) / 2)
    idx, lo, hi = _ext.svo_intersect(rs[None], rd[None], cen[None].float().to(device),
                                     ch[None].int().to(device), float(np.float32(vs)), n_max)
    idx, lo, hi = idx[0], lo[0], hi[0]
    key = torch.where(idx == -1, torch.full_like(lo, 1e9), lo)
    key, at = key.sort(dim=1, stable=True)
    want = torch.stack([lo.gather(1, at).view(torch.int32), hi.gather(1, at).view(torch.int32),
                        idx.gather(1, at)], 2)
    row, cnt, *_ = hits(dsc, rs, rd, n_max)
    assert torch.equal(cnt, (idx != -1).sum(1).int()) and int(cnt.max()) > 64
    live = torch.arange(n_max, device=device)[None] < cnt[:, None]
    ties = (key[:, 1:] == key[:, :-1]) & live[:, 1:]
    assert bool((ties.any(1) & (cnt > 64)).any())
    assert torch.equal(row[:, :, :3][live], want[live])
