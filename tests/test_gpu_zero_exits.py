"""Exit depths of zero: a ray that starts on a voxel's face, edge or corner and
leaves it there has bounds of both zeros, and the depth keeps the sign that the
reference's comparisons leave it with, in the ops and in the fused traversal."""
import ctypes

import numpy as np
import pytest
import torch

import nsvf_oracle as O
from _cases import shell, shell_octree
from nsvf_amd import _ext
from nsvf_amd._lib import lib
from nsvf_amd.render import DeviceScene

pytestmark = pytest.mark.gpu


def _rays(points, half, n, seed):
    """Origins on faces, edges and corners of voxels, directions away from
    them, with zero components of both signs."""
    rng = np.random.default_rng(seed)
    c = points[rng.integers(0, len(points), n)]
    side = rng.integers(-1, 2, (n, 3)).astype(np.float32)
    rs = (c + side * np.float32(half)).astype(np.float32)
    rd = rng.uniform(0.1, 1, (n, 3)).astype(np.float32) * np.where(side == 0, 1, side)
    rd *= rng.choice(np.float32([-1, 0, 1, 1]), (n, 3))
    rd[(rd == 0).all(1)] = (1, 0, 0)
    return rs, rd.astype(np.float32)


def _bits(x):
    return np.ascontiguousarray(x).view(np.int32)


def test_zero_exits(device):
    sc = shell()
    rs, rd = _rays(sc.points, np.float32(sc.voxel_size) / 2, 6000, 51)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(device)
    ref = O.aabb_intersect(rs[None], rd[None], sc.points[None], sc.voxel_size, 60)
    zero = ref[2][(ref[0] >= 0) & (ref[2] == 0)]
    assert (np.signbit(zero)).sum() > 20 and (~np.signbit(zero)).sum() > 20
    got = _ext.aabb_intersect(dev(rs[None]), dev(rd[None]), dev(sc.points[None]), sc.voxel_size, 60)
    for g, r in zip(got, ref):
        assert np.array_equal(_bits(g.cpu().numpy()), _bits(r))
    cen, ch = shell_octree()
    ref = O.svo_intersect(rs[None], rd[None], cen[None], ch[None], sc.voxel_size, 60)
    got = _ext.svo_intersect(dev(rs[None]), dev(rd[None]), dev(cen[None]), dev(ch[None]),
                             sc.voxel_size, 60)
    for g, r in zip(got, ref):
        assert np.array_equal(_bits(g.cpu().numpy()), _bits(r))
    # the fused traversal's rows (sorted by entry depth) hold the same records;
    # its two walks: rays alone, and 64 sharing one
    ds, P, R0 = DeviceScene(sc, device), 60, len(rs)
    lo, hi = ref[1][0], ref[2][0]
    for copies in (1, 33):
        R = R0 * copies
        assert bool(lib().nsvf_render_hits_alone(R)) == (copies == 1)
        drs, drd = dev(np.tile(rs, (copies, 1))), dev(np.tile(rd, (copies, 1)))
        hits = torch.zeros((R, P, 4), dtype=torch.int32, device=device)
        out = [torch.empty(R, dtype=d, device=device)
               for d in (torch.int32, torch.float32, torch.int32, torch.int32)]
        p = lambda t: ctypes.c_void_p(t.data_ptr())
        assert lib().nsvf_render_hits(p(drs), p(drd), R, 0, p(ds.tree_records), ds.num_nodes,
                                      ds.tree_depth, P, ds.step_size, p(hits),
                                      *(p(o) for o in out), None) == 0
        torch.cuda.synchronize()
        h = hits[-R0:].cpu().numpy()
        count = out[0][-R0:].cpu().numpy()
        assert np.array_equal(count, (ref[0][0] >= 0).sum(1))
        # by entry depth, bits of the exit depth
        for r in np.nonzero(((ref[2][0] == 0) & (ref[0][0] >= 0)).any(1))[0]:
            n = count[r]
            order = np.argsort(lo[r, :n], kind="stable")
            assert np.array_equal(h[r, :n, 0], _bits(lo[r, :n][order]))
            assert np.array_equal(h[r, :n, 1], _bits(hi[r, :n][order]))
