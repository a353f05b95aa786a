"""The intersection ops' tile and octant culling against the oracle, where it
could lose or reorder a hit: voxel counts around the 64-voxel tiles and past
the 65,536 voxels a block holds boxes for, voxels in no order, NaN centres,
zero direction components, truncated rows; and trees the octant check must
refuse, or accept with leaves beside internal nodes."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import nsvf_oracle as O
from _cases import axis_rays, random_rays, shell, shell_octree, shell_rays
from nsvf_amd import _ext, _lib

pytestmark = pytest.mark.gpu


def _same(outs, refs, what):
    for o, r, w in zip(outs, refs, ("idx", "min_depth", "max_depth")):
        assert np.array_equal(o.cpu().numpy(), r), f"{what}: {w}"


def _dev(a, device):
    return torch.from_numpy(np.ascontiguousarray(a)).to(device)


@pytest.mark.parametrize("n,n_max", [(1, 4), (63, 3), (64, 64), (65, 60), (6568, 1), (70_001, 60)])
@pytest.mark.parametrize("nan", [False, True])
def test_aabb_tiles(device, n, n_max, nan):
    rng = np.random.default_rng(n)
    pts = rng.uniform(-0.8, 0.8, (n, 3)).astype(np.float32)
    if n == 6568:
        pts = shell().points.copy()
    if nan:
        pts[rng.integers(0, n, 1 + n // 200), rng.integers(0, 3)] = np.nan
    a, b = random_rays(300, seed=n), axis_rays(shell(), 100, seed=n)
    rs, rd = (np.concatenate(x) for x in zip(a, b))
    size = 0.0625 if n < 10_000 else 0.02
    ref = O.aabb_intersect(rs[None], rd[None], pts[None], size, n_max)
    out = _ext.aabb_intersect(_dev(rs[None], device), _dev(rd[None], device),
                              _dev(pts[None], device), size, n_max)
    _same(out, ref, f"aabb n={n} n_max={n_max} nan={nan}")


def _trees():
    cen, ch = (x.copy() for x in shell_octree())
    yield "as built", cen, ch
    moved = cen.copy()
    moved[100] += 0.4                        # a leaf far outside its octant
    yield "moved leaf", moved, ch
    mixed = ch.copy()
    T = ch.shape[0]
    for node in range(T - 1, 0, -1):         # a leaf beside internal nodes, held by the octant
        kids, leaf = mixed[node, :8], node
        if mixed[node, 8] < 8 or not (kids < 0).any():
            continue
        while mixed[leaf, 8] != 1:
            leaf = mixed[leaf, :8].max()
        kids[np.nonzero(kids < 0)[0][0]] = leaf
    yield "mixed children", cen, mixed
    nan = cen.copy()
    nan[T - 2] = np.nan
    yield "NaN centre", nan, ch


@pytest.mark.parametrize("case", range(4))
@pytest.mark.parametrize("n_max", [60, 5])
def test_svo_trees(device, case, n_max):
    name, cen, ch = list(_trees())[case]
    sc = shell()
    rays = (random_rays(1500, seed=3), axis_rays(sc, 500, seed=4), shell_rays(width=24))
    rs, rd = (np.concatenate(x) for x in zip(*rays))
    rd[::7] *= np.float32(-1.0)              # turns zero components into -0
    ref = O.svo_intersect(rs[None], rd[None], cen[None], ch[None], sc.voxel_size, n_max)
    args = [_dev(x[None], device) for x in (rs, rd, cen, ch)]
    _same(_ext.svo_intersect(*args, sc.voxel_size, n_max), ref, f"svo {name}")
    # without a workspace, and with a tree per batch: the reference's boxes
    idx = torch.empty((1, rs.shape[0], n_max), dtype=torch.int32, device=device)
    lo, hi = (torch.empty(idx.shape, device=device) for _ in range(2))
    for shared in (1, 0):
        _lib.check(_lib.lib().nsvf_svo_intersect(
            *[a.data_ptr() for a in args], 1, rs.shape[0], cen.shape[0], shared,
            float(sc.voxel_size), n_max, idx.data_ptr(), lo.data_ptr(), hi.data_ptr(),
            torch.cuda.current_stream(device).cuda_stream), "svo_intersect")
        _same((idx, lo, hi), ref, f"svo {name} shared={shared}")
