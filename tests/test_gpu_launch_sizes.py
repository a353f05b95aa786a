"""Calls of more rays or batches than one launch's 2^32 threads hold."""
import ctypes

import pytest
import torch

from nsvf_amd._lib import lib

pytestmark = pytest.mark.gpu
_p = lambda t: ctypes.c_void_p(t.data_ptr())


def test_aabb_batches(device):
    """2^22 batches of one ray, a block of 1,024 threads each: rays along +x
    past one voxel at the origin, every third one beside it."""
    B = (1 << 22) + 5
    rs = torch.zeros((B, 3), device=device)
    rs[:, 0] = -1 - torch.arange(B, device=device) % 7
    rs[::3, 1] = 2
    rd = torch.tensor([1.0, 0.0, 0.0], device=device).expand(B, 3).contiguous()
    pts = torch.zeros((1, 3), device=device)
    idx = torch.empty(B, dtype=torch.int32, device=device)
    lo, hi = torch.empty(B, device=device), torch.empty(B, device=device)
    assert lib().nsvf_aabb_intersect(_p(rs), _p(rd), _p(pts), B, 1, 1, 1, 0.5, 1, _p(idx), _p(lo),
                                     _p(hi), None) == 0, lib().nsvf_last_error()
    torch.cuda.synchronize()
    miss = torch.arange(B, device=device) % 3 == 0
    assert torch.equal(idx, torch.where(miss, -1, 0).int())
    assert torch.equal(lo, torch.where(miss, 0.0, -rs[:, 0] - 0.25))
    assert torch.equal(hi, torch.where(miss, 0.0, -rs[:, 0] + 0.25))


def test_svo_rays(device):
    """2^29 rays and some, eight threads each, against a tree of one leaf; start
    and direction are one buffer."""
    R = (1 << 29) + 100
    rays = torch.full((R, 3), 0.5, device=device)
    miss = [0, 1 << 28, (1 << 28) - 1, (1 << 29) - 1, 1 << 29, R - 1]
    rays[miss] = -0.5
    cen = torch.full((1, 3), 1.5, device=device)
    ch = torch.tensor([[-1] * 8 + [1]], dtype=torch.int32, device=device)
    idx = torch.full((R,), -7, dtype=torch.int32, device=device)
    lo, hi = torch.full((R,), -7.0, device=device), torch.full((R,), -7.0, device=device)
    assert lib().nsvf_svo_intersect(_p(rays), _p(rays), _p(cen), _p(ch), 1, R, 1, 1, 0.5, 1,
                                    _p(idx), _p(lo), _p(hi), None) == 0, lib().nsvf_last_error()
    torch.cuda.synchronize()
    assert idx[miss].eq(-1).all() and lo[miss].eq(0).all() and hi[miss].eq(0).all()
    assert int(idx.eq(0).sum()) == R - len(miss)
    assert int(lo.eq(1.5).sum()) == R - len(miss) and int(hi.eq(2.5).sum()) == R - len(miss)
