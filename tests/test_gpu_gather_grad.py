"""The gather's backward at the edges of its sort (2,048-sample tiles, one to
three digits), its eight-sample steps and its feature widths, and the gather
itself with rows that can and cannot be read four features at a time."""
import numpy as np
import pytest
import torch

from nsvf_amd.train import trilinear_gather, trilinear_gather_backward

pytestmark = pytest.mark.gpu
VS = 0.5


def scene(N, K, M, D, seed):
    """Positions at quarters of a voxel, small whole gradients and values:
    every weight (n / 64) and sum below 2^24 / 64 is exact in FP32."""
    rng = np.random.default_rng(seed)
    centers = rng.integers(-8, 8, (N, 3)).astype(np.float32)
    feats = rng.integers(0, K, (N, 8)).astype(np.int32)
    s_idx = rng.integers(-1, N, M).astype(np.int32)
    q = rng.integers(0, 5, (M, 3)).astype(np.float32) / 4
    xyz = centers[s_idx] + (q - 0.5).astype(np.float32) * np.float32(VS)
    grad = rng.integers(-3, 4, (M, D)).astype(np.float32)
    values = rng.integers(-9, 10, (K, D)).astype(np.float32)
    return centers, feats, s_idx, xyz, q, grad, values


def weights(q):
    p = [1 - q.astype(np.float64), q.astype(np.float64)]
    return np.stack([p[c >> 2 & 1][:, 0] * p[c >> 1 & 1][:, 1] * p[c & 1][:, 2]
                     for c in range(8)], 1)


CASES = [(1, 3, 1, 4), (7, 5, 2047, 32), (255, 100, 2048, 32), (256, 300, 2049, 64),
         (300, 70_000, 6_000, 128), (65_535, 9, 40_000, 36), (66_000, 65_000, 10_001, 32),
         (40, 60, 3, 8), (3, 8, 5_000, 100)]


@pytest.mark.parametrize("N,K,M,D", CASES)
def test_backward_sums_exactly(device, N, K, M, D):
    centers, feats, s_idx, xyz, q, grad, _ = scene(N, K, M, D, N + M)
    want = np.zeros((K, D))
    live = s_idx >= 0
    w = weights(q)
    for c in range(8):
        np.add.at(want, feats[s_idx[live], c], w[live, c:c + 1] * grad[live])
    t = lambda a: torch.from_numpy(a).to(device)
    got = trilinear_gather_backward(t(s_idx), t(xyz), t(centers), t(feats), K, t(grad), VS)
    np.testing.assert_array_equal(got.cpu().numpy(), want)


def test_backward_keeps_the_sample_order(device):
    """One voxel: its sums run over the samples in their order, each product
    and sum rounded once."""
    rng = np.random.default_rng(5)
    M, D = 4_133, 32
    centers, feats = np.zeros((2, 3), np.float32), np.arange(16).reshape(2, 8).astype(np.int32)
    s_idx = rng.integers(0, 2, M).astype(np.int32)
    q = rng.random((M, 3)).astype(np.float32)
    grad = rng.standard_normal((M, D)).astype(np.float32)
    xyz = q - np.float32(0.5)
    p1 = xyz + np.float32(0.5)
    p = [np.float32(1) - p1, p1]
    want = np.zeros((16, D), np.float32)
    for m in range(M):
        for c in range(8):
            w = (p[c >> 2 & 1][m, 0] * p[c >> 1 & 1][m, 1]) * p[c & 1][m, 2]
            k = s_idx[m] * 8 + c
            want[k] = want[k] + w * grad[m]
    t = lambda a: torch.from_numpy(a).to(device)
    got = trilinear_gather_backward(t(s_idx), t(xyz), t(centers), t(feats), 16, t(grad), 1.0)
    np.testing.assert_array_equal(got.cpu().numpy(), want)


@pytest.mark.parametrize("D,shift", [(32, 0), (36, 0), (32, 1), (5, 0), (1, 0), (4, 2)])
def test_gather_forms(device, D, shift):
    """shift: the values start that many floats past an aligned address."""
    centers, feats, s_idx, xyz, q, _, values = scene(50, 77, 1_003, D, D)
    w = weights(q)
    want = np.where(s_idx[:, None] >= 0,
                    (w[:, :, None] * values[feats[s_idx]]).sum(1), 0)
    t = lambda a: torch.from_numpy(a).to(device)
    flat = torch.zeros(77 * D + 8, device=device)
    flat[shift:shift + 77 * D] = t(values).view(-1)
    v = flat[shift:shift + 77 * D].view(77, D)
    got = trilinear_gather(v, t(s_idx), t(xyz), t(centers), t(feats), VS)
    np.testing.assert_array_equal(got.cpu().numpy(), want)
