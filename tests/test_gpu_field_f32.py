"""nsvf_field_eval_f32's gather rounds every product and sum by itself, corner
after corner, as does the FP32 field's path for tiles that are not finite: a
network that hands one feature through shows its bits."""
import ctypes

import numpy as np
import pytest
import torch

from nsvf_amd._lib import lib
from nsvf_amd.field import pack_mlp
from nsvf_amd.scene import FieldMLP

pytestmark = pytest.mark.gpu

# the field's built shapes: embedding, width, hidden layers
SHAPES = [(32, 128, 3), (48, 256, 4), (32, 256, 4)]


def _scene(D, vs, M=1000, N=50, K=90):
    rng = np.random.default_rng(31)
    centers = rng.uniform(-1, 1, (N, 3)).astype(np.float32)
    feats = rng.integers(0, K, (N, 8)).astype(np.int32)
    values = rng.uniform(0.1, 1, (K, D)).astype(np.float32)
    idx = rng.integers(-1, N, M).astype(np.int32)
    x = centers[idx.clip(0)] + (rng.uniform(-0.5, 0.5, (M, 3)) * vs).astype(np.float32)
    samples = np.zeros((M, 4), np.int32)
    samples[:, 0], samples[:, 3] = idx, np.arange(M)     # a ray per sample, depth 0
    return centers, feats, values, idx, x, samples


def _pass_through(D, H, L, feature):
    ws = [np.zeros((H, D), np.float32)] + [np.zeros((H, H), np.float32) for _ in range(L - 1)]
    ws.append(np.zeros((4, H), np.float32))
    ws[0][0, feature] = 1
    for w in ws[1:]:
        w[0, 0] = 1
    return FieldMLP(ws, [np.zeros(w.shape[0], np.float32) for w in ws])


def _rounded(centers, feats, values, idx, x, vs, feature):
    v = idx.clip(0)
    p = (x - centers[v]) / np.float32(vs) + np.float32(0.5)
    q = np.float32(1) - p
    out = np.zeros(len(idx), np.float32)
    for c in range(8):
        w = ((p if c & 4 else q)[:, 0] * (p if c & 2 else q)[:, 1]) * (p if c & 1 else q)[:, 2]
        out = out + w * values[feats[v, c], feature]
    return np.where(idx < 0, np.float32(0), out)


def _eval(fn, scene, vs, mlp, device):
    t = [torch.from_numpy(a).to(device) for a in (scene[0], scene[1], scene[2], scene[4],
                                                   scene[5])]
    centers, feats, values, x, samples = t
    packed = pack_mlp(mlp, device)
    M = samples.shape[0]
    dirs = torch.ones_like(x)
    m_dev = torch.tensor([M], dtype=torch.int32, device=device)
    out = torch.empty((M, 4), device=device)
    p = lambda a: ctypes.c_void_p(a.data_ptr())
    D, H, L = mlp.weights[0].shape[1], mlp.weights[0].shape[0], len(mlp.weights) - 1
    args = (D, H, L, p(centers), p(feats), p(values), vs, p(x), p(dirs), p(samples), None,
            p(m_dev), M, p(packed["f32"]), p(packed["bias"]), p(out))
    assert fn(args) == 0
    torch.cuda.synchronize()
    return out.cpu().numpy()


@pytest.mark.parametrize("vs", [0.25, 0.3])
@pytest.mark.parametrize("D,H,L", SHAPES)
def test_gather_rounds_every_operation(device, D, H, L, vs):
    scene = _scene(D, vs)
    for feature in (0, 5, 17, D - 1):
        mlp = _pass_through(D, H, L, feature)
        got = _eval(lambda a: lib().nsvf_field_eval_f32(*a, None), scene, vs, mlp, device)
        np.testing.assert_array_equal(got[:, 0], _rounded(*scene[:5], vs, feature))


def test_tiles_on_the_fp32_units(device):
    """One infinite feature per 32 samples sends every tile there."""
    D, H, L, vs = 32, 128, 3, 0.3
    centers, feats, values, idx, x, samples = _scene(D, vs)
    mlp = _pass_through(D, H, L, 5)
    values = np.concatenate([values, np.full((8, D), np.inf, np.float32)])
    centers = np.concatenate([centers, np.full((1, 3), 3, np.float32)])
    feats = np.concatenate([feats, np.arange(90, 98, dtype=np.int32)[None]])
    wild = np.arange(len(idx)) % 32 == 7
    idx = np.where(wild, 50, idx).astype(np.int32)
    x = np.where(wild[:, None], np.float32(3), x)
    samples[:, 0] = idx
    scene = (centers, feats, values, idx, x, samples)
    got = _eval(lambda a: lib().nsvf_field_eval(1, *a, None, 0, None), scene, vs, mlp, device)
    with np.errstate(invalid="ignore"):
        want = _rounded(*scene[:5], vs, 5)
    np.testing.assert_array_equal(got[~wild, 0], want[~wild])
