"""Layers whose rows or columns lie too far apart for one scale of FP16 pairs
(2^-10 of the layer's largest weight) run on the FP32 units: the training MLP,
forward and backward, and the FP32 field.

Tolerance: the training tests' bar for FP32, 2e-5 of a tensor's largest entry,
and of each row's and column's for the weight gradients."""
import numpy as np
import pytest
import torch

from nsvf_amd.scene import FieldMLP as SceneMLP
from nsvf_amd._lib import lib
from nsvf_amd.train import FieldMLP
from test_gpu_field_f32 import _eval, _scene
from test_gpu_mlp_rows import BAR, _grads, _grads64, _params

pytestmark = pytest.mark.gpu


def _spread(kind, layer, size, seed):
    ps = _params(seed)
    if kind == "off":        # two units of large weights, switched off by their biases
        ps[2 * layer][[17, 90]] *= np.float32(size)
        ps[2 * layer + 1][[17, 90]] = -100 * size
    elif kind == "columns":
        ps[2 * layer][:, 3::9] /= np.float32(size)
    elif kind == "rows":
        ps[2 * layer][1::3] /= np.float32(size)
    return ps


CASES = [("off", l, s) for l in range(3) for s in (1e2, 2e3, 1e5, 1e7)] + [
    (k, l, s) for k in ("columns", "rows") for l in range(4) for s in (1e2, 2e3, 1e6)]


@pytest.mark.parametrize("kind,layer,size", CASES)
def test_training_mlp(device, kind, layer, size):
    M = 64 * 3 + 20
    rng = np.random.default_rng(31)
    ps = _spread(kind, layer, size, 31)
    emb = (rng.standard_normal((M, 32)) * 0.1).astype(np.float32)
    dout = rng.standard_normal((M, 4)).astype(np.float32)
    want = _grads64(emb, ps, dout)
    got = _grads(FieldMLP, emb, ps, dout, device)
    for i, (a, b) in enumerate(zip(got, want)):
        assert (a - b).abs().max() <= BAR * b.abs().max(), i
    for a, b in zip(got[1::2], want[1::2]):   # rows and columns by their largest entry
        for d in (0, 1):
            assert ((a - b).abs().amax(d) <= 10 * BAR * b.abs().amax(d)).all(), (a.shape, d)
    h = torch.from_numpy(emb).double()
    for i in range(0, 8, 2):
        h = h @ torch.from_numpy(ps[i]).double().T + torch.from_numpy(ps[i + 1]).double()
        h = torch.relu(h) if i < 6 else torch.cat([h[:, :1], torch.sigmoid(h[:, 1:])], 1)
    with torch.no_grad():
        out = FieldMLP.apply(*(torch.from_numpy(x).to(device) for x in (emb, *ps))).cpu().double()
    assert (out - h).abs().max() <= BAR * h.abs().max()


@pytest.mark.parametrize("kind,layer,size", [c for c in CASES if c[2] > 1e3])
def test_field(device, kind, layer, size):
    """The FP32 field of such a network is the FP32 units', bit for bit."""
    ps = _spread(kind, layer, size, 32)
    mlp = SceneMLP(ps[0::2], ps[1::2])
    scene = _scene(32, 0.3)
    a = _eval(lambda a: lib().nsvf_field_eval(1, *a, None, 0, None), scene, 0.3, mlp, device)
    b = _eval(lambda a: lib().nsvf_field_eval_f32(*a, None), scene, 0.3, mlp, device)
    np.testing.assert_array_equal(a, b)
    ps = _spread(kind, layer, 10, 32)
    mlp = SceneMLP(ps[0::2], ps[1::2])
    a = _eval(lambda a: lib().nsvf_field_eval(1, *a, None, 0, None), scene, 0.3, mlp, device)
    b = _eval(lambda a: lib().nsvf_field_eval_f32(*a, None), scene, 0.3, mlp, device)
    assert not np.array_equal(a, b) and np.abs(a - b).max() <= BAR * np.abs(b).max()
