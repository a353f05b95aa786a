"""The FP32 MLP on the FP16 matrix units (csrc/mlp_f16x3.h) where its scaling
could fail: sample counts around its 32-sample tiles, operands far from 1 in
either direction, columns of zeros, and inputs that are not finite (which run
on the FP32 units).

Tolerance: an FP32 evaluation rounds every layer's sums; each layer adds at
most about K/32 + 4 roundings of 2^-24 of its sum of absolute products, which
the following layers multiply by |W|.  So the error of an output is held to
2^-20 of the network of absolute values, evaluated in float64."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from nsvf_amd import scene as S
from nsvf_amd.train import FieldMLP

pytestmark = pytest.mark.gpu


def _mlp(seed, scales=(1.0, 1.0, 1.0, 1.0)):
    mlp = S.make_mlp(32, 128, 3, seed)
    return ([w * np.float32(s) for w, s in zip(mlp.weights, scales)], list(mlp.biases))


def _run(emb, ws, bs, device):
    params = []
    for w, b in zip(ws, bs):
        params += [torch.from_numpy(w).to(device), torch.from_numpy(b).to(device)]
    with torch.no_grad():
        return FieldMLP.apply(torch.from_numpy(emb).to(device), *params).cpu().numpy()


def _sums64(emb, ws, bs):
    """The head's sums, the same network over absolute values, and the largest
    value in any layer of that."""
    h, a = emb.astype(np.float64), np.abs(emb).astype(np.float64)
    top = a.max()
    for i, (w, b) in enumerate(zip(ws, bs)):
        w, b = w.astype(np.float64), b.astype(np.float64)
        h, a = h @ w.T + b, a @ np.abs(w).T + np.abs(b)
        top = max(top, a.max())
        if i + 1 < len(ws):
            h = np.maximum(h, 0)
    return h, a, top


def _check(out, emb, ws, bs):
    z, a, _ = _sums64(emb, ws, bs)
    tol = a * 2.0 ** -20
    assert (np.abs(out[:, 0] - z[:, 0]) <= tol[:, 0]).all()
    with np.errstate(over="ignore"):
        rgb = 1 / (1 + np.exp(-z[:, 1:]))
    assert (np.abs(out[:, 1:] - rgb) <= tol[:, 1:] / 4 + 2.0 ** -22).all()


@pytest.mark.parametrize("M", [1, 15, 16, 17, 31, 32, 33, 255, 257, 4097])
def test_sample_counts(device, M):
    ws, bs = _mlp(3)
    emb = (np.random.default_rng(M).standard_normal((M, 32)) * 0.1).astype(np.float32)
    emb[::5] = 0
    _check(_run(emb, ws, bs, device), emb, ws, bs)


@pytest.mark.parametrize("emb_scale", [1e-30, 1e-3, 1e4, 1e30])
@pytest.mark.parametrize("scales", [(1, 1, 1, 1), (1e-12, 1e12, 1e-6, 1e6), (1e9, 1e-20, 1, 1e8),
                                    (1e-30, 1, 1, 1)])
def test_scales(device, emb_scale, scales):
    ws, bs = _mlp(4, scales)
    rng = np.random.default_rng(7)
    emb = (rng.standard_normal((100, 32)) * 0.1 * emb_scale).astype(np.float32)
    # columns of mixed magnitudes
    emb[50:] *= (10.0 ** rng.uniform(-6, 0, (50, 32))).astype(np.float32)
    if _sums64(emb, ws, bs)[2] > 1e37:
        pytest.skip("beyond FP32's range")
    _check(_run(emb, ws, bs, device), emb, ws, bs)


def test_not_finite(device):
    """A NaN feature gives layer-0 sums of NaN, which the ReLU (fmax) turns
    into 0; an infinite one gives infinities of the weights' signs.  Only the
    samples that hold them are affected, in every tile position."""
    ws, bs = _mlp(5)
    emb = (np.random.default_rng(8).standard_normal((96, 32)) * 0.1).astype(np.float32)
    clean = emb.copy()
    emb[3, 5] = np.nan
    emb[40, 0] = np.inf
    emb[95, 31] = -np.inf
    out = _run(emb, ws, bs, device)
    ok = np.ones(96, bool)
    ok[[3, 40, 95]] = False
    _check(out[ok], clean[ok], ws, bs)
    h = np.zeros(128, np.float64)
    for w, b in zip(ws[1:-1], bs[1:-1]):
        h = np.maximum(w.astype(np.float64) @ h + b, 0)
    assert abs(out[3, 0] - (ws[-1][0].astype(np.float64) @ h + bs[-1][0])) < 1e-5
    with np.errstate(invalid="ignore", over="ignore"):
        for s in (40, 95):
            h = emb[s]
            for w, b in zip(ws[:-1], bs[:-1]):
                h = np.fmax(w @ h + b, np.float32(0))
            want = ws[-1][0] @ h + bs[-1][0]
            assert np.isnan(out[s, 0]) == np.isnan(want) or np.isinf(out[s, 0]) == np.isinf(want)


def test_weights_not_finite(device):
    ws, bs = _mlp(6)
    emb = (np.random.default_rng(9).standard_normal((64, 32)) * 0.1).astype(np.float32)
    ws[2] = ws[2].copy()
    ws[2][7] = np.nan                        # row 7 of the last hidden layer: ReLU gives 0
    out = _run(emb, ws, bs, device)
    ws[2][7] = 0
    bs[2] = bs[2].copy()
    bs[2][7] = 0
    _check(out, emb, ws, bs)


def _backward(emb, ws, bs, dout, device):
    leaves = [torch.from_numpy(a).to(device).requires_grad_()
              for a in [emb] + [x for wb in zip(ws, bs) for x in wb]]
    out = FieldMLP.apply(*leaves)
    return [g.cpu().double() for g in
            torch.autograd.grad(out, leaves, torch.from_numpy(dout).to(device))]


def _backward64(emb, ws, bs, dout, dead=()):
    """float64 autograd, and dout with the samples near a ReLU kink zeroed;
    dead: samples whose first layer's outputs are taken as 0."""
    e = torch.from_numpy(emb).double().requires_grad_()
    ps = [torch.from_numpy(x).double().requires_grad_() for wb in zip(ws, bs) for x in wb]
    h, near = e, torch.zeros(len(emb), dtype=torch.bool)
    for i in range(len(ws)):
        z = h @ ps[2 * i].T + ps[2 * i + 1]
        if i + 1 < len(ws):
            scale = (h.detach().abs() @ ps[2 * i].detach().abs().T + ps[2 * i + 1].detach().abs())
            near |= (z.detach().abs() < 1e-5 * scale).any(1)
            h = torch.relu(z)
            if i == 0 and len(dead):
                keep = torch.ones(len(emb), 1, dtype=torch.float64)
                keep[list(dead)] = 0
                h = h * keep
    near[list(dead)] = False
    out = torch.cat([z[:, :1], torch.sigmoid(z[:, 1:])], 1)
    dout = dout.copy()
    dout[near.numpy()] = 0
    return torch.autograd.grad(out, [e, *ps], torch.from_numpy(dout).double()), dout


def _close(got, want, what):
    # FP32's bar of the training tests: 2e-5 of a tensor's largest entry
    for i, (a, b) in enumerate(zip(got, want)):
        assert (a - b).abs().max() <= 2e-5 * max(float(b.abs().max()), 1e-37), (what, i)


@pytest.mark.parametrize("M", [1, 63, 64, 65, 130, 64 * 256 + 3])
def test_backward_sample_counts(device, M):
    ws, bs = _mlp(7)
    rng = np.random.default_rng(M)
    emb = (rng.standard_normal((M, 32)) * 0.1).astype(np.float32)
    dout = rng.standard_normal((M, 4)).astype(np.float32)
    want, dout = _backward64(emb, ws, bs, dout)
    _close(_backward(emb, ws, bs, dout, device), want, M)


@pytest.mark.parametrize("emb_scale,dout_scale,scales", [
    (1.0, 1e-25, (1, 1, 1, 1)), (1.0, 1e15, (1, 1, 1, 1)), (1e4, 1.0, (1, 1e-3, 1, 1e-2)),
    (1e-4, 1.0, (1e3, 1e2, 1e-4, 1)), (1e-30, 1.0, (1, 1, 1, 1)), (1.0, 1.0, (1e25, 1, 1, 1e-25))])
def test_backward_scales(device, emb_scale, dout_scale, scales):
    """Gradients over 20 decades in one call, samples without any, operands
    far from 1 -- the last two beyond the FP16 form's window, so FP32 MFMAs."""
    ws, bs = _mlp(8, scales)
    rng = np.random.default_rng(11)
    emb = (rng.standard_normal((300, 32)) * 0.1 * emb_scale).astype(np.float32)
    dout = (rng.standard_normal((300, 4)) * dout_scale
            * 10.0 ** rng.uniform(-12, 0, (300, 1))).astype(np.float32)
    dout[::7] = 0
    want, dout = _backward64(emb, ws, bs, dout)
    got = _backward(emb, ws, bs, dout, device)
    _close(got, want, (emb_scale, dout_scale))
    # a sample's own gradient, however small beside the others'
    size = want[0].abs().amax(1)
    err = (got[0] - want[0]).abs().amax(1)
    assert (err <= 1e-4 * size + 1e-37).all()


def test_backward_not_finite(device):
    """A NaN feature: its sample's first layer is all 0 (fmax), so the NaN
    reaches that feature's column of dW_0 only; the call runs on the FP32
    MFMAs."""
    ws, bs = _mlp(9)
    rng = np.random.default_rng(12)
    emb = (rng.standard_normal((200, 32)) * 0.1).astype(np.float32)
    dout = rng.standard_normal((200, 4)).astype(np.float32)
    want, dout = _backward64(emb, ws, bs, dout, dead=(70,))
    bad = emb.copy()
    bad[70, 5] = np.nan
    got = _backward(bad, ws, bs, dout, device)
    assert got[1][:, 5].isnan().all()
    got[1][:, 5] = want[1][:, 5]
    _close(got, want, "NaN feature")


def test_backward_gradient_not_finite(device):
    """An infinite output gradient stays with its sample's input gradient."""
    ws, bs = _mlp(10)
    rng = np.random.default_rng(13)
    emb = (rng.standard_normal((150, 32)) * 0.1).astype(np.float32)
    dout = rng.standard_normal((150, 4)).astype(np.float32)
    want, dout = _backward64(emb, ws, bs, dout)
    dout[33, 0] = np.inf
    got = _backward(emb, ws, bs, dout, device)
    keep = np.arange(150) != 33
    _close([got[0][keep]], [want[0][keep]], "infinite gradient")
    assert not got[0][33].isfinite().all() and not got[1].isfinite().all()
