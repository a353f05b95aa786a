"""The training backward where a tensor's largest entry says nothing: rows of
the weight gradients that only samples with far smaller gradients than their
neighbours' reach, units with a large negative bias, and the split-BF16
backward's logits.

Tolerance: the training tests' bar for FP32, 2e-5 of a tensor's largest entry,
for each row (or column) by itself."""
import numpy as np
import pytest
import torch

from nsvf_amd import scene as S
from nsvf_amd.train import FieldMLP, FieldMLPx3

pytestmark = pytest.mark.gpu

BAR = 2e-5


def _grads(fn, emb, params, dout, device):
    leaves = [torch.from_numpy(x).to(device).requires_grad_() for x in (emb, *params)]
    out = fn.apply(*leaves)
    return [g.cpu().double() for g in
            torch.autograd.grad(out, leaves, torch.from_numpy(dout).to(device))]


def _grads64(emb, params, dout, margin=1e-5):
    """float64 autograd; samples near a ReLU kink lose their gradient (dout is
    changed)."""
    leaves = [torch.from_numpy(x).double().requires_grad_() for x in (emb, *params)]
    h, near = leaves[0], torch.zeros(len(emb), dtype=torch.bool)
    for i in range(1, len(leaves), 2):
        z = h @ leaves[i].T + leaves[i + 1]
        if i + 2 < len(leaves):
            scale = h.detach().abs() @ leaves[i].detach().abs().T
            near |= (z.detach().abs() < margin * scale).any(1)
            h = torch.relu(z)
    dout[near.numpy()] = 0
    out = torch.cat([z[:, :1], torch.sigmoid(z[:, 1:])], 1)
    return torch.autograd.grad(out, leaves, torch.from_numpy(dout).double())


def _rows_close(got, want, what):
    err, size = (got - want).abs().amax(-1), want.abs().amax(-1)
    assert (size > 0).any()
    assert (err <= BAR * size).all(), (what, float((err / size.clamp(min=1e-300)).max()))


def _params(seed):
    mlp = S.make_mlp(32, 128, 3, seed)
    return [x.copy() for wb in zip(mlp.weights, mlp.biases) for x in wb]


@pytest.mark.parametrize("ratio", [1e-2, 1e-4, 1e-6, 1e-7, 1e-8, 1e-9, 1e-12, 1e-20])
def test_rows_of_small_samples(device, ratio):
    """Unit 5 of the first layer, 7 of the second and 9 of the third are active
    on every fourth sample only, whose gradients are `ratio` of the others'."""
    M = 64 * 5 + 9
    rng = np.random.default_rng(21)
    ps = _params(21)
    for l, unit, source in ((0, 5, 0), (1, 7, 5), (2, 9, 7)):
        ps[2 * l][unit], ps[2 * l + 1][unit] = 0, 0
        ps[2 * l][unit, source] = 1
    emb = (rng.standard_normal((M, 32)) * 0.1).astype(np.float32)
    small = np.arange(M) % 4 == 1
    emb[:, 0] = np.where(small, 0.5, -0.5)
    dout = rng.standard_normal((M, 4)).astype(np.float32)
    dout[small] *= np.float32(ratio)
    want = _grads64(emb, ps, dout)
    got = _grads(FieldMLP, emb, ps, dout, device)
    for l, unit in ((0, 5), (1, 7), (2, 9)):
        _rows_close(got[1 + 2 * l][unit][None], want[1 + 2 * l][unit][None], f"dW_{l} row")
        _rows_close(got[3 + 2 * l][:, unit][None], want[3 + 2 * l][:, unit][None],
                    f"dW_{l + 1} column")
        _rows_close(got[2 + 2 * l][unit].reshape(1, 1), want[2 + 2 * l][unit].reshape(1, 1),
                    f"db_{l}")
    for i, (a, b) in enumerate(zip(got, want)):
        assert (a - b).abs().max() <= BAR * b.abs().max(), i


def test_every_sample_of_another_size(device):
    """Gradients that fall by a factor of 2 from sample to sample, 2^-62 in a
    chunk of 64."""
    M = 64 * 3
    rng = np.random.default_rng(22)
    ps = _params(22)
    emb = (rng.standard_normal((M, 32)) * 0.1).astype(np.float32)
    dout = (rng.standard_normal((M, 4)) * 2.0 ** -(np.arange(M) % 63)[:, None]).astype(np.float32)
    want = _grads64(emb, ps, dout)
    got = _grads(FieldMLP, emb, ps, dout, device)
    _rows_close(got[0], want[0], "demb")
    for i, (a, b) in enumerate(zip(got, want)):
        assert (a - b).abs().max() <= BAR * b.abs().max(), i


@pytest.mark.parametrize("bias", [-1e3, -1e6, -1e9, -1e20, -np.inf])
def test_units_switched_off(device, bias):
    """A large negative bias in each layer switches its unit off and is no bound
    of what the others give."""
    M = 150
    rng = np.random.default_rng(23)
    ps = _params(23)
    for l in range(3):
        ps[2 * l + 1][11 * l + 3] = bias
    emb = (rng.standard_normal((M, 32)) * 0.1).astype(np.float32)
    dout = rng.standard_normal((M, 4)).astype(np.float32)
    want = _grads64(emb, ps, dout)
    got = _grads(FieldMLP, emb, ps, dout, device)
    for i, (a, b) in enumerate(zip(got, want)):
        assert (a - b).abs().max() <= BAR * b.abs().max(), i


def test_split_bf16_backward_logits(device):
    """Two head weights of opposite sign on two outputs that agree in their
    first 16 bits: the logit is a difference that FP32 holds exactly and a pair
    of BF16 parts does not hold at all.  Every other product is of whole
    numbers within 24 bits, so the gradients have FP32's error."""
    M = 200
    rng = np.random.default_rng(25)
    emb = np.zeros((M, 32), np.float32)
    emb[:, :5] = rng.integers(1, 256, (M, 5))
    w = [np.zeros(s, np.float32) for s in ((128, 32), (128, 128), (128, 128), (4, 128))]
    b = [np.zeros(s, np.float32) for s in (128, 128, 128, 4)]
    w[0][range(5), range(5)] = 1
    w[1][0, 0], w[1][0, 1] = 256, 1          # 16 bits
    w[1][1, 2], w[1][1, 3] = 256, 1
    w[1][2, 4] = 1
    w[2][0, 0], w[2][0, 1] = 128, 1          # 23 bits, nearly equal
    w[2][1, 0], w[2][1, 2] = 128, 1
    w[3][0, 0] = 2.0 ** -20
    w[3][1:, 0], w[3][1:, 1] = 2.0 ** -15, -2.0 ** -15
    ps = [x for wb in zip(w, b) for x in wb]
    dout = rng.standard_normal((M, 4)).astype(np.float32)
    want = _grads64(emb, ps, dout, margin=0.0)
    got = _grads(FieldMLPx3, emb, ps, dout, device)
    assert ((got[8] - want[8]).abs() <= BAR * want[8].abs().max()).all()
    # the gradients behind the head are split BF16: 2^-16 of a product's parts
    # each, three layers
    for i, (x, y) in enumerate(zip(got, want)):
        assert (x - y).abs().max() <= 2e-4 * y.abs().max(), i


@pytest.mark.parametrize("wild", [(0,), (63,), (64,), (127, 128), (70, 400), (588,), "all"])
def test_chunks_beyond_the_window(device, wild):
    """Samples whose largest feature is below 2^-40 send their chunk of 64 to
    the FP32 MFMAs, and no other: the others' input gradients keep their bits."""
    M = 64 * 9 + 13
    wild = list(range(0, M, 64)) if wild == "all" else list(wild)
    rng = np.random.default_rng(26)
    ps = _params(26)
    emb = (rng.standard_normal((M, 32)) * 0.1).astype(np.float32)
    emb[wild] = 0
    dout = rng.standard_normal((M, 4)).astype(np.float32)
    want = _grads64(emb, ps, dout)
    tame = _grads(FieldMLP, emb, ps, dout, device)
    emb[wild] = (rng.standard_normal((len(wild), 32)) * 1e-14).astype(np.float32)
    got = _grads(FieldMLP, emb, ps, dout, device)
    there = np.isin(np.arange(M) // 64, np.array(wild) // 64)
    assert torch.equal(got[0][~there], tame[0][~there])
    assert not torch.equal(got[0][there], tame[0][there])
    for i, (a, b) in enumerate(zip(got, want)):   # 1e-14 moves nothing by 2e-5
        assert (a - b).abs().max() <= BAR * b.abs().max(), i
    again = _grads(FieldMLP, emb, ps, dout, device)
    assert all(torch.equal(a, b) for a, b in zip(got, again))


@pytest.mark.parametrize("ratio", [1e-3, 1e-5, 1e-7, 1e-10])
def test_logits_of_other_sizes(device, ratio):
    """Colour gradients far below the samples' density gradients (saturated
    colours, for one): the head's weight rows by themselves."""
    M = 64 * 4 + 5
    rng = np.random.default_rng(27)
    ps = _params(27)
    emb = (rng.standard_normal((M, 32)) * 0.1).astype(np.float32)
    dout = rng.standard_normal((M, 4)).astype(np.float32)
    dout[:, 1:] *= np.float32(ratio) * np.float32([1, 1e-2, 1e2])
    want = _grads64(emb, ps, dout)
    got = _grads(FieldMLP, emb, ps, dout, device)
    _rows_close(got[7], want[7], "dW of the head")
    _rows_close(got[8][:, None], want[8][:, None], "db of the head")
