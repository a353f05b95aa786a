"""What the training MLP's packing hands to its kernels."""
import numpy as np
import pytest
import torch

from nsvf_amd import scene as S
from nsvf_amd._lib import lib
from nsvf_amd.train import pack_mlp_train

pytestmark = pytest.mark.gpu


def test_packed_bounds_are_summed_in_one_order(device):
    """The largest column sums of |W|, which choose the backward's scales: a
    wave's rows in order, then the 16 waves in order."""
    mlp = S.make_mlp(32, 128, 3, 24)
    ps = [x.copy() for wb in zip(mlp.weights, mlp.biases) for x in wb]
    rng = np.random.default_rng(24)
    for l in range(4):   # magnitudes far apart: another order rounds otherwise
        ps[2 * l] *= (10.0 ** rng.uniform(-3, 3, ps[2 * l].shape)).astype(np.float32)
    dev = [torch.from_numpy(x).to(device) for x in ps]
    packed = pack_mlp_train(dev[0::2], dev[1::2]).cpu().numpy()
    base = packed.size - 512 * (int(lib().nsvf_mlp_train_x3_frags(32, 128, 3)) + 4) - 16
    for l in range(4):
        W = np.abs(ps[2 * l])
        cols = np.zeros(W.shape[1], np.float32)
        for wave in range(16):
            mine = np.zeros(W.shape[1], np.float32)
            for row in W[wave::16]:
                mine = mine + row
            cols = cols + mine
        assert packed[base + 8 + l] == cols.max() * np.float32(1.001), l
        lines = np.concatenate([W.max(0), W.max(1)])
        spread = lines[lines > 0].min() < W.max() * np.float32(2.0 ** -10)
        assert packed[base + l] == (np.inf if spread else W.max()), l
        assert spread == (l == 3)   # columns of 4 weights: both forms of the rule
