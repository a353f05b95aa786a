"""The inverse-CDF ops give a wavefront a row: bit-equal to the oracle's walk
at the edges of its 64-lane passes and 256 or 1,024 staged bins, and on the rows that
the closed form does not cover."""
import ctypes

import numpy as np
import pytest
import torch

import nsvf_oracle as O
from nsvf_amd import _ext, _lib, clib

pytestmark = pytest.mark.gpu


def rows(N, P, seed, full=0.2, mean_steps=70.0):
    """N rows of up to P bins: increasing depths, some rows full, some bins
    without probability."""
    rng = np.random.default_rng(seed)
    pv = np.where(rng.random(N) < full, P, rng.integers(1, P + 1, N))
    valid = np.arange(P) < pv[:, None]
    gap = rng.uniform(0.01, 0.2, (N, 2 * P)).astype(np.float32).cumsum(1)
    lo = np.where(valid, gap[:, 0::2], 10000).astype(np.float32)
    hi = np.where(valid, gap[:, 1::2], 10000).astype(np.float32)
    pr = np.where(valid & (rng.random((N, P)) < 0.9), hi - lo, 0).astype(np.float32)
    pr[:, 0] = np.where(valid[:, 0], hi[:, 0] - lo[:, 0], 0)
    pr /= pr.sum(1, keepdims=True)
    idx = np.where(valid, rng.integers(0, 5000, (N, P)), -1).astype(np.int32)
    steps = rng.uniform(0.5, 2 * mean_steps, N).astype(np.float32)
    steps[::7] = np.ceil(steps[::7])
    return idx, lo, hi, pr, steps


def spoil(kind, a, noise):
    idx, lo, hi, pr, steps = a
    rng = np.random.default_rng(1)
    if kind == "negative":
        pr[::3, 1] = -0.01
    elif kind == "nan":
        pr[::5, 0] = np.nan
    elif kind == "short":        # the probabilities end before the last steps
        pr *= np.float32(0.6)
    elif kind == "long":
        pr *= np.float32(1.4)
    elif kind == "noise_ends":
        noise[:] = rng.integers(0, 2, noise.shape)
    elif kind == "noise_out":
        noise[::4] = rng.uniform(-2, 3, noise[::4].shape)
    elif kind == "no_steps":
        steps[::3], steps[1::3] = 0, -4
    elif kind == "no_bins":
        idx[::3] = -1
    elif kind == "pads":         # pads with a depth range of their own
        lo[idx == -1], hi[idx == -1] = 1.0, 2.0


CASES = [(p, "plain") for p in (1, 2, 63, 64, 65, 128, 255, 256, 257, 300, 1024, 1025)] + [
    (20, k) for k in ("negative", "nan", "short", "long", "noise_ends", "noise_out", "no_steps",
                      "no_bins", "pads")]


@pytest.mark.parametrize("compat", [True, False])
@pytest.mark.parametrize("P,kind", CASES)
def test_rows_match_the_walk(device, P, kind, compat):
    N = 203
    a = rows(N, P, P)
    S = int(np.ceil(a[4]).max()) + P + 1
    noise = np.random.default_rng(2).uniform(0.001, 0.999, (N, S)).astype(np.float32)
    spoil(kind, a, noise)
    t = [torch.from_numpy(x).to(device) for x in a]
    nz = torch.from_numpy(noise).to(device)
    for fixed in (-1.0, 0.013):
        ref = O.inverse_cdf_sampling_op(*(x[None] for x in a[:3]), noise[None], a[3][None],
                                        a[4][None], fixed, compat)
        got = _ext.inverse_cdf_sampling(*(x[None] for x in t[:3]), nz[None], t[3][None],
                                        t[4][None], fixed, compat=compat)
        for g, r in zip(got, ref):
            np.testing.assert_array_equal(g.cpu().numpy(), r)
        for n in (None, nz):
            ri, rd, rx, rs, _ = O.inverse_cdf_sampling(
                *a, fixed, n is None, None if n is None else noise[:, :rS(a)], compat)
            gi, gd, gx, gs, most = clib._icdf_rows(
                *t, fixed, None if n is None else nz[:, :rS(a)].contiguous(), rS(a), compat)
            assert gs == rs
            assert int(most) == max(int((gi != -1).sum(1).max()), 0)
            L = ri.shape[1]
            for g, r, pad in ((gi, ri, -1), (gd, rd, 0), (gx, rx, 0)):
                np.testing.assert_array_equal(g.cpu().numpy()[:, :L], r)
            assert bool((gi[:, L:] == -1).all())


def rS(a):
    return int(np.ceil(a[4]).max()) + a[0].shape[1]


@pytest.mark.parametrize("S", [1, 64, 100])
def test_full_rows_are_counted(device, S):
    """Fewer slots than samples: what fits is written, and flags[1] says that
    some did not, as the oracle's does."""
    N, P = 130, 40
    a = rows(N, P, 3)
    noise = np.random.default_rng(2).uniform(0.001, 0.999, (N, S)).astype(np.float32)
    ref = O.inverse_cdf_sampling_op(*(x[None] for x in a[:3]), noise[None], a[3][None],
                                    a[4][None], -1.0, True)
    t = [torch.from_numpy(x).to(device) for x in (*a, noise)]
    out = [torch.empty((N, S), dtype=d, device=device)
           for d in (torch.int32, torch.float32, torch.float32)]
    p = lambda x: ctypes.c_void_p(x.data_ptr())
    for count in (False, True):
        flags = torch.zeros(4, dtype=torch.int64, device=device)
        rc = _lib.lib().nsvf_inverse_cdf_sampling(
            *(p(x) for x in t[:3]), p(t[5]), p(t[3]), p(t[4]), 1, N, P, S, -1.0, 1,
            *(p(o) for o in out), p(flags) if count else None, None)
        assert rc == 0
        torch.cuda.synchronize()
        for g, r in zip(out, ref):
            np.testing.assert_array_equal(g.cpu().numpy(), r[0])
        if count:
            assert (int(flags[1]) > 0) == (int(ref[3][1]) > 0)
