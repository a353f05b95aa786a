"""Rows of few slots are walked by a lane each: the same outputs as the oracle's
walk and as a wavefront per row, on both sides of the rule's edges."""
import ctypes

import numpy as np
import pytest
import torch

import nsvf_oracle as O
from nsvf_amd import _lib, clib
from test_gpu_icdf_rows import rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["plain", "no_bins", "negative"])
@pytest.mark.parametrize("S,P", [(2, 1), (4, 2), (8, 3), (9, 3)])
def test_narrow_rows_match_the_walk(device, S, P, kind):
    N = 403
    a = rows(N, P, 100 * S + P, mean_steps=(S - P) / 2)
    a[4][:] = np.minimum(a[4], S - P).astype(np.float32)
    a[4][0] = S - P
    if kind == "no_bins":
        a[0][::3] = -1
    elif kind == "negative":
        a[3][::3, P - 1] = -0.01
    noise = np.random.default_rng(3).uniform(0.001, 0.999, (N, S)).astype(np.float32)
    t = [torch.from_numpy(x).to(device) for x in a]
    for compat in (True, False):
        for n in (None, noise):
            ref = O.inverse_cdf_sampling(*a, -1.0, n is None, n, compat)
            assert ref[3] == S
            got = clib._icdf_rows(*t, -1.0, None if n is None else torch.from_numpy(n).to(device),
                                  S, compat)
            L = ref[0].shape[1]
            for g, r in zip(got[:3], ref[:3]):
                np.testing.assert_array_equal(g.cpu().numpy()[:, :L], r)
            assert int(got[4]) == int((got[0] != -1).sum(1).max())
            assert bool((got[0][:, L:] == -1).all())


@pytest.mark.parametrize("N", [(1 << 16) - 1, 1 << 16, (1 << 16) + 1])
@pytest.mark.parametrize("S", [16, 24, 25])
def test_many_narrow_rows(device, N, S):
    P = 5
    a = rows(N, P, S, mean_steps=(S - P - 2) / 2)
    a[4][:] = np.minimum(a[4], S - 2 * P).astype(np.float32)
    t = [torch.from_numpy(x).to(device) for x in a]
    got = clib._icdf_rows(*t, -1.0, None, S, True)
    wide = clib._icdf_rows(*t, -1.0, None, 64, True)   # a wavefront per row
    assert bool((wide[0][:, S:] == -1).all()) and int(got[4]) == int(wide[4])
    for g, w in zip(got[:3], wide[:3]):
        assert torch.equal(g, w[:, :S])


@pytest.mark.parametrize("S", [3, 8])
def test_full_narrow_rows_are_counted(device, S):
    N, P = 130, 10
    a = rows(N, P, 3)
    noise = np.random.default_rng(2).uniform(0.001, 0.999, (N, S)).astype(np.float32)
    ref = O.inverse_cdf_sampling_op(*(x[None] for x in a[:3]), noise[None], a[3][None],
                                    a[4][None], -1.0, True)
    t = [torch.from_numpy(x).to(device) for x in (*a, noise)]
    out = [torch.empty((N, S), dtype=d, device=device)
           for d in (torch.int32, torch.float32, torch.float32)]
    p = lambda x: ctypes.c_void_p(x.data_ptr())
    flags = torch.zeros(4, dtype=torch.int64, device=device)
    assert _lib.lib().nsvf_inverse_cdf_sampling(
        *(p(x) for x in t[:3]), p(t[5]), p(t[3]), p(t[4]), 1, N, P, S, -1.0, 1,
        *(p(o) for o in out), p(flags), None) == 0
    torch.cuda.synchronize()
    for g, r in zip(out, ref):
        np.testing.assert_array_equal(g.cpu().numpy(), r[0])
    assert int(flags[1]) > 0 and int(ref[3][1]) > 0


@pytest.mark.parametrize("S", [40, 41])
def test_counted_rows(device, S):
    """The same outputs with and without counting, in the forms that each takes."""
    N, P = 1 << 16, 6
    a = rows(N, P, S, mean_steps=(S - P) / 2)
    a[4][:] = np.minimum(a[4], S - 2).astype(np.float32)
    a[4][::50] = S - 0.5                      # as many steps as slots: some are dropped
    noise = torch.rand(N, S, generator=torch.Generator().manual_seed(1)).clamp_(0.001, 0.999)
    t = [torch.from_numpy(x).to(device) for x in a] + [noise.to(device)]
    p = lambda x: ctypes.c_void_p(x.data_ptr())
    outs = []
    for count in (False, True):
        flags = torch.zeros(4, dtype=torch.int64, device=device)
        out = [torch.empty((N, S), dtype=d, device=device)
               for d in (torch.int32, torch.float32, torch.float32)]
        assert _lib.lib().nsvf_inverse_cdf_sampling(
            *(p(x) for x in t[:3]), p(t[5]), p(t[3]), p(t[4]), 1, N, P, S, -1.0, 1,
            *(p(o) for o in out), p(flags) if count else None, None) == 0
        torch.cuda.synchronize()
        outs.append(out)
    assert int(flags[1]) > 0
    for x, y in zip(*outs):
        assert torch.equal(x, y)
