"""Statistics kernels at the sizes where they can go wrong: the matrix-core
correlation (tiles of 64 positions, 16 lines per turn, the sweep for axes it
does not take) against the oracle, and the moments with rows on and off
16-byte boundaries.

Tolerance: a lag is a mean of N products of magnitude ~1 in FP64; summed in any
order its error is below N eps max|v|^2 / N ~ 16 * 2.2e-16 * log2(N) < 1e-13 for
the values here, and the oracle's sequential sum is off by at most N eps ~ 1e-11
of the rms in the worst case, 1e-13 typically: 1e-12 absolute.
"""
import numpy as np
import pytest

import randomfield_amd as R
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("nstep", [(64, 16), (16, 65), (15, 17), (63, 2, 9), (66, 20, 17), (129, 5, 130), (2, 16, 1),
                                   (3, 191, 4), (2048, 17), (2049, 16), (257, 16, 2)])
def test_corr_edges_match_oracle(ctx, dtype, nstep):
    import torch
    rng = np.random.default_rng(sum(nstep))
    N = int(np.prod(nstep))
    f = rng.normal(0.4, 2.0, (2, N)).astype(dtype)
    u = f[1].astype(np.float64)
    avg, sd = float(u.mean()), float(u.std())
    got, cl = R.corr(ctx, torch.from_numpy(f).cuda(), R.DTYPE_F64 if dtype == np.float64 else R.DTYPE_F32, nstep,
                     [0.5] * len(nstep), avg, sd, 1)
    ref = O.corr(u, nstep, avg, sd)
    for a in range(len(nstep)):
        assert len(got[a]) == nstep[a] // 2
        assert np.allclose(got[a], ref[a], rtol=0.0, atol=1e-12), (a, np.abs(got[a] - ref[a]).max())


@pytest.mark.parametrize("nstep", [(1100, 16, 4), (5, 700, 40), (3, 65, 1500)])
def test_corr_axes_of_unequal_length(ctx, nstep):
    """A long axis of many tile pairs beside short ones of many lines, whose
    lines are dealt to more blocks than an even share per pair."""
    import torch
    f = np.random.default_rng(7).normal(0.4, 2.0, int(np.prod(nstep)))
    avg, sd = float(f.mean()), float(f.std())
    got, _ = R.corr(ctx, torch.from_numpy(f[None]).cuda(), R.DTYPE_F64, nstep, [0.5] * 3, avg, sd, 0)
    ref = O.corr(f, nstep, avg, sd)
    for a in range(3):
        assert len(got[a]) == nstep[a] // 2
        assert np.allclose(got[a], ref[a], rtol=0.0, atol=1e-12), (a, np.abs(got[a] - ref[a]).max())


def test_corr_not_finite(ctx):
    """A value that is not finite reaches every lag of its lines and only
    those sums: no lag of the field stays finite, as in the plain sum."""
    import torch
    nstep = (70, 20, 18)
    for bad in (np.nan, np.inf):
        f = np.random.default_rng(3).normal(size=int(np.prod(nstep)))
        f[1234] = bad
        got, _ = R.corr(ctx, torch.from_numpy(f[None]).cuda(), R.DTYPE_F64, nstep, [1.0] * 3, 0.0, 1.0, 0)
        for a in range(3):
            assert not np.isfinite(got[a]).any()
        if bad == np.inf:
            assert all(np.isposinf(got[a][0]) for a in range(3))


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("N,Nmc,off", [(1, 1, 0), (3, 5, 0), (1024, 2, 0), (1025, 3, 0), (4096, 1, 1), (99999, 4, 3),
                                       (300000, 300, 0), (10, 2500, 0)])
def test_moments_edges(ctx, dtype, N, Nmc, off):
    import torch
    g = torch.Generator().manual_seed(N + Nmc)
    flat = (torch.randn(N * Nmc + off, generator=g, dtype=torch.float64) * 2.0 + 0.5).to(getattr(torch, dtype))
    d = flat.cuda()[off:].reshape(Nmc, N)
    avg, sd, tot = R.stats(ctx, d, N, Nmc, R.DTYPE_F64 if dtype == "float64" else R.DTYPE_F32)
    ref = flat[off:].reshape(Nmc, N).double().numpy()
    assert np.allclose(avg, ref.mean(axis=1), rtol=0.0, atol=1e-12)
    var = (ref ** 2).mean(axis=1) - ref.mean(axis=1) ** 2
    assert np.allclose(np.nan_to_num(sd) ** 2, np.maximum(var, 0.0), rtol=0.0, atol=1e-11)
    assert np.allclose(tot[0], ref.mean(), rtol=0.0, atol=1e-12)
