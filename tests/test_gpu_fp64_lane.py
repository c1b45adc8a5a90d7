"""The FP64 sum with one point per lane -- few wavevectors or many points, and
per-realization directions -- at its edges: blocks of 256 points, realization
chunks of 1 .. 16, sums of more than one flush of 32 wavevectors, the sine's range
inside a wave, masks, points that are not finite; against the oracle.

Tolerance 1e-12 of the field's rms, the argument's rounding (|t| 2^-53 ~ 2e-14 at
|t| ~ 200).  Far points: one dimension and zero phases, so that both sides form
the same argument."""
import numpy as np
import pytest

import randomfield_amd as R
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.sqrt(np.mean((a - b) ** 2)) / np.sqrt(np.mean(b ** 2)))


def _pick(N, rng):
    return np.unique(np.r_[0, 63, 64, 255, 256, N - 257, N - 1, rng.integers(0, N, 300)])


@pytest.mark.parametrize("xr", [(4.0,), (60.0,), (2.0, 3.0), (1.5, 1.0, 1.2)])
@pytest.mark.parametrize("N,Nmc", [(40000, 1), (40192, 2), (40193, 3), (40447, 7), (40448, 16), (40449, 17)])
@pytest.mark.parametrize("mode", [R.FIXED, R.REF_COMPAT])
def test_shared_table(ctx, xr, N, Nmc, mode):
    d = len(xr)
    rng = np.random.default_rng(N + Nmc)
    x = rng.random((N, d)) * np.array(xr)
    p = R.make_params(nDim=d, method=R.SHINOZUKA, mode=mode, form=R.FORM_FP64, Nmc=Nmc, xRange=xr)
    _, phU = R.reference_draws(p, R.reference_seed(5))
    got = R.generate(ctx, p, x, None, phU, dtype=np.float64)
    s = _pick(N, rng)
    po = O.make_plan(d, O.SHINOZUKA, mode, list(xr))
    k = O.kpoints(po)
    ref = O.shinozuka(po, x[s], k, O.skvec(po, k), phU)
    assert np.isfinite(got).all() and _rel(got[:, s], ref) <= 1e-12


@pytest.mark.parametrize("nDim", [2, 3])
@pytest.mark.parametrize("N,Nmc", [(30000, 2), (9001, 5), (4095, 17)])
def test_per_realization_directions(ctx, nDim, N, Nmc):
    rng = np.random.default_rng(N)
    x = rng.random((N, nDim)) * 4.0
    p = R.make_params(nDim=nDim, method=R.ISOTROPIC, mode=R.FIXED, form=R.FORM_FP64, Nmc=Nmc, xRange=[4.0] * nDim)
    _, U = R.reference_draws(p, R.reference_seed(6))
    got = R.generate(ctx, p, x, None, U, dtype=np.float64)
    s = _pick(N, rng)
    po = O.make_plan(nDim, O.ISOTROPIC, O.FIXED, [4.0] * nDim)
    k = O.kpoints(po)
    ref = O.isotropic(po, x[s], k, O.skvec(po, k), U)
    assert np.isfinite(got).all() and _rel(got[:, s], ref) <= 1e-12


@pytest.mark.parametrize("big", [1e6, 3e8, 1e10, 1e13])
def test_large_arguments(ctx, big):
    rng = np.random.default_rng(1)
    x = (rng.random((20000, 1)) - 0.5) * 3.0
    x[70:90] *= big                                  # inside one wave, and a whole wave
    x[128:192] *= big
    p = R.make_params(nDim=1, method=R.SHINOZUKA, mode=R.FIXED, form=R.FORM_FP64, Nmc=2, xRange=(4.0,))
    phU = np.zeros((2, R.plan_spectrum(p).nPhaseUniform))
    got = R.generate(ctx, p, x, None, phU, dtype=np.float64)
    po = O.make_plan(1, O.SHINOZUKA, O.FIXED, [4.0])
    k = O.kpoints(po)
    ref = O.shinozuka(po, x[:400], k, O.skvec(po, k), phU)
    assert _rel(got[:, :400], ref) <= 1e-12


def test_masked_and_not_finite(ctx):
    x = np.random.default_rng(2).random((20000, 1)) * 4.0
    calc = np.array([1, 0, 1], dtype=np.uint8)
    p = R.make_params(nDim=1, method=R.SHINOZUKA, mode=R.FIXED, form=R.FORM_FP64, Nmc=3, xRange=(4.0,))
    _, phU = R.reference_draws(p, R.reference_seed(5))
    ok = R.generate(ctx, p, x, None, phU, calc, dtype=np.float64)
    x2 = x.copy()
    x2[3, 0], x2[19999, 0] = np.nan, np.inf
    got = R.generate(ctx, p, x2, None, phU, calc, dtype=np.float64)
    assert np.all(got[1] == 0.0) and np.all(ok[1] == 0.0)
    keep = np.ones(20000, bool)
    keep[[3, 19999]] = False
    assert np.isnan(got[[0, 2]][:, ~keep]).all()
    assert _rel(got[[0, 2]][:, keep], ok[[0, 2]][:, keep]) <= 1e-14
