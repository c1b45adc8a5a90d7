"""The FP64 point-wise sum at the sizes where it can go wrong: blocks of 16
points, chunks of 1 .. 16 realizations, 128 shares of the wavevectors, the
sine's range, masks; against the oracle.

Tolerance 1e-12 of the field's rms: the argument's rounding (|t| 2^-53 ~ 2e-14
at |t| ~ 200) dominates; where arguments are large the phases are zero and the
space one-dimensional, so both sides form the same argument.
"""
import numpy as np
import pytest

import randomfield_amd as R
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _field(nDim, method, mode, Nmc, x, xr, phU=None, calc=None):
    p = R.make_params(nDim=nDim, method=method, mode=mode, form=R.FORM_FP64, Nmc=Nmc, xRange=xr)
    if phU is None:
        _, phU = R.reference_draws(p, R.reference_seed(5))
    return p, phU


def _rel(a, b):
    return float(np.sqrt(np.mean((a - b) ** 2)) / np.sqrt(np.mean(b ** 2)))


@pytest.mark.parametrize("nDim", [1, 2, 3])
@pytest.mark.parametrize("N,Nmc", [(1, 1), (63, 2), (64, 3), (65, 5), (130, 16), (200, 17), (3, 33)])
@pytest.mark.parametrize("mode", [R.FIXED, R.REF_COMPAT])
def test_shared_table(ctx, nDim, N, Nmc, mode):
    xr = (4.0, 3.0, 2.5)[:nDim]
    x = np.random.default_rng(N + Nmc).random((N, nDim)) * np.array(xr)
    p, phU = _field(nDim, R.SHINOZUKA, mode, Nmc, x, xr)
    got = R.generate(ctx, p, x, None, phU, dtype=np.float64)
    po = O.make_plan(nDim, O.SHINOZUKA, mode, list(xr))
    k = O.kpoints(po)
    ref = O.shinozuka(po, x, k, O.skvec(po, k), phU)
    assert _rel(got, ref) <= 1e-12


@pytest.mark.parametrize("N", [15, 16, 17, 31, 33])
@pytest.mark.parametrize("Nmc", [1, 4, 16])
def test_block_edges(ctx, N, Nmc):
    xr = (4.0, 3.0, 2.5)
    x = np.random.default_rng(N).random((N, 3)) * np.array(xr)
    p, phU = _field(3, R.SHINOZUKA, R.FIXED, Nmc, x, xr)
    got = R.generate(ctx, p, x, None, phU, dtype=np.float64)
    po = O.make_plan(3, O.SHINOZUKA, O.FIXED, list(xr))
    k = O.kpoints(po)
    assert _rel(got, O.shinozuka(po, x, k, O.skvec(po, k), phU)) <= 1e-12


@pytest.mark.parametrize("big", [1e3, 1e6, 3e8, 1e10, 1e13])
def test_large_arguments(ctx, big):
    """Both sides of the fast sine's range, one-dimensional, zero phases."""
    xr = (4.0,)
    x = (np.random.default_rng(1).random((100, 1)) - 0.5) * big
    x[:64] *= 1e-3                                   # a block of its own inside the range
    p = R.make_params(nDim=1, method=R.SHINOZUKA, mode=R.FIXED, form=R.FORM_FP64, Nmc=2, xRange=xr)
    phU = np.zeros((2, R.plan_spectrum(p).nPhaseUniform))
    got = R.generate(ctx, p, x, None, phU, dtype=np.float64)
    po = O.make_plan(1, O.SHINOZUKA, O.FIXED, list(xr))
    k = O.kpoints(po)
    ref = O.shinozuka(po, x, k, O.skvec(po, k), phU)
    assert _rel(got, ref) <= 1e-12


def test_masked_and_not_finite(ctx):
    """A masked realization is zero everywhere; a point that is not finite
    gives NaN in the others and leaves its neighbours alone."""
    xr = (4.0, 3.0)
    x = np.random.default_rng(2).random((70, 2)) * np.array(xr)
    calc = np.array([1, 0, 1], dtype=np.uint8)
    p, phU = _field(2, R.SHINOZUKA, R.FIXED, 3, x, xr)
    ok = R.generate(ctx, p, x, None, phU, calc, dtype=np.float64)
    x2 = x.copy()
    x2[3, 0], x2[66, 1] = np.nan, np.inf
    got = R.generate(ctx, p, x2, None, phU, calc, dtype=np.float64)
    assert np.all(got[1] == 0.0) and np.all(ok[1] == 0.0)
    keep = np.ones(70, bool)
    keep[[3, 66]] = False
    assert np.isnan(got[[0, 2]][:, ~keep]).all()
    assert _rel(got[[0, 2]][:, keep], ok[[0, 2]][:, keep]) <= 1e-14
