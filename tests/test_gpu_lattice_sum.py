"""The product form of the Shinozuka sum on points (FP16 / BF16 matrix-core
forms) at the sizes where it can go wrong: odd lattice axes, blocks of 128 and
256 points and the line between them, tiles of 32 realizations, lattices too
wide for it; against the FP64 oracle.

Tolerance: the FP16 hi/lo operands carry 22 bits, the per-axis sines ~2^-23, the
two-level FP32 sums ~4e-7 of the field's rms: 2e-6.  BF16 hi/lo: 16 bits, 4e-5.
"""
import numpy as np
import pytest

import randomfield_amd as R
from oracle import oracle as O

pytestmark = pytest.mark.gpu
TOL = {R.FORM_MFMA_F16: 2e-6, R.FORM_MFMA_BF16: 4e-5}


def _run(ctx, form, xr, N, Nmc, sample=None, mode=R.FIXED, dtype="float32", margi=R.FOM_NONE):
    import torch
    d = len(xr)
    corrL = (0.5, 2.0, 1.5)[:d]
    rng = np.random.default_rng(N + Nmc)
    x = rng.random((N, d)) * (np.array(xr) * np.array(corrL))
    p = R.make_params(nDim=d, method=R.SHINOZUKA, mode=mode, form=form, Nmc=Nmc, corrL=corrL, margiFirst=margi,
                      fieldAvg=1.0, fieldVar=0.25, xRange=[a * c for a, c in zip(xr, corrL)])
    _, phU = R.reference_draws(p, R.reference_seed(3))
    plan = R.FieldPlan(ctx, p, None, phU)
    out = torch.full((Nmc, N), 7.0, dtype=getattr(torch, dtype), device="cuda")
    plan.execute(torch.from_numpy(x).cuda(), out)
    ctx.sync()
    plan.close()
    s = slice(None) if sample is None else np.unique(np.r_[0, N - 1, rng.integers(0, N, sample)])
    po = O.make_plan(d, O.SHINOZUKA, O.FIXED, list(xr))
    k = O.kpoints(po)
    ref = O.shinozuka(po, (x / np.array(corrL))[s], k, O.skvec(po, k), phU)
    if margi != R.FOM_NONE:
        ref = O.marginal(margi, 1.0, 0.25, ref)
    got = out.cpu().numpy().astype(np.float64)
    assert np.isfinite(got).all()
    got = got[:, s]
    return float(np.sqrt(np.mean((got - ref) ** 2)) / np.sqrt(np.mean(ref ** 2)))


@pytest.mark.parametrize("form", [R.FORM_MFMA_F16, R.FORM_MFMA_BF16])
@pytest.mark.parametrize("xr,N,Nmc", [((3.1, 2.2, 4.3), 1, 1), ((3.1, 3.9, 2.2), 127, 32), ((2.2, 3.1, 3.9), 129, 33),
                                      ((0.7, 5.0, 0.7), 128, 65), ((6.0, 0.7, 1.5), 300, 97), ((5.0, 0.7), 31, 5),
                                      ((0.7, 9.0), 257, 70), ((8.3, 7.7), 128, 300), ((12.0, 3.0), 500, 64)])
def test_edges(ctx, form, xr, N, Nmc):
    assert _run(ctx, form, xr, N, Nmc) <= TOL[form]


@pytest.mark.parametrize("N", [32768, 32769])
@pytest.mark.parametrize("Nmc", [4, 40])
def test_both_block_shapes(ctx, N, Nmc):
    assert _run(ctx, R.FORM_MFMA_F16, (3.1, 2.2, 3.9), N, Nmc, sample=200) <= TOL[R.FORM_MFMA_F16]


@pytest.mark.parametrize("xr", [(36.5, 36.5), (37.5, 37.5), (60.0, 30.0), (70.0, 3.0)])
@pytest.mark.parametrize("N", [200, 33000])
def test_wide_lattices(ctx, xr, N):
    """Tables that just fit, fit for 128 points only, or do not fit (the
    general form)."""
    assert _run(ctx, R.FORM_MFMA_F16, xr, N, 3, sample=100) <= 4e-6


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("margi", [R.FOM_GAUSSIAN, R.FOM_LOGNORMAL])
def test_marginals(ctx, dtype, margi):
    assert _run(ctx, R.FORM_MFMA_F16, (3.1, 2.2, 3.9), 200, 6, dtype=dtype, margi=margi) <= TOL[R.FORM_MFMA_F16]


@pytest.mark.parametrize("xr,Nmc", [((2.2, 1.5, 2.2), 129), ((3.1, 3.9), 65)])
@pytest.mark.parametrize("N", [32768, 32769])
def test_many_realizations(ctx, xr, N, Nmc):
    """Small fields keep the product form, larger ones of many realizations take
    the general form (its tolerance: hardware sines, one-level FP32 sums)."""
    assert _run(ctx, R.FORM_MFMA_F16, xr, N, Nmc, sample=100) <= 1e-5
