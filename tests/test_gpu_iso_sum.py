"""The direct isotropic FP32 sum at its edges: realization counts around the
16-row packing (1 .. 16 wavevectors per row block, several chunks), point counts
around a wave's 32 and a block's 128, 2-D and 3-D, and arguments past 2^19
revolutions, where the fixed-point reduction gives way to the FP64 one.

Tolerance: arguments good to 2^-24 revolution (4e-7 rad), the hardware cosine to
~5e-7, FP32 sums of up to ~120 terms: 3e-6 of the field's rms; far points add
2^-53 * 2^25 revolutions * 2 pi = 2e-8."""
import numpy as np
import pytest

import randomfield_amd as R
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _run(ctx, nDim, N, Nmc, far=0.0, xr=4.0, dtype="float32"):
    import torch
    rng = np.random.default_rng(N + Nmc)
    corrL = (0.5, 2.0, 1.5)[:nDim]
    x = rng.random((N, nDim)) * xr * np.array(corrL)
    x[: (N + 1) // 2] += far
    p = R.make_params(nDim=nDim, method=R.ISOTROPIC, mode=R.FIXED, form=R.FORM_FP32, Nmc=Nmc, corrL=corrL,
                      xRange=[xr * c for c in corrL])
    _, phU = R.reference_draws(p, R.reference_seed(3))
    plan = R.FieldPlan(ctx, p, None, phU)
    out = torch.full((Nmc, N), 7.0, dtype=getattr(torch, dtype), device="cuda")
    plan.execute(torch.from_numpy(x).cuda(), out)
    ctx.sync()
    plan.close()
    po = O.make_plan(nDim, O.ISOTROPIC, O.FIXED, [xr] * nDim)
    k = O.kpoints(po)
    ref = O.isotropic(po, x / np.array(corrL), k, O.skvec(po, k), phU)
    got = out.cpu().numpy()
    return float(np.sqrt(np.mean((got - ref) ** 2) / np.mean(ref ** 2)))


@pytest.mark.parametrize("nDim", [2, 3])
@pytest.mark.parametrize("N,Nmc", [(1, 1), (31, 2), (32, 3), (33, 5), (127, 8), (128, 9), (129, 16), (257, 17), (100, 33)])
def test_edges(ctx, nDim, N, Nmc):
    assert _run(ctx, nDim, N, Nmc) <= 3e-6


@pytest.mark.parametrize("far", [1e5, 1e7])
@pytest.mark.parametrize("nDim", [2, 3])
def test_far_points(ctx, nDim, far):
    assert _run(ctx, nDim, 200, 6, far=far) <= 3e-6


def test_fp64_output(ctx):
    assert _run(ctx, 3, 150, 4, dtype="float64") <= 3e-6
