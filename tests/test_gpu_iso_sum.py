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


def _plan(nDim, Nmc, xr=4.0):
    p = R.make_params(nDim=nDim, method=R.ISOTROPIC, mode=R.FIXED, form=R.FORM_FP32, Nmc=Nmc, xRange=[xr] * nDim)
    return p, R.reference_draws(p, R.reference_seed(3))[1]


def _sampled(ctx, nDim, N, Nmc, far=(), bad=(), xr=4.0):
    """Error of a field too large for the oracle, at the first and last points,
    around its blocks' edges, at `far` (moved 1e6 away) and at random; `bad`
    points are NaN and have to stay the only ones."""
    import torch
    rng = np.random.default_rng(N + Nmc)
    x = rng.random((N, nDim)) * xr
    x[list(far)] += 1e6
    x[list(bad), 0] = np.nan
    p, phU = _plan(nDim, Nmc, xr)
    plan = R.FieldPlan(ctx, p, None, phU)
    out = torch.full((Nmc, N), 7.0, dtype=torch.float32, device="cuda")
    plan.execute(torch.from_numpy(x).cuda(), out)
    ctx.sync()
    plan.close()
    got = out.cpu().numpy()
    nan = np.zeros(N, bool)
    nan[list(bad)] = True
    assert np.isnan(got[:, nan]).all() and np.isfinite(got[:, ~nan]).all()
    s = np.unique(np.r_[np.arange(70), np.arange(250, 262), np.arange(N - 300, N), np.array(far, dtype=int),
                        rng.integers(0, N, 300)])
    s = s[~nan[s]]
    po = O.make_plan(nDim, O.ISOTROPIC, O.FIXED, [xr] * nDim)
    k = O.kpoints(po)
    ref = O.isotropic(po, np.ascontiguousarray(x[s]), k, O.skvec(po, k), phU)
    return float(np.sqrt(np.mean((got[:, s] - ref) ** 2) / np.mean(ref ** 2)))


@pytest.mark.parametrize("nDim,N,Nmc", [(2, 98303, 16), (2, 98304, 9), (2, 131072, 16), (2, 131073, 16), (2, 98369, 17),
                                        (2, 262401, 13), (3, 294911, 16), (3, 294912, 9), (3, 147457, 20), (3, 300001, 16)])
def test_one_point_per_lane(ctx, nDim, N, Nmc):
    """Both sides of the lines between the FMA and the matrix-core form."""
    assert _sampled(ctx, nDim, N, Nmc, far=(5, 64, 65, N - 1), bad=(3, N - 2)) <= 3e-6


@pytest.mark.parametrize("nDim", [2, 3])
def test_both_forms_give_the_same_bits(ctx, nDim):
    """The FMA form of a large field against the matrix-core form of its first
    points, far ones among them."""
    import torch
    N, n, Nmc = 300000, 20000, 19
    x = torch.rand((N, nDim), dtype=torch.float64, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1)) * 4
    x[100:140] *= 1e5
    p, phU = _plan(nDim, Nmc)
    plan = R.FieldPlan(ctx, p, None, phU)
    big = torch.empty((Nmc, N), dtype=torch.float32, device="cuda")
    small = torch.empty((Nmc, n), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    plan.execute(x, big)
    plan.execute(x[:n].contiguous(), small)
    ctx.sync()
    plan.close()
    assert torch.equal(big[:, :64], small[:, :64]) and torch.equal(big[:, 192:n], small[:, 192:])


@pytest.mark.parametrize("N", [2 ** 20 - 1, 2 ** 20 + 77])
@pytest.mark.parametrize("nDim,Nmc", [(3, 1), (3, 5), (2, 3), (3, 8)])
def test_waves_of_64_points(ctx, nDim, N, Nmc):
    """From 1,048,576 points a wave of the matrix-core form takes 64 points: a
    ragged end, rows of 2 .. 16 wavevectors, far points in one wave and in the last;
    the first case is just below."""
    assert _sampled(ctx, nDim, N, Nmc, far=(64, 65, 66, 130, N - 1), bad=(3, N - 70)) <= 3e-6
