"""Strip GEMMs of isotropic and method-4 grids with several table tiles per wave:
planes of 128 x 128 and enough realizations give every SIMD a strip, so that the
table axis is not split down to single tiles as on small grids; last axes of whole
and broken tiles and of more than one group of five.

Tolerance: operands carry 22 bits, FP32 tables and sums: 3e-6 over the ~300 terms of
an isotropic sum; method 4, whose tables reach 2 and whose sums are of up to 128
terms in three contractions, 1e-5."""
import numpy as np
import pytest

import randomfield_amd as R
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n2", [33, 64, 97, 160, 170])
def test_isotropic(ctx, n2):
    import torch
    n, step, Nmc = (128, 128, n2), (0.05, 0.05, 0.05), 2
    ext = [(v - 1) * 0.05 for v in n]
    p = R.make_params(nDim=3, method=R.ISOTROPIC, mode=R.FIXED, form=R.FORM_FP32, Nmc=Nmc, corrL=(1.0,) * 3, xRange=ext)
    _, U = R.reference_draws(p, R.reference_seed(5))
    plan = R.FieldPlan(ctx, p, None, U)
    N = int(np.prod(n))
    out = torch.full((Nmc, N), float("nan"), dtype=torch.float32, device="cuda")
    plan.execute_grid((0.5, -1.0, 0.0), step, n, out)
    ctx.sync()
    plan.close()
    got = out.cpu().numpy()
    assert np.isfinite(got).all()
    # whole columns of the last axis, and points at random
    pick = np.unique(np.r_[np.arange(0, N, 128 * 128) + 37, np.arange(0, N, 128 * 128) + 16383,
                           np.random.default_rng(1).integers(0, N, 500), N - 1])
    x = np.stack([0.5 + pick % 128 * 0.05, -1.0 + pick // 128 % 128 * 0.05, pick // 16384 * 0.05], 1)
    po = O.make_plan(3, O.ISOTROPIC, O.FIXED, ext)
    k = O.kpoints(po)
    ref = O.isotropic(po, x, k, O.skvec(po, k), U)
    assert float(np.sqrt(np.mean((got[:, pick] - ref) ** 2) / np.mean(ref ** 2))) <= 3e-6


@pytest.mark.parametrize("gn", [(128, 128, 97), (100, 130, 128), (128, 65, 170)])
def test_real_operands(ctx, gn):
    """Against the FP64 oracle, and bit for bit the same from a batch, whose
    operands are complex."""
    import torch
    Nmc, xs = 3, 0.1
    ext = [(v - 1) * xs for v in gn]
    p = R.make_params(nDim=3, method=R.FFT, mode=R.FIXED, form=R.FORM_FP32, Nmc=Nmc, corrL=(1.0,) * 3, xRange=ext, gridN=gn)
    u = np.random.default_rng(3).random((Nmc, 3 * int(np.prod(gn)) - 1))
    plan = R.FieldPlan(ctx, p, phU=u)
    out = [torch.full((Nmc, int(np.prod(gn))), float("nan"), dtype=torch.float32, device="cuda") for _ in range(2)]
    plan.execute_grid([0.0] * 3, [xs] * 3, gn, out[0])
    b = R.GridBatch(ctx, [plan], [[0.0] * 3], [[xs] * 3], [list(gn)], [out[1]], R.DTYPE_F32)
    b.execute()
    ctx.sync()
    b.close()
    plan.close()
    got = [o.cpu().numpy() for o in out]
    assert np.array_equal(got[0], got[1])
    po = O.fft_plan(3, ext, gn)
    ref = O.fft(po, O.skvec(po, O.kpoints(po)), u, [xs] * 3, Nmc, None)
    assert float(np.sqrt(np.mean((got[0] - ref) ** 2) / np.mean(ref ** 2))) <= 1e-5
