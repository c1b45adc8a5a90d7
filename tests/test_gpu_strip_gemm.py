"""The grid form's strip GEMMs at their edges: table axes of one entry, whole
and broken 32-entry tiles, more than one group of five tiles; lines below, at and
past a block's 128; K of whole and broken 8-entry steps.

Tolerance: operands carry 22 bits (2^-22 = 2.4e-7 per contraction), the FP32
tables and sums of up to ~100 terms ~5e-7 more, in three contractions: 3e-6."""
import numpy as np
import pytest

import randomfield_amd as R
from oracle import oracle as O
from randomfield_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nstep,step", [
    ((1, 1), (0.5, 0.5)), ((2, 33), (0.5, 0.3)), ((32, 4), (0.25, 0.5)), ((161, 3), (0.1, 0.5)),
    ((4, 330), (0.5, 0.05)), ((127, 129), (0.1, 0.1)),
    ((1, 40, 2), (0.5, 0.2, 0.5)), ((33, 31, 5), (0.2, 0.2, 0.5)), ((8, 161, 4), (0.4, 0.1, 0.5)),
    ((4, 16, 170), (0.5, 0.4, 0.1)), ((64, 2, 32), (0.25, 0.5, 0.25)),
])
def test_strip_edges(ctx, nstep, step):
    import torch
    d, Nmc = len(nstep), 2
    ext = [max(nstep[a] - 1, 1) * step[a] for a in range(d)]
    p = R.make_params(nDim=d, method=R.SHINOZUKA, mode=R.FIXED, form=R.FORM_FP32, Nmc=Nmc, corrL=(1.0,) * d, xRange=ext)
    _, phU = R.reference_draws(p, R.reference_seed(3))
    plan = R.FieldPlan(ctx, p, None, phU)
    out = torch.empty((Nmc, int(np.prod(nstep))), dtype=torch.float64, device="cuda")
    plan.execute_grid((0.5,) * d, step, nstep, out)
    ctx.sync()
    po = O.make_plan(d, O.SHINOZUKA, O.FIXED, ext)
    k = O.kpoints(po)
    ref = O.shinozuka(po, W.grid_points(nstep, step, (0.5,) * d), k, O.skvec(po, k), phU)
    got = out.cpu().numpy()
    e = float(np.sqrt(np.mean((got - ref) ** 2) / np.mean(ref ** 2)))
    print(f"[parity] strip {nstep}: rel_rms={e:.3e}", flush=True)
    assert e <= 3e-6
    plan.close()


def test_batch_of_uneven_axes(ctx):
    """Fields whose table axes need different numbers of tiles share a
    launch; a first axis past five tiles takes the stored coefficients.  Every
    split of the table axes and every way of forming the coefficients gives the
    bits of the single calls."""
    import torch
    shapes = [(170, 5, 4), (20, 70, 33), (131, 8)]
    plans, outs, single = [], [], []
    for i, n in enumerate(shapes):
        d = len(n)
        st = (0.2,) * d
        pl = R.FieldPlan(ctx, R.make_params(nDim=d, method=R.SHINOZUKA, mode=R.FIXED, form=R.FORM_FP32, Nmc=2,
                                            corrL=(1.0,) * d, xRange=[(v - 1) * 0.2 for v in n], seed=50 + i))
        o = torch.empty((2, int(np.prod(n))), dtype=torch.float32, device="cuda")
        pl.execute_grid((0.0,) * d, st, n, o)
        ctx.sync()
        single.append(o.cpu().numpy().copy())
        plans.append(pl)
        outs.append(o)
    pad = lambda v: list(v) + [1] * (3 - len(v))
    b = R.GridBatch(ctx, plans, [[0.0] * 3] * 3, [[0.2] * 3] * 3, [pad(n) for n in shapes], outs, R.DTYPE_F32)
    for step in ("plain", "redraw", "tuned"):
        if step == "redraw":
            b.redraw(0)
        if step == "tuned":
            b.autotune()
        for o in outs:
            o.fill_(-1.0)
        b.execute()
        ctx.sync()
        for i, o in enumerate(outs):
            assert np.array_equal(o.cpu().numpy(), single[i]), (step, i)
    b.close()
    for pl in plans:
        pl.close()


@pytest.mark.parametrize("gn", [(2, 2), (33, 161), (5, 40, 9), (170, 3, 33)])
def test_real_operands(ctx, gn):
    """Method 4: single calls run on real operands, a batch on complex ones; K and
    axes of broken steps and tiles.  Bit for bit equal, and the FP64 oracle."""
    import torch
    d, Nmc, xs = len(gn), 3, 0.2
    ext = [(v - 1) * xs for v in gn]
    p = R.make_params(nDim=d, method=R.FFT, mode=R.FIXED, form=R.FORM_FP32, Nmc=Nmc, corrL=(1.0,) * d, xRange=ext, gridN=gn)
    u = np.random.default_rng(3).random((Nmc, 3 * int(np.prod(gn)) - 1))
    plan = R.FieldPlan(ctx, p, phU=u)
    out = [torch.empty((Nmc, int(np.prod(gn))), dtype=torch.float32, device="cuda") for _ in range(2)]
    plan.execute_grid([0.0] * d, [xs] * d, gn, out[0])
    pad = lambda v, f: list(v) + [f] * (3 - d)
    b = R.GridBatch(ctx, [plan], [[0.0] * 3], [pad([xs] * d, 1.0)], [pad(gn, 1)], [out[1]], R.DTYPE_F32)
    b.execute()
    ctx.sync()
    got = [o.cpu().numpy() for o in out]
    assert np.array_equal(got[0], got[1])
    po = O.fft_plan(d, ext, gn)
    ref = O.fft(po, O.skvec(po, O.kpoints(po)), u, [xs] * d, Nmc, None)
    e = float(np.sqrt(np.mean((got[0] - ref) ** 2) / np.mean(ref ** 2)))
    assert e <= 1e-5
    b.close()
    plan.close()


def test_wide_planes(ctx):
    """A plane of a million points stays on the strips (64 points against the oracle)."""
    import torch
    n, step = (1000, 1024, 2), (0.02, 0.02, 0.5)
    ext = [(n[a] - 1) * step[a] for a in range(3)]
    p = R.make_params(nDim=3, method=R.SHINOZUKA, mode=R.FIXED, form=R.FORM_FP32, Nmc=1, corrL=(1.0,) * 3, xRange=ext)
    _, phU = R.reference_draws(p, R.reference_seed(3))
    plan = R.FieldPlan(ctx, p, None, phU)
    out = torch.empty((1, int(np.prod(n))), dtype=torch.float32, device="cuda")
    plan.execute_grid((0.0,) * 3, step, n, out)
    ctx.sync()
    pick = np.unique(np.r_[0, np.prod(n) - 1, np.random.default_rng(1).integers(0, np.prod(n), 62)])
    x = np.stack([pick % n[0] * step[0], pick // n[0] % n[1] * step[1], pick // (n[0] * n[1]) * step[2]], 1)
    po = O.make_plan(3, O.SHINOZUKA, O.FIXED, ext)
    k = O.kpoints(po)
    ref = O.shinozuka(po, x, k, O.skvec(po, k), phU)
    got = out.cpu().numpy()[:, pick]
    assert float(np.sqrt(np.mean((got - ref) ** 2) / np.mean(ref ** 2))) <= 3e-6
    plan.close()
