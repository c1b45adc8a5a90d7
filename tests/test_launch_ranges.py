"""Fields of more points than one grid of work-items holds (2^32): the kernels
that give a point several work-items launch them in ranges.

FP64 with the wavevectors dealt to shares (many wavevectors): 32 work-items per
point, the line at 134,217,712 points; with one point per lane no line is near.
The product form on a lattice whose per-axis tables only fit 128 points per block:
8 per point, the line at 536,870,784.  Points beside the line and at both ends
against FP64 torch on the device; tolerances: the argument's rounding (|t| 2^-53,
6e-12 at the long lattice's |t| ~ 5e4), the FP16 form's 4e-6.
"""
import math
import shutil
import subprocess
from pathlib import Path

import pytest

import randomfield_amd as R

ROOT = Path(__file__).resolve().parent.parent


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_block_ranges(tmp_path):
    exe = tmp_path / "ranges_test"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-o", str(exe),
                    str(ROOT / "tests" / "cpp" / "ranges_test.cpp")], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True)
    assert "ranges ok" in out.stdout


def _sum64(x, k, S, U, ampMult):
    """ampMult sum_j sqrt(S_j) cos(k_j.x + 2 pi U_rj) of a few points, FP64."""
    import torch
    t = x @ torch.from_numpy(k).cuda().T
    ph = 2.0 * 3.1415926535898 * torch.from_numpy(U).cuda()
    a = torch.from_numpy(S).cuda().sqrt()
    return ampMult * torch.stack([(a * torch.cos(t + p)).sum(1) for p in ph])


@pytest.mark.gpu
@pytest.mark.parametrize("form,xr,Nmc,line,tol", [(R.FORM_FP64, (9000.0,), 4, 134217712, 2e-11),
                                                  (R.FORM_FP64, (200.0,), 1, 134217712, 1e-12),
                                                  (R.FORM_MFMA_F16, (38.0, 0.9), 1, 536870784, 4e-6)])
def test_more_work_items_than_a_grid(ctx, form, xr, Nmc, line, tol):
    import torch
    d, N = len(xr), line + 77
    p = R.make_params(nDim=d, method=R.SHINOZUKA, mode=R.FIXED, form=form, Nmc=Nmc, xRange=list(xr))
    _, phU = R.reference_draws(p, R.reference_seed(2))
    plan = R.FieldPlan(ctx, p, None, phU)
    x = torch.rand((N, d), dtype=torch.float64, device="cuda",
                   generator=torch.Generator(device="cuda").manual_seed(4))
    for a in range(d):
        x[:, a] *= xr[a]
    f64 = form == R.FORM_FP64
    out = torch.full((Nmc, N), math.nan, dtype=torch.float64 if f64 else torch.float32, device="cuda")
    torch.cuda.synchronize()
    plan.execute(x, out)
    ctx.sync()
    info = plan.info
    plan.close()
    assert bool(torch.isfinite(out).all())
    i = torch.cat([torch.arange(300), torch.arange(line - 300, N)]).cuda()
    k, S = R.spectrum_tables(p)
    ref = _sum64(x[i], k, S, phU, info.ampMult)
    err = (out[:, i].double() - ref).square().mean().sqrt() / ref.square().mean().sqrt()
    assert float(err) <= tol
