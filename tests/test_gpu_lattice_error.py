"""The product form of the Shinozuka sum is no further from 64 bits than the
general matrix-core form of the same operand type.

The general form is reached by a plan of 129 realizations on more than 32,768
points; its first 32 realizations are those of the plan under test (same device
stream), on the same points.  The bound is the general form's own error, measured
beside it against the FP64 form."""
import pytest

import randomfield_amd as R

pytestmark = pytest.mark.gpu
NBIG, NR = 33000, 32


def _field(ctx, form, xr, Nmc, x, dtype):
    import torch
    p = R.make_params(nDim=len(xr), method=R.SHINOZUKA, mode=R.FIXED, form=form, Nmc=Nmc, xRange=xr, seed=3)
    plan = R.FieldPlan(ctx, p)
    out = torch.empty((Nmc, x.shape[0]), dtype=dtype, device="cuda")
    torch.cuda.synchronize()
    plan.execute(x, out)
    ctx.sync()
    plan.close()
    return out[:NR].double()


@pytest.mark.parametrize("form", [R.FORM_MFMA_F16, R.FORM_MFMA_BF16])
@pytest.mark.parametrize("xr", [(7.0, 7.0), (10.0, 10.0), (3.0, 3.0, 3.0), (6.0, 6.0, 6.0), (9.0, 5.0, 7.0)])
def test_error_not_above_the_general_form(ctx, form, xr):
    import torch
    x = torch.rand((NBIG, len(xr)), dtype=torch.float64, device="cuda",
                   generator=torch.Generator(device="cuda").manual_seed(1)) * torch.tensor(xr, device="cuda")
    x = x.double().contiguous()
    ref = _field(ctx, R.FORM_FP64, xr, NR, x, torch.float64)
    general = _field(ctx, form, xr, 129, x, torch.float32)

    def err(u, n):
        return float(((u - ref[:, :n]).square().mean() / ref[:, :n].square().mean()).sqrt())

    for n in (20000, NBIG):                          # both block shapes
        got = _field(ctx, form, xr, NR, x[:n].contiguous(), torch.float32)
        assert err(got, n) <= err(general[:, :n], n), n
