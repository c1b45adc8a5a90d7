"""Fresh realizations of a grid batch on each route of their coefficients: formed
by the first contraction (every first axis within a wave's 160 points), by the
grouped fold (any longer one), and with the autotuner between redraws.

Draw d of a batch is draw d of each field's plan: the same bits from
rf_plan_redraw and rf_plan_execute_grid, eagerly and replayed from a captured
graph whose counter advances, compared on every replay."""
import numpy as np
import pytest

import randomfield_amd as R

pytestmark = pytest.mark.gpu

FOLD = [((170, 6, 5), (0.1, 0.3, 0.4), 3, 51), ((20, 33, 12), (0.3, 0.2, 0.3), 2, 52), ((161, 9), (0.1, 0.3), 2, 53)]
FORMED = [((160, 6, 5), (0.1, 0.3, 0.4), 3, 51), ((20, 33, 12), (0.3, 0.2, 0.3), 2, 52), ((97, 9), (0.1, 0.3), 2, 53)]


def _plan(ctx, spec):
    n, step, Nmc, seed = spec
    return R.FieldPlan(ctx, R.make_params(nDim=len(n), method=R.SHINOZUKA, mode=R.FIXED, form=R.FORM_FP32, Nmc=Nmc,
                                          xRange=[(a - 1) * s for a, s in zip(n, step)], seed=seed))


def _plan_draws(ctx, specs, draws):
    import torch
    ref = {d: [] for d in draws}
    for n, step, Nmc, seed in specs:
        plan = _plan(ctx, (n, step, Nmc, seed))
        for d in draws:
            o = torch.empty((Nmc, int(np.prod(n))), dtype=torch.float32, device="cuda")
            torch.cuda.synchronize()
            plan.redraw(d)
            plan.execute_grid([0.0] * len(n), step, n, o)
            ctx.sync()
            ref[d].append(o)
        plan.close()
    return ref


@pytest.mark.parametrize("specs,tiles", [(FOLD, None), (FORMED, 5), (FORMED[1:], 4), (FORMED[1:2], 1)],
                         ids=["fold", "formed5", "formed4", "formed1"])
def test_redraws_equal_the_plans(ctx, specs, tiles):
    import torch
    ref = _plan_draws(ctx, specs, (0, 1, 2, 3, 7))
    plans = [_plan(ctx, s) for s in specs]
    outs = [torch.empty((s[2], int(np.prod(s[0]))), dtype=torch.float32, device="cuda") for s in specs]
    torch.cuda.synchronize()
    b = R.GridBatch(ctx, plans, [[0.0] * len(s[0]) for s in specs], [s[1] for s in specs], [s[0] for s in specs], outs,
                    R.DTYPE_F32)

    def check(d):
        torch.cuda.synchronize()
        ctx.sync()
        for i, o in enumerate(outs):
            assert torch.equal(o, ref[d][i]), (d, i)
            o.fill_(-1.0)
        torch.cuda.synchronize()

    b.execute()
    check(0)
    for d in (2, 7):
        b.redraw(d)
        b.execute()
        check(d)
    # the tuner keeps the current realizations, and how redraws get theirs
    for d in (3, 1):
        chosen = b.autotune()
        assert tiles is None or chosen[0] == tiles
        check(7 if d == 3 else 3)
        b.execute()
        check(7 if d == 3 else 3)
        b.redraw(d)
        b.execute()
        check(d)
    stream = torch.cuda.Stream()
    sp = stream.cuda_stream
    b.redraw(1, sp)                                  # the counter's next value
    torch.cuda.synchronize()
    graph = R.Graph(ctx, sp)
    with graph:
        b.redraw(R.DRAW_NEXT, sp)
        b.execute(sp)
    for d in (1, 2, 3):
        graph.launch(sp)
        check(d)
    graph.close()
    b.close()
    for p in plans:
        p.close()
