"""Interpolation to nodes on both of a block's paths (corners gathered from a
box in LDS, or directly) and both block sizes: FP64 bit for bit the oracle's."""
import numpy as np
import pytest

import randomfield_amd as R
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _nodes(nDim, nstep, m, order, rng):
    hi = np.array(nstep[:nDim]) - 1.0
    x = rng.random((m, nDim)) * hi
    if order == "mesh":                       # neighbours in the list are neighbours in space
        x = x[np.lexsort(np.floor(x / (hi / 12)).T)]
    x[0] = hi
    return np.ascontiguousarray(x)


@pytest.mark.parametrize("nDim,nstep", [(3, (40, 33, 21)), (2, (300, 41)), (1, (5000,)), (3, (2, 2, 2))])
@pytest.mark.parametrize("order", ["mesh", "random"])
@pytest.mark.parametrize("m,Nmc", [(1, 1), (255, 5), (1025, 4), (3000, 9)])
@pytest.mark.parametrize("dt", ["float64", "float32"])
def test_blocks_of_256(ctx, nDim, nstep, order, m, Nmc, dt):
    import torch
    rng = np.random.default_rng(m + Nmc)
    grid = rng.standard_normal((Nmc, int(np.prod(nstep)))).astype(dt)
    x = _nodes(nDim, nstep, m, order, rng)
    out = torch.empty((Nmc, m), dtype=getattr(torch, dt), device="cuda")
    assert not R.interpolate(ctx, nstep, [0.0] * nDim, [1.0] * nDim, Nmc, torch.from_numpy(grid).cuda(),
                             torch.from_numpy(x).cuda(), out)
    ref, bad = O.interp(grid.astype(np.float64), nstep, [0.0] * nDim, [1.0] * nDim, x)
    assert bad == 0 and np.array_equal(out.cpu().numpy(), ref.astype(dt))


@pytest.mark.parametrize("order", ["mesh", "random"])
@pytest.mark.parametrize("dt", ["float64", "float32"])
def test_blocks_of_1024(ctx, order, dt):
    """Half a million nodes and a ragged end; some outside the grid."""
    import torch
    rng = np.random.default_rng(4)
    nstep, Nmc, m = (90, 70, 50), 3, 512 * 1024 + 77
    grid = rng.standard_normal((Nmc, int(np.prod(nstep)))).astype(dt)
    x = _nodes(3, nstep, m, order, rng)
    out_of = rng.integers(0, m, 50)
    x[out_of, 1] += 1000.0
    x[2048:3072, 0] = -5.0                    # a whole block outside
    out = torch.full((Nmc, m), 7.0, dtype=getattr(torch, dt), device="cuda")
    assert R.interpolate(ctx, nstep, [0.0] * 3, [1.0] * 3, Nmc, torch.from_numpy(grid).cuda(), torch.from_numpy(x).cuda(),
                         out)
    got = out.cpu().numpy()
    outside = np.zeros(m, bool)
    outside[out_of] = True
    outside[2048:3072] = True
    assert np.isnan(got[:, outside]).all() and np.isfinite(got[:, ~outside]).all()
    s = np.flatnonzero(~outside)[::37]
    ref, bad = O.interp(grid.astype(np.float64), nstep, [0.0] * 3, [1.0] * 3, np.ascontiguousarray(x[s]))
    assert bad == 0 and np.array_equal(got[:, s], ref.astype(dt))


@pytest.mark.parametrize("nstep,Nmc", [((120, 110, 160), 5), ((170, 130, 150), 2), ((170, 130, 150), 7), ((160, 160, 160), 6)])
@pytest.mark.parametrize("dt", ["float64", "float32"])
def test_many_nodes_of_sparse_grids(ctx, nstep, Nmc, dt):
    """Half a million nodes with four, between four and six, and more grid points
    to a node: blocks of 1024 and 256 nodes, all realizations or four a block."""
    import torch
    rng = np.random.default_rng(Nmc)
    m = 512 * 1024 + 129
    grid = rng.standard_normal((Nmc, int(np.prod(nstep)))).astype(dt)
    x = _nodes(3, nstep, m, "mesh", rng)
    out = torch.full((Nmc, m), 7.0, dtype=getattr(torch, dt), device="cuda")
    assert not R.interpolate(ctx, nstep, [0.0] * 3, [1.0] * 3, Nmc, torch.from_numpy(grid).cuda(),
                             torch.from_numpy(x).cuda(), out)
    s = np.r_[np.arange(0, m, 41), m - 1]
    ref, bad = O.interp(grid.astype(np.float64), nstep, [0.0] * 3, [1.0] * 3, np.ascontiguousarray(x[s]))
    assert bad == 0 and np.array_equal(out.cpu().numpy()[:, s], ref.astype(dt))
