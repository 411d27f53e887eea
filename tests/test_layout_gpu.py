"""Grid arrays across the ABI (IDX order on the host, track-major on the
device): uploads, downloads and the costs computed in between equal the
oracle's on grids whose sides are no multiple of the transpose's 32 x 32
tile, in both orientations of the first layer, on either side of the 32768
cells above which the order changes on the device."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.ascontiguousarray(a).view(np.uint32 if a.dtype == np.float32 else np.uint64)


@pytest.mark.parametrize("DIR", [0, 1])
@pytest.mark.parametrize("L,X,Y", [(1, 2, 2), (2, 33, 31), (2, 128, 128), (3, 5, 2185), (9, 95, 65), (15, 811, 3)])
def test_grid_arrays_keep_their_cells(ga, ora, L, X, Y, DIR):
    rng = np.random.default_rng(L * 1000 + X)
    cells = L * X * Y
    t = dict(L=L, X=X, Y=Y, DIR=DIR, unit_length_wire_cost=0.01, unit_via_cost=4.0,
             unit_length_short_costs=rng.random(L) + 0.5, x_edge_len=rng.integers(1, 400, X - 1).astype(np.int32),
             y_edge_len=rng.integers(1, 400, Y - 1).astype(np.int32),
             capacity=rng.integers(0, 6, cells).astype(np.float32))
    demand = (rng.integers(0, 30, cells) * 0.5).astype(np.float32)
    print(f"grid arrays L={L} {X}x{Y} DIR={DIR}", flush=True)
    ctx = ga.Context(t)
    ctx.upload_demand(demand)
    assert np.array_equal(ctx.demand(), demand)
    assert not ctx.timestamps().any()
    ctx.refresh()
    for got, want in zip(ctx.costs(), ora.Grid(t).refresh(demand)):
        assert np.array_equal(_bits(got), _bits(want.ravel()))
    ctx.close()


def _context(ga, L, X, Y):
    t = dict(L=L, X=X, Y=Y, DIR=0, unit_length_wire_cost=0.01, unit_via_cost=4.0,
             unit_length_short_costs=np.ones(L), x_edge_len=np.full(X - 1, 30, np.int32),
             y_edge_len=np.full(Y - 1, 30, np.int32), capacity=np.full(L * X * Y, 8, np.float32))
    return ga.Context(t)


@pytest.mark.parametrize("X,Y", [(8192, 2), (2, 8192)])
def test_narrow_grids_cost_what_their_cells_do(ga, X, Y):
    """The order change of a narrow grid takes about the time of a square one
    of as many cells (a launch over the square of the longer side took 8 times
    it on 2 x 8192)."""
    print(f"narrow grid {X}x{Y}", flush=True)
    best = []
    for x, y in ((X, Y), (128, 128)):
        ctx = _context(ga, 15, x, y)
        demand = np.arange(15 * x * y, dtype=np.float32) % 31
        runs = []
        for _ in range(15):
            start = time.perf_counter()
            ctx.upload_demand(demand)
            back = ctx.demand()
            runs.append(time.perf_counter() - start)
            assert np.array_equal(back, demand)
        best.append(min(runs))
        ctx.close()
    assert best[0] < 3 * best[1], best
