"""GPU Z-shape stage (reset, solve, convert, commit per batch) against the
oracle's restatement on the same plan: route words, demand, timestamps and
statistics identical."""
import numpy as np
import pytest

from tests._instances import topology

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.ascontiguousarray(a).view(np.uint32 if a.dtype == np.float32 else np.uint64)


@pytest.mark.parametrize("config,seed,scale", [(6, 0, 1.0), (6, 5, 1.0), (1, 2, 0.25)])
def test_zshape_stage_matches_oracle(ga, ora, config, seed, scale):
    d, t = topology(config, seed, net_scale=scale)
    z = d.zshape_stage()
    print(f"zshape stage config={config} seed={seed} nets={z['nets']}", flush=True)
    geom = (z["pt_off"], z["pts"], z["hs_off"], z["hsegs"], z["vs_off"], z["vsegs"])
    color, nb = ora.batches(t["X"], t["Y"], *geom)
    plan = d.zshape_plan(color, nb)
    routes_o, demand_o, ts_o, wl_o, vias_o, rc = ora.Grid(t).zshape_stage(plan, t["pin_acc_num"], threads=8)
    assert rc == 0
    ctx = ga.Context(t)
    ctx.set_routes(t["pin_acc_num"], 256)
    ctx.set_cost_params(integer_wire=True)
    gcolor, gnb = ctx.batch_plan(*geom)
    assert gnb == nb and np.array_equal(gcolor, color)
    ctx.zshape_upload(plan)
    ms = ctx.zshape_run(first_stamp=1)
    assert ms > 0
    assert np.array_equal(ctx.routes(), routes_o)
    assert np.array_equal(_bits(ctx.demand()), _bits(demand_o))
    assert np.array_equal(ctx.timestamps(), ts_o)
    assert ctx.stats() == (wl_o, vias_o)
    # host post-processing on the GPU's routes gives the oracle's result
    r_gpu, r_o = ctx.routes(), routes_o.copy()
    assert d.zshape_finish(r_gpu) == d.zshape_finish(r_o)
    assert np.array_equal(r_gpu, r_o)
    ctx.close()


def _tree_record(rng, X, Y, L, nodes, shape):
    """Records of one random tree: at most three children per node."""
    n = max(X, Y)
    cells = rng.choice(X * Y, nodes, replace=False)
    if shape == "line":  # straight edges only, on one column
        cells = np.arange(nodes) % Y + (X // 2) * Y
    kids = [[] for _ in range(nodes)]
    for k in range(1, nodes):
        free = [i for i in range(max(0, k - 6), k) if len(kids[i]) < 3]
        kids[int(rng.choice(free))].append(k)
    order, stack = [], [0]
    while stack:
        v = stack.pop()
        order.append(v)
        stack.extend(reversed(kids[v]))
    at = {v: i for i, v in enumerate(order)}
    rec = []
    for v in order:
        layer = -1 if kids[v] and v and rng.random() < 0.5 else int(rng.integers(1, L + 1))
        c = int(cells[v])
        rec.append([c // Y * n + c % Y, layer, layer] + [6 * at[w] for w in kids[v]] + [-1] * (3 - len(kids[v])))
    return [0, nodes] + [w for r in rec for w in r]


@pytest.mark.parametrize("L,X,Y,nodes", [(1, 9, 7, (1, 2, 9)), (2, 17, 33, (2, 3, 40)), (4, 31, 40, (5, 219, 220)),
                                         (8, 64, 20, (17, 70, 129)), (15, 23, 23, (6, 79, 80))])
def test_zshape_trees_of_every_size_and_form(ga, ora, L, X, Y, nodes):
    """Trees around the LDS bound of the per-net kernel (48 KiB: 219 nodes on
    4 layers, 79 on 15; the general kernels take the larger ones), straight
    and bent edges, one net per batch: equal to the oracle."""
    rng = np.random.default_rng(100 * L + X)
    t = dict(L=L, X=X, Y=Y, DIR=L & 1, unit_length_wire_cost=0.01, unit_via_cost=4.0,
             unit_length_short_costs=np.full(L, 5.0), x_edge_len=np.full(X - 1, 300, np.int32),
             y_edge_len=np.full(Y - 1, 300, np.int32),
             capacity=rng.integers(0, 6, L * X * Y).astype(np.float32))
    shapes = ["tree", "tree", "line"] if L > 1 else ["line"]
    records, rec_off = [], [0]
    for k in range(3 * len(shapes)):
        m = nodes[k % 3]
        shape = shapes[k // 3]
        records += [1] + _tree_record(rng, X, Y, L, min(m, Y) if shape == "line" else m, shape)
        rec_off.append(len(records))
    nets = len(rec_off) - 1
    pins = 8 * max(nodes)
    plan = dict(batch_off=np.arange(nets + 1, dtype=np.int32), net_ids=np.arange(nets, dtype=np.int32)[::-1].copy(),
                rec_off=np.array(rec_off, np.int64), records=np.array(records, np.int32),
                raw_cap=np.full(nets, 256 * pins, np.int32))
    acc = (np.arange(nets + 1) * pins).astype(np.int32)
    print(f"zshape trees L={L} {X}x{Y} nodes={nodes}", flush=True)
    routes_o, demand_o, ts_o, wl_o, vias_o, rc = ora.Grid(t).zshape_stage(plan, acc, threads=1)
    assert rc == 0
    ctx = ga.Context(t)
    ctx.set_routes(acc, 256)
    ctx.set_cost_params(integer_wire=True)
    ctx.zshape_upload(plan)
    ctx.zshape_run(first_stamp=1)
    assert np.array_equal(ctx.routes(), routes_o)
    assert np.array_equal(_bits(ctx.demand()), _bits(demand_o))
    assert np.array_equal(ctx.timestamps(), ts_o)
    assert ctx.stats() == (wl_o, vias_o)
    ctx.close()
