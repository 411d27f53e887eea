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


def _boxed(rec, ox, oy, w, n):
    """The record of a tree drawn in a w-wide box, moved to (ox, oy) of a map
    of side n."""
    out = np.array(rec, np.int32)
    pos = out[2::6]
    out[2::6] = (pos // w + ox) * n + pos % w + oy
    return out


def _odd(rec):
    """The first node's only child in its second slot, or a leaf at its
    parent's place."""
    r = rec[2:].reshape(-1, 6)
    if r[0, 4] == -1:
        r[0, 3:5] = -1, r[0, 3]
        return rec
    leaf = int(np.flatnonzero((r[1:, 3:] == -1).all(1))[0]) + 1
    parent = int(np.flatnonzero((r[:, 3:] == 6 * leaf).any(1))[0])
    r[leaf, 0] = r[parent, 0]
    return rec


def _with_second_parent(rec):
    """The last node is the child of two nodes."""
    r = rec[2:].reshape(-1, 6)
    last = 6 * (len(r) - 1)
    free = [i for i in range(len(r) - 1) if r[i, 5] == -1 and not (r[i, 3:] == last).any()]
    slots = r[free[0], 3:]
    slots[int(np.flatnonzero(slots == -1)[0])] = last
    return rec


@pytest.mark.parametrize("L,DIR,batches,odd", [(3, 1, 6, False), (6, 0, 260, False), (4, 1, 6, True)])
def test_zshape_batches_of_both_kernels(ga, ora, L, DIR, batches, odd):
    """Batches of nets in boxes of their own, most with trees for the per-net
    kernel and, in some batches and at any position, nets for the general one
    (a tree beyond the LDS bound, a node with two parents), beside batches of
    one kind only; nodes with a range of layers.  6 batches are planned on one
    thread, 260 on several.  `odd`: gaps in the child slots and two nodes at one
    place, which take nodes' layers from what earlier nets left on the map: the
    words and the error are the oracle's in a new context."""
    rng = np.random.default_rng(L)
    X, Y, w = 53, 44, 10
    n = max(X, Y)
    t = dict(L=L, X=X, Y=Y, DIR=DIR, unit_length_wire_cost=0.01, unit_via_cost=4.0,
             unit_length_short_costs=np.full(L, 5.0), x_edge_len=np.full(X - 1, 300, np.int32),
             y_edge_len=np.full(Y - 1, 300, np.int32),
             capacity=(rng.integers(0, 6, L * X * Y) + batches // 2).astype(np.float32))
    change = _odd if odd else _with_second_parent
    batch_off, rec_off, records, raw_cap = [0], [0], [], []
    kinds = set()
    for b in range(batches):
        boxes = [(x * w + 1, y * w + 1, w) for x in range(5) for y in range(4)]
        if b % 6 == 5:  # a large box instead of the first eight
            boxes = [(0, 0, 20)] + [q for q in boxes if q[0] >= 21 or q[1] >= 21]
        rng.shuffle(boxes)
        recs = []
        for ox, oy, side in boxes:
            nodes = 330 if side == 20 else int(rng.integers(4, 12))
            rec = _boxed(_tree_record(rng, side, side, L, nodes, "tree"), int(ox), int(oy), int(side), n)
            r = rec[2:].reshape(-1, 6)
            pick = (r[:, 1] != -1) & (rng.random(len(r)) < 0.5)
            r[pick, 2] = rng.integers(r[pick, 1], L + 1)
            # every sixth batch is all of one kind, the others mix them
            general = b % 6 != 0 and (b % 6 == 1 or rng.random() < 0.3)
            if general and side != 20:
                rec = change(rec)
            kinds.add((b % 6, general or side == 20))
            recs.append(rec)
        cap = [8192 if len(r) > 1000 else 512 for r in recs]
        at, raw = len(recs), 0
        offs = []
        for rec, c in zip(recs, cap):
            rec[0] = raw
            raw += c
            offs.append(at)
            at += len(rec)
        records += offs + [v for rec in recs for v in rec]
        raw_cap += cap
        batch_off.append(batch_off[-1] + len(recs))
        rec_off.append(len(records))
    assert (0, True) not in kinds and (1, False) not in kinds
    nets = batch_off[-1]
    plan = dict(batch_off=np.array(batch_off, np.int32), net_ids=rng.permutation(nets).astype(np.int32),
                rec_off=np.array(rec_off, np.int64), records=np.array(records, np.int32),
                raw_cap=np.array(raw_cap, np.int32))
    pins = np.empty(nets, np.int64)
    pins[plan["net_ids"]] = np.array(raw_cap) // 256
    acc = np.concatenate([[0], np.cumsum(pins)]).astype(np.int32)
    print(f"zshape batches of both kernels L={L} nets={nets}", flush=True)
    routes_o, demand_o, ts_o, wl_o, vias_o, rc = ora.Grid(t).zshape_stage(plan, acc, threads=1)
    assert rc == (3 if odd else 0)
    ctx = ga.Context(t)
    ctx.set_routes(acc, 256)
    ctx.set_cost_params(integer_wire=True)
    for _ in range(1 if odd else 2):  # the second upload finds the first one's arrays
        ctx.reset()
        ctx.zshape_upload(plan)
        if odd:
            with pytest.raises(ga.GrError, match="outside the grid"):
                ctx.zshape_run(first_stamp=1)
        else:
            ctx.zshape_run(first_stamp=1)
        assert np.array_equal(ctx.routes(), routes_o)
        assert np.array_equal(_bits(ctx.demand()), _bits(demand_o))
        assert np.array_equal(ctx.timestamps(), ts_o)
        assert ctx.stats() == (wl_o, vias_o)
    ctx.close()
