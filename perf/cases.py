"""Performance cases of the routing hot path.

Each case is one call, or the short sequence of calls that belongs together,
of grotor_amd's public entry points on a synthetic instance of one of the
generator's configurations (1: 128x128x5, 20k nets; 2 and 4: 512x512x9, 300k
nets; 3: 1024x1024x10, 1M nets; 6: 64x64x5, 2k nets), at the sizes and at
scaled sizes of the same density, odd grid sides among them.

A case holds its kind (`work`), the configuration, the fraction of its nets,
the grid side and the options of that kind.
"""
import math

import numpy as np
import torch

import grotor_amd as ga
from grotor_amd.soft import soft_dag_cost, soft_lshape_cost

# per configured net: routed subnets, tree nodes and pins (averages of the
# generator's instances), routing layers and net count of the configuration
_PER_NET = {1: (0.97, 3.10, 2.88), 2: (1.28, 6.23, 5.84), 3: (1.18, 5.81, 5.23), 4: (1.28, 6.23, 5.84),
            6: (0.97, 3.10, 2.88)}
_LAYERS = {1: 4, 2: 8, 3: 9, 4: 8, 6: 4}
_NETS = {1: 20000, 2: 300000, 3: 1000000, 4: 300000, 6: 2000}
# six standard deviations of one net's pins
_PIN_SPREAD = {1: 12, 2: 120, 3: 50, 4: 120, 6: 12}
_SIDE = {1: 128, 2: 512, 3: 1024, 4: 512, 6: 64}

_SOFT_BIG = 1e20


def listed():
    return [
        # the smallest stage: launches and latency of one rip-up iteration on
        # a block-sized instance, in the form the command line runs
        dict(name="lshape_block_64", work="lshape", config=6, scale=1.0, side=64, mode=2),
        # an ordinary block on an odd grid in the entry point's default form
        dict(name="lshape_plain_131", work="lshape", config=1, scale=1.0, side=131, mode=0),
        # the large L-shape stage of the rip-up pipeline (half a million nets)
        dict(name="lshape_large_768", work="lshape", config=3, scale=0.5, side=768, mode=2),
        # batch colouring of a stage's nets, repeated in every stage
        dict(name="batch_colors_512", work="batch", config=2, scale=0.5, side=512),
        # between the stages of the rip-up pipeline: the nets to reroute and
        # the congestion view their topologies are built from
        dict(name="ripup_view_384", work="ripup", config=3, scale=0.14, side=384),
        # FLT rerouting of a tenth of a design's nets over a given demand map
        dict(name="flt_251", work="flt", config=2, scale=0.24, side=251, share=0.1, mode=1),
        # the Z-shape stage (batches of bounding-box disjoint nets)
        dict(name="zshape_128", work="zshape", config=1, scale=1.0, side=128),
        # costs of a demand map, exchanged with a host program (a maze router
        # or another stage that runs on the host)
        dict(name="cost_exchange_333", work="cost", config=2, scale=0.002, side=333),
        # soft DP training step on the cost-model parameters, binary32 tables
        dict(name="soft_params_256", work="soft", config=4, scale=0.25, side=256, kind=0, tau=1.0, precision=32),
        # the same over the Z-shape route family, at a low temperature
        dict(name="soft_zshape_160", work="soft", config=4, scale=0.1, side=160, kind=1, tau=0.1, precision=32),
        # soft DP over given cost tensors in binary64 (small instance)
        dict(name="soft_costs_64", work="softcost", config=6, scale=1.0, side=64, kind=1, tau=1.0, precision=64),
        # evaluator score of a routed stage
        dict(name="score_256", work="score", config=2, scale=0.25, side=256),
    ]


def draw(rng):
    work = rng.choice(["lshape", "lshape", "lshape", "batch", "ripup", "flt", "zshape", "cost", "soft", "soft",
                       "softcost", "score"])

    def size(config, lo, hi):
        """A side spread over its logarithm, and the fraction of the nets that
        keeps the configuration's density on it (between half and all of it)."""
        side = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        return dict(config=config, scale=round((side / _SIDE[config]) ** 2 * rng.uniform(0.5, 1.0), 6), side=side)

    if work == "lshape":
        return dict(work=work, **size(*rng.choice([(6, 48, 128), (1, 64, 400), (2, 96, 500), (3, 200, 700)])),
                    mode=rng.choice([0, 1, 2, 2]))
    if work == "batch":
        return dict(work=work, **size(*rng.choice([(1, 64, 300), (2, 96, 360), (3, 200, 600)])))
    if work == "ripup":
        return dict(work=work, **size(*rng.choice([(1, 64, 400), (3, 96, 384)])))
    if work == "flt":
        return dict(work=work, **size(*rng.choice([(1, 64, 251), (2, 96, 251)])),
                    share=round(rng.uniform(0.02, 0.1), 3), mode=rng.choice([0, 1, 1]))
    if work == "zshape":
        return dict(work=work, **size(*rng.choice([(6, 48, 128), (1, 64, 128), (2, 64, 110)])))
    if work == "cost":
        return dict(work=work, config=2, scale=0.002, side=rng.randint(48, 333))
    if work == "soft":
        kind = rng.randint(0, 1)
        return dict(work=work, **size(4, 64, 160 if kind else 256), kind=kind, tau=rng.choice([0.1, 1.0, 10.0]),
                    precision=rng.choice([32, 32, 64]))
    if work == "softcost":
        return dict(work=work, **size(6, 40, 90), kind=rng.randint(0, 1), tau=rng.choice([0.1, 1.0, 10.0]),
                    precision=rng.choice([32, 64, 64]))
    return dict(work=work, **size(*rng.choice([(1, 64, 256), (2, 96, 256), (3, 128, 360)])))


# ---- inputs ----------------------------------------------------------------


def _design(case, seed):
    d = ga.Design.generate(case["config"], seed=seed, net_scale=case["scale"], grid_side=case["side"])
    d.prepare(16)
    return d, d.topology()


def _geometry(t):
    return t["pt_off"], t["pts"], t["hs_off"], t["hsegs"], t["vs_off"], t["vsegs"]


def _ranges(off, rows):
    """Indices of the rows' entries in a CSR array, row after row."""
    size = (off[rows + 1] - off[rows]).astype(np.int64)
    ends = np.cumsum(size)
    return np.arange(int(ends[-1]) if len(ends) else 0) - np.repeat(ends - size - off[rows], size), ends


def _subset(t, rows):
    """Batching geometry of the nets `rows` of a stage."""
    out = []
    for off, data, width in (("pt_off", "pts", 1), ("hs_off", "hsegs", 2), ("vs_off", "vsegs", 2)):
        idx, ends = _ranges(t[off], rows)
        out += [np.concatenate([[0], ends]).astype(np.int32), t[data].reshape(-1, width)[idx].reshape(-1)]
    return out


def _schedule(t, color, nb):
    """Execution order of a stage: batches last colour first."""
    slots = np.argsort(nb - 1 - color, kind="stable")
    idx, ends = _ranges(t["node_off"], slots)
    counts = np.bincount(nb - 1 - color, minlength=nb)
    return dict(net_ids=t["order"][slots], node_off=np.concatenate([[0], ends]).astype(np.int32), nodes=t["nodes"][idx],
                parents=t["parents"][idx], batch_off=np.concatenate([[0], np.cumsum(counts)]).astype(np.int32))


def _capacity(case):
    """Subnets and pins that route storage holds for any instance of the case."""
    nets = _NETS[case["config"]] * case["scale"]
    subnets, _, pins = (1.05 * nets * k for k in _PER_NET[case["config"]])
    spread = _PIN_SPREAD[case["config"]] * math.sqrt(nets)
    return int(subnets + spread / 10) + 8, int(pins + spread) + 16


def _storage(case, t):
    """pin_acc_num of a route store of the case's fixed size: the instance's
    subnets, then empty ones."""
    acc = t["pin_acc_num"]
    subnets, pins = _capacity(case)
    out = np.full(max(subnets, len(acc) - 1) + 1, acc[-1], np.int32)
    out[:len(acc)] = acc
    out[-1] = max(pins, acc[-1])
    return out


def _demand(t, seed):
    """Demand around the capacities, in the half units that commits add."""
    r = np.random.default_rng(seed)
    cap = t["capacity"]
    full = np.maximum(cap, 2.0) * r.gamma(3.0, 0.25, cap.size)
    return (np.round(2.0 * np.minimum(full, cap + 6.0)) / 2.0).astype(np.float32)


def _lshape_stage(case, t, ctx):
    """The L-shape stage in the context, ready to run; returns its batch offsets."""
    ctx.set_routes(_storage(case, t))
    color, nb = ctx.batch_plan(*_geometry(t))
    s = _schedule(t, color, nb)
    ctx.lshape_upload(s["net_ids"], s["node_off"], s["nodes"], s["parents"])
    return s["batch_off"]


def _flt_plan(d, ctx, reroute, xsum, ysum):
    f = d.flt_stage(reroute, xsum, ysum, threads=16)
    color, nb = ctx.batch_plan(*_geometry(f), limit=300000)
    return f, d.flt_plan(color, nb)


def prepare(case, seed):
    work = case["work"]
    d, t = _design(case, seed)
    ctx = ga.Context(t)
    s = dict(case=case, design=d, t=t, ctx=ctx)
    if work == "lshape":
        s["batch_off"] = _lshape_stage(case, t, ctx)
    elif work == "batch":
        n = int(0.9 * _NETS[case["config"]] * case["scale"] * _PER_NET[case["config"]][0])
        ctx.batch_geometry(*_subset(t, np.sort(np.random.default_rng(seed).permutation(t["nets"])[:n])))
    elif work == "ripup":
        ctx.lshape_run(_lshape_stage(case, t, ctx), 1, 2)
    elif work == "flt":
        ctx.set_routes(t["pin_acc_num"])
        s["demand"] = _demand(t, seed)
        ctx.upload_demand(s["demand"])
        _, xs, ys = ctx.congestion_view()
        flags = (np.random.default_rng(seed + 1).random(t["subnets"]) < case["share"]).astype(np.uint8)
        flags[0] = 1
        s["flt"], s["plan"] = _flt_plan(d, ctx, flags, xs, ys)
        s["pins2"] = max(int(1.2 * case["share"] * _capacity(case)[1]) + 400, s["flt"]["pins2"])
    elif work == "zshape":
        z = d.zshape_stage()
        color, nb = ctx.batch_plan(*_geometry(z))
        ctx.set_cost_params(integer_wire=True)
        ctx.set_routes(_storage(case, t), words_per_pin=256)
        ctx.zshape_upload(d.zshape_plan(color, nb))
    elif work == "cost":
        s["demand"] = _demand(t, seed)
    elif work == "soft":
        ctx.set_routes(t["pin_acc_num"])
        ctx.lshape_upload(t["order"], t["node_off"], t["nodes"], t["parents"])
        s["demand"] = _demand(t, seed)
        ctx.upload_demand(s["demand"])
        ctx.set_soft_kind(case["kind"])
    elif work == "softcost":
        ctx.set_routes(t["pin_acc_num"])
        ctx.lshape_upload(t["order"], t["node_off"], t["nodes"], t["parents"])
        w, v = _given_costs(t, seed)
        s["wcost"] = torch.from_numpy(w).requires_grad_()
        s["vcost"] = torch.from_numpy(v).requires_grad_()
    elif work == "score":
        batch_off = _lshape_stage(case, t, ctx)
        ctx.lshape_run(batch_off, 1, 2)
        s["nets"], s["grid"] = d.nets(), d.metal_grid()
    else:
        raise ValueError(work)
    return s


def _given_costs(t, seed):
    r = np.random.default_rng(seed)
    n = t["L"] * t["X"] * t["Y"]
    return r.gamma(2.0, 3.0, n), 4.0 + r.gamma(2.0, 1.0, n)


# ---- one pass --------------------------------------------------------------


def run(s):
    case, ctx, t = s["case"], s["ctx"], s["t"]
    work = case["work"]
    if work == "lshape":
        ctx.reset()
        ctx.lshape_run(s["batch_off"], 1, case["mode"])
        return dict(routes=ctx.routes(), stats=np.array(ctx.stats()))
    if work == "batch":
        color, nb = ctx.batch_colors()
        return dict(color=color, batches=nb)
    if work == "ripup":
        flags = ctx.ripup(ctx.nets)
        congested, xs, ys = ctx.congestion_view()
        return dict(flags=flags, congested=congested, xsum=xs, ysum=ys)
    if work == "flt":
        ctx.reset()
        ctx.upload_demand(s["demand"])
        ctx.set_routes_phase2(s["flt"]["pin_off2"], s["pins2"])
        ctx.flt_upload(s["plan"])
        ctx.flt_run(1, remove=0, mode=case["mode"])
        return dict(routes2=ctx.routes2())
    if work == "zshape":
        ctx.reset()
        ctx.zshape_run(1)
        return dict(routes=ctx.routes())
    if work == "cost":
        ctx.upload_demand(s["demand"])
        ctx.refresh()
        w, v, p = ctx.costs()
        return dict(wcost=w, vcost=v, presum=p)
    if work == "soft":
        params = torch.tensor([0.5, 1.5, 1.0], dtype=torch.float64, requires_grad=True)
        total = soft_lshape_cost(ctx, params, 0, t["nets"], tau=case["tau"], precision=case["precision"])
        total.backward()
        gw, gv = ctx.soft_edge_grads()
        return dict(total=total.detach(), params=params.grad, wires=gw, vias=gv)
    if work == "softcost":
        s["wcost"].grad = s["vcost"].grad = None
        total = soft_dag_cost(ctx, s["wcost"], s["vcost"], 0, t["nets"], tau=case["tau"], precision=case["precision"],
                              kind=case["kind"])
        total.backward()
        return dict(total=total.detach(), wires=s["wcost"].grad, vias=s["vcost"].grad)
    if work == "score":
        g = s["grid"]
        r = ctx.score(s["nets"], g["dir"], g["capacity"], g["overflow_cost"], demand=True)
        return dict(costs=np.array([r["wirelength"], r["via"], r["overflow"], r["total"]]), rejected=r["rejected"],
                    demand=r["demand"].astype(np.int32))
    raise ValueError(work)


# ---- what a pass cannot do without -----------------------------------------


def work(case):
    cfg = case["config"]
    nets = _NETS[cfg] * case["scale"]
    subnets, nodes, pins = (nets * k for k in _PER_NET[cfg])
    L = _LAYERS[cfg]
    cells = L * case["side"] ** 2
    words = 4 * 12 * pins
    kind = case["work"]
    if kind == "lshape":
        return dict(bytes=8 * cells + 8 * nodes + words, flops=nodes * L * L * 8)
    if kind == "batch":
        return dict(bytes=8 * nodes + 12 * nodes + 8 * subnets, flops=nodes * 16)
    if kind == "ripup":
        return dict(bytes=8 * cells + 32 * nodes + subnets + 9 * case["side"] ** 2, flops=6 * cells + 8 * nodes)
    if kind == "flt":
        f = case["share"] * nodes * 6
        return dict(bytes=8 * cells + 28 * f + 400 * case["share"] * pins, flops=f * L * L * 8)
    if kind == "zshape":
        return dict(bytes=8 * cells + 24 * nodes + 4 * 256 * pins, flops=nodes * L * 8 * 12)
    if kind == "cost":
        return dict(bytes=24 * cells, flops=40 * cells)
    if kind in ("soft", "softcost"):
        routes = (L * L / 2) * (8 if case["kind"] else 1)
        return dict(bytes=(8 if kind == "soft" else 16) * cells + 8 * nodes + 16 * cells,
                    flops=nodes * (L * L * L + routes) * 2 * 20)
    return dict(bytes=words + 4 * pins + 8 * (cells + case["side"] ** 2) + 2 * (cells + case["side"] ** 2),
                flops=10 * cells)


def tolerance(case):
    kind = case["work"]
    if kind in ("soft", "softcost"):
        # four times the distance to exact() measured on the listed and drawn
        # cases: with binary32 tables 5e-5 at tau = 1 and 1.5e-4 at tau = 0.1
        # (a table entry's 2^-24 grows by cost / tau in the exponent), with
        # binary64 tables some 1e-14
        if case["precision"] == 64:
            return dict(rel=1e-12)
        return dict(rel=6e-4 if case["tau"] < 0.5 else 2e-4)
    if kind == "score":
        return dict(rel=1e-12, differ=0.0)
    return "exact"  # the routes are defined bit for bit, and with them the costs


# ---- references in 64 bits -------------------------------------------------


def exact(case, seed):
    kind = case["work"]
    if kind == "cost":
        d, t = _design(case, seed)
        return _exact_costs(t, _demand(t, seed))
    if kind in ("soft", "softcost"):
        d, t = _design(case, seed)
        return _exact_soft(case, t, seed)
    if kind == "score":
        return _exact_score(prepare(case, seed))
    if kind == "ripup":
        return _exact_view(prepare(case, seed))
    return None


def _dirs(t):
    """1 where a routing layer runs along y."""
    return [(l & 1) ^ t["DIR"] for l in range(t["L"])]


def _exact_costs(t, demand):
    """Wire and via costs and exclusive prefix sums along the tracks (IDX order)."""
    L, X, Y = t["L"], t["X"], t["Y"]
    cap = t["capacity"].reshape(L, X, Y).astype(np.float64)
    dem = demand.reshape(L, X, Y).astype(np.float64)

    def e(d):
        with np.errstate(over="ignore"):
            return np.where(cap > 0.001, np.exp(np.minimum(0.5 * (d - cap), 700)),
                            np.where(d > 0, np.exp(np.minimum(1.5 * d, 700)), 0.0))

    w, v, p = np.empty_like(cap), np.empty_like(cap), np.zeros_like(cap)
    for l, along_y in enumerate(_dirs(t)):
        sc = t["unit_length_short_costs"][l]
        one = np.minimum(1e12, (e(dem + 1.0)[l] - e(dem)[l]) * sc)
        half = np.minimum(1e12, (e(dem + 0.5)[l] - e(dem)[l]) * sc)
        one, half = (one, half) if along_y else (one.T, half.T)  # [track, position]
        elen = t["y_edge_len"] if along_y else t["x_edge_len"]
        wl, vl = one.copy(), np.empty_like(one)
        wl[:, :-1] += t["unit_length_wire_cost"] * elen
        vl[:, 1:] = half[:, 1:] + half[:, :-1]
        vl[:, 0] = one[:, 0]
        vl[:, -1] = one[:, -2]
        pl = np.zeros_like(one)
        pl[:, 1:] = np.cumsum(wl[:, :-1], axis=1)
        vl += t["unit_via_cost"]
        w[l], v[l], p[l] = (wl, vl, pl) if along_y else (wl.T, vl.T, pl.T)
    return dict(wcost=w.reshape(-1), vcost=v.reshape(-1), presum=p.reshape(-1))


def _exact_view(s):
    """Worst overflow over the layers per place, its exclusive prefix sums along x and y."""
    t = s["t"]
    L, X, Y = t["L"], t["X"], t["Y"]
    over = s["ctx"].demand().astype(np.float64) - t["capacity"]
    worst = np.maximum(over.reshape(L, X, Y).max(0), 0.0)
    xs, ys = np.zeros((X, Y)), np.zeros((X, Y))
    xs[1:], ys[:, 1:] = np.cumsum(worst, 0)[:-1], np.cumsum(worst, 1)[:, :-1]
    return dict(flags=None, congested=None, xsum=xs.reshape(-1), ysum=ys.reshape(-1))


def _soft_model(t, demand, params, device):
    """Smooth wire and via costs [L, X, Y] as torch functions of the parameters."""
    L, X, Y = t["L"], t["X"], t["Y"]
    cap = torch.from_numpy(t["capacity"].reshape(L, X, Y).astype(np.float64)).to(device)
    dem = torch.from_numpy(demand.reshape(L, X, Y).astype(np.float64)).to(device)
    slope, zero, via = params
    has = cap > 0.001

    def e(d):
        return torch.where(has, torch.exp(slope * torch.where(has, d - cap, torch.zeros_like(d))),
                           torch.where((d > 0) & ~has, torch.exp(zero * torch.where(has, torch.zeros_like(d), d)),
                                       torch.zeros_like(d)))

    wl, vl = [], []
    sc = torch.from_numpy(t["unit_length_short_costs"]).to(device)[:, None, None]
    one, half = (torch.clamp((e(dem + k) - e(dem)) * sc, max=1e12) for k in (1.0, 0.5))
    for l, along_y in enumerate(_dirs(t)):
        o, h = (one[l], half[l]) if along_y else (one[l].T, half[l].T)
        elen = torch.from_numpy((t["y_edge_len"] if along_y else t["x_edge_len"]).astype(np.float64)).to(device)
        w = o + torch.cat([t["unit_length_wire_cost"] * elen, elen.new_zeros(1)])
        v = torch.cat([o[:, :1], h[:, 1:-1] + h[:, :-2], o[:, -2:-1]], 1) + via * t["unit_via_cost"]
        wl.append(w if along_y else w.T)
        vl.append(v if along_y else v.T)
    return torch.stack(wl), torch.stack(vl)


def _smin(x, tau, dim):
    return -tau * torch.logsumexp(-x / tau, dim)


def _soft_total(t, w, v, tau, kind):
    """Sum over the nets of the soft DP value at costs w, v [L, X, Y]."""
    dev = w.device
    L, X, Y = t["L"], t["X"], t["Y"]
    dirs = _dirs(t)
    big = 1e22
    prefix = []  # exclusive prefix of w along the tracks
    for l in range(L):
        c = torch.cumsum(w[l], 1 if dirs[l] else 0)
        prefix.append(c - w[l])
    prefix = torch.stack(prefix)
    up = torch.cat([torch.zeros_like(v[:1]), torch.cumsum(v, 0)])  # [L + 1]: vias below each layer

    nodes, off = t["nodes"].astype(np.int64), t["node_off"]
    start = np.repeat(off[:-1], np.diff(off)).astype(np.int64)
    par = t["parents"].astype(np.int64)
    root = par < 0
    par = np.where(root, np.arange(len(par)), par + start)
    height = np.zeros(len(nodes), np.int64)
    while True:  # a parent lies above its highest child
        nxt = height.copy()
        np.maximum.at(nxt, par[~root], height[~root] + 1)
        if np.array_equal(nxt, height):
            break
        height = nxt
    X_, Y_ = nodes // Y % X, nodes % Y
    put = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    nx, ny, fixed = put(X_), put(Y_), put(nodes // (X * Y))
    lo, hi = (put(np.array(a)) for a in zip(*[(a, b) for a in range(L) for b in range(a, L)]))
    col = up[:, nx, ny]
    D = (col[hi] - col[lo]).T
    D = torch.where((fixed[:, None] < L) & ((lo > fixed[:, None]) | (hi < fixed[:, None])), torch.full_like(D, big), D)
    layers = torch.arange(L, device=dev)
    inside = (lo[:, None] <= layers) & (layers <= hi[:, None])  # [T, L]
    out = torch.where(inside, 0.0, big).to(torch.float64)
    vert = torch.tensor(dirs, device=dev) == 1
    cl, pl = torch.meshgrid(layers, layers, indexing="ij")
    stack_lo, stack_hi = torch.minimum(cl, pl), torch.maximum(cl, pl)

    def legs(along_y, fixed_, a, b):
        """Per layer the wire cost between positions a and b of the track through fixed_."""
        p = (lambda q: prefix[:, fixed_, q]) if along_y else (lambda q: prefix[:, q, fixed_])
        return (p(torch.maximum(a, b)) - p(torch.minimum(a, b))).T

    def columns(x, y, first, last):
        """Vias of layers first .. last - 1 at (x, y): [nodes, L, L]."""
        c = up[:, x, y]
        return (c[last] - c[first]).permute(2, 0, 1)

    def masked(x, keep):
        return torch.where(keep, x, torch.full_like(x, big))

    for h in range(int(height.max()) if len(height) else 0):
        e = put(np.flatnonzero((height == h) & ~root))
        p = put(par)[e]
        x, y, px, py = nx[e], ny[e], nx[p], ny[p]
        best = _smin(D[e][:, :, None] + out, tau, 1)
        col_edge, row_edge = x == px, (y == py) & (x != px)
        bent = ~(col_edge | row_edge)
        wv, wh = legs(True, x, y, py), legs(False, y, x, px)
        pwv, pwh = legs(True, px, y, py), legs(False, py, x, px)
        straight = best + torch.where(vert, wv, wh)
        # a column edge takes vertical layers; both coordinates alike: L-shape edges any layer
        along = torch.where(vert, col_edge[:, None], row_edge[:, None] | (col_edge & (y == py) & (kind == 0))[:, None])
        diag = masked(straight, along)
        first, last = torch.where(vert, wv, wh), torch.where(vert, pwv, pwh)
        if kind == 0:
            a, b = torch.minimum(stack_lo + 1, stack_hi), stack_hi
            turn = torch.where(vert[:, None], columns(x, py, a, b), columns(px, y, a, b))
            ok = ((cl ^ pl) & 1) == 1
        else:
            turn = torch.where(vert[:, None], columns(x, py, stack_lo, stack_hi), columns(px, y, stack_lo, stack_hi))
            ok = vert[:, None] != vert[None, :]
        cand = masked((best + first)[:, :, None] + turn + last[:, None, :], ok)
        route = _smin(cand, tau, 1)
        if kind == 1:
            for d1 in (1, 0):  # rows strictly between y and py, then columns between x and px
                one = vert if d1 else ~vert
                a0, a1 = (torch.minimum(y, py), torch.maximum(y, py)) if d1 else (torch.minimum(x, px), torch.maximum(x, px))
                count = torch.where(bent, a1 - a0 - 1, torch.zeros_like(a0))
                k = torch.repeat_interleave(torch.arange(len(e), device=dev), count)
                if not len(k):
                    continue
                bend = a0[k] + 1 + torch.arange(len(k), device=dev) - torch.repeat_interleave(torch.cumsum(count, 0) - count, count)
                xk, yk, pxk, pyk = x[k], y[k], px[k], py[k]
                if d1:
                    l1, l2, l3 = legs(True, xk, yk, bend), legs(False, bend, xk, pxk), legs(True, pxk, bend, pyk)
                    s1, s2 = columns(xk, bend, stack_lo, stack_hi), columns(pxk, bend, stack_lo, stack_hi)
                else:
                    l1, l2, l3 = legs(False, yk, xk, bend), legs(True, bend, yk, pyk), legs(False, pyk, bend, pxk)
                    s1, s2 = columns(bend, yk, stack_lo, stack_hi), columns(bend, pyk, stack_lo, stack_hi)
                pair = one[:, None] & ~one[None, :]
                f1 = _smin(masked((best[k] + l1)[:, :, None] + s1, pair), tau, 1) + l2
                mv = _smin(masked(f1[:, :, None] + s2, pair.T), tau, 1) + l3
                mv = masked(mv, one)
                base = torch.full((len(e), L), 1e30, dtype=torch.float64, device=dev)
                base = base.scatter_reduce(0, k[:, None].expand(-1, L), mv.detach(), "amin")
                s = torch.zeros_like(base).index_add(0, k, torch.exp(-(mv - base[k]) / tau))
                zs = torch.where(s > 0, base - tau * torch.log(torch.where(s > 0, s, torch.ones_like(s))), torch.full_like(s, big))
                route = _smin(torch.stack([route, zs]), tau, 0)
        diag = torch.where(bent[:, None], route, diag)
        C = _smin(diag[:, None, :] + out, tau, 2)
        D = D.index_add(0, p, C)
    value = _smin(D[put(np.flatnonzero(root))], tau, 1)
    return value[value < _SOFT_BIG].sum() if len(value) else value.sum()


def _exact_soft(case, t, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    L, X, Y = t["L"], t["X"], t["Y"]
    if case["work"] == "softcost":
        w, v = (torch.from_numpy(a).to(dev).reshape(L, X, Y).requires_grad_() for a in _given_costs(t, seed))
        total = _soft_total(t, w, v, case["tau"], case["kind"])
        total.backward()
        return dict(total=total.detach().cpu(), wires=w.grad.reshape(-1).cpu(), vias=v.grad.reshape(-1).cpu())
    params = torch.tensor([0.5, 1.5, 1.0], dtype=torch.float64, device=dev, requires_grad=True)
    w, v = _soft_model(t, _demand(t, seed), params, dev)
    w.retain_grad()
    v.retain_grad()
    total = _soft_total(t, w, v, case["tau"], case["kind"])
    total.backward()
    return dict(total=total.detach().cpu(), params=params.grad.cpu(), wires=w.grad.reshape(-1).cpu().numpy(),
                vias=v.grad.reshape(-1).cpu().numpy())


def _exact_score(s):
    """The evaluator's costs of the resident routes: per net its lines (a via
    under each metal-0 pin, the extra pairs, the subnets' route pairs one
    metal layer up), unit wires, via steps, and a stacked-via demand at each
    via place of the net that none of its own wires covers."""
    t, nets, g = s["t"], s["nets"], s["grid"]
    X, Y, M = t["X"], t["Y"], g["layers"]
    XY, cells = X * Y, g["layers"] * X * Y
    words, acc = s["ctx"].routes().astype(np.int64), t["pin_acc_num"].astype(np.int64)
    n = len(nets["pin_off"]) - 1
    net, a, b = [], [], []
    who = np.repeat(np.arange(n), np.diff(nets["pin_off"]))
    low = nets["pins"] < XY
    net.append(who[low]), a.append(nets["pins"][low]), b.append(nets["pins"][low] + XY)
    half = np.diff(nets["extra_off"]) // 2
    net.append(np.repeat(np.arange(n), half)), a.append(nets["extra"][0::2]), b.append(nets["extra"][1::2])
    sub = nets["subs"].astype(np.int64)
    pairs = (words[12 * acc[sub]] - 1) // 2
    first = np.repeat(12 * acc[sub] + 1, pairs) + 2 * (np.arange(pairs.sum()) - np.repeat(np.cumsum(pairs) - pairs, pairs))
    net.append(np.repeat(np.repeat(np.arange(n), np.diff(nets["sub_off"])), pairs))
    a.append(words[first] + XY), b.append(words[first + 1] + XY)
    net, a, b = (np.concatenate(q).astype(np.int64) for q in (net, a, b))
    a, b = np.minimum(a, b), np.maximum(a, b)
    za, zb = a // XY, b // XY
    wire = za == zb
    along_y = np.asarray(g["dir"])[za] != 0
    step = np.where(along_y, 1, Y)
    count = np.where(wire, (b - a) // step, 0)

    def spread(rows, size, stride):
        k = np.repeat(np.flatnonzero(rows), size[rows])
        i = np.arange(len(k)) - np.repeat(np.cumsum(size[rows]) - size[rows], size[rows])
        return k, a[k] + i * stride[k]

    k, edges = spread(wire, count, step)
    wires = np.bincount(edges, minlength=cells)
    k, ends = spread(wire, count + 1, step)
    covered = np.unique(net[k] * cells + ends)
    k, via = spread(~wire, zb - za, np.full(len(a), XY))
    vias = np.bincount(via // XY, minlength=M)
    place = np.unique(net[k] * cells + via)
    place = place[~np.isin(place, covered)] % cells
    z, x, y = place // XY, place // Y % X, place % Y
    vert = np.asarray(g["dir"])[z] != 0
    pos, length, step = np.where(vert, y, x), np.where(vert, Y, X), np.where(vert, 1, Y)
    here, before = pos < length - 1, pos > 0
    amount = np.where(here & before, 1, 2)
    stacked = np.bincount(place[here], amount[here], cells) + np.bincount((place - step)[before], amount[before], cells)
    demand = (2 * wires + stacked.astype(np.int64)) & 0xFFFF
    demand[:XY] = 0  # metal 0 is no routing layer
    cap = g["capacity"].astype(np.float64)
    loss = np.where(cap > 0.001, np.exp(0.25 * (demand - 2.0 * cap)), np.where(demand > 0, np.exp(0.75 * demand), 0.0))
    loss = loss.reshape(M, XY)
    loss[0] = 0.0
    wl = t["unit_length_wire_cost"] * sum(
        (wires[m * XY:(m + 1) * XY].reshape(X, Y)[:, :-1] * t["y_edge_len"]).sum() if g["dir"][m]
        else (wires[m * XY:(m + 1) * XY].reshape(X, Y)[:-1] * t["x_edge_len"][:, None]).sum() for m in range(M))
    via_cost = float(vias.sum()) * t["unit_via_cost"]
    over = float((loss.sum(1) * g["overflow_cost"]).sum())
    return dict(costs=np.array([wl, via_cost, over, wl + via_cost + over]), rejected=None, demand=demand)
