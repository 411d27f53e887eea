"""GPU soft (log-sum-exp) DP, over L-shape edges and over the Z-shape route
family, against the FP64 oracle (oracle/soft.c) on the 64x64x5, 2k-net
instance: values, per-cell gradients, parameter gradients against FP64
central finite differences (h = 1e-4), and the torch.autograd.Functions
(over the cost-model parameters, and over the per-cell cost tensors, whose
gradients are checked against FP64 central differences of the GPU forward,
h = 1e-4, relative error at most 1e-4)."""
import numpy as np
import pytest

from tests._instances import random_demand, topology

pytestmark = pytest.mark.gpu

TAUS = (0.1, 1.0, 10.0)
THETA = (0.5, 1.5, 1.0)


def _setup(ga, seed=0):
    _, t = topology(6, seed)
    ctx = ga.Context(t)
    ctx.set_routes(t["pin_acc_num"])
    ctx.lshape_upload(t["order"], t["node_off"], t["nodes"], t["parents"])
    demand = random_demand(t, seed + 11, high=4)
    ctx.upload_demand(demand)
    return t, ctx, demand


def _fd(grid, t, demand, tau, j, h=1e-4, kind=0):
    tp, tm = list(THETA), list(THETA)
    tp[j] += h
    tm[j] -= h
    args = (demand, t["node_off"], t["nodes"], t["parents"], tau)
    return (grid.soft_stage(*args, *tp, kind=kind) - grid.soft_stage(*args, *tm, kind=kind)) / (2 * h)


@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("tau", TAUS)
def test_soft_fp64_matches_oracle(ga, ora, tau, kind):
    t, ctx, demand = _setup(ga)
    n = t["nets"]
    print(f"soft fp64 kind={kind} tau={tau} nets={n}", flush=True)
    grid = ora.Grid(t)
    F_o, gw_o, gv_o, gp_o = grid.soft_stage(demand, t["node_off"], t["nodes"], t["parents"], tau, *THETA, grads=True,
                                            kind=kind)
    ctx.set_soft_kind(kind)
    total, per_net, _ = ctx.soft_forward(0, n, *THETA, tau=tau, precision=64, per_net=True)
    assert abs(total - F_o) <= 1e-10 * abs(F_o)
    gp, _ = ctx.soft_backward()
    gw, gv = ctx.soft_edge_grads()
    assert np.allclose(gw, gw_o, rtol=1e-8, atol=1e-10)
    assert np.allclose(gv, gv_o, rtol=1e-8, atol=1e-10)
    assert np.allclose(gp, gp_o, rtol=1e-8, atol=1e-10)
    for j in range(3):
        fd = _fd(grid, t, demand, tau, j, kind=kind)
        assert abs(gp[j] - fd) <= 1e-4 * abs(fd), (j, gp[j], fd)
    ctx.close()


@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("tau", TAUS)
def test_soft_fp32_backward_matches_finite_differences(ga, ora, tau, kind):
    """FP32 tables: relative error of d total / d params against FP64 central
    differences of the oracle, bound 1e-4."""
    t, ctx, demand = _setup(ga, 1)
    n = t["nets"]
    print(f"soft fp32 kind={kind} tau={tau} nets={n}", flush=True)
    grid = ora.Grid(t)
    F_o = grid.soft_stage(demand, t["node_off"], t["nodes"], t["parents"], tau, *THETA, kind=kind)
    ctx.set_soft_kind(kind)
    total, _, _ = ctx.soft_forward(0, n, *THETA, tau=tau, precision=32)
    assert abs(total - F_o) <= 1e-4 * abs(F_o)
    gp, _ = ctx.soft_backward()
    errs = []
    for j in range(3):
        fd = _fd(grid, t, demand, tau, j, kind=kind)
        errs.append(abs(gp[j] - fd) / abs(fd))
    print("fp32 relative errors", errs, flush=True)
    assert max(errs) <= 1e-4, errs
    ctx.close()


def test_soft_autograd_function(ga, ora):
    torch = pytest.importorskip("torch")
    from grotor_amd.soft import soft_lshape_cost
    t, ctx, demand = _setup(ga, 2)
    n = t["nets"]
    params = torch.tensor(THETA, dtype=torch.float64, requires_grad=True)
    total = soft_lshape_cost(ctx, params, 0, n, tau=1.0, precision=64)
    total.backward()
    grid = ora.Grid(t)
    _, _, _, gp_o = grid.soft_stage(demand, t["node_off"], t["nodes"], t["parents"], 1.0, *THETA, grads=True)
    assert np.allclose(params.grad.numpy(), gp_o, rtol=1e-8)
    # a later forward invalidates an earlier graph's tables
    p2 = torch.tensor(THETA, dtype=torch.float64, requires_grad=True)
    first = soft_lshape_cost(ctx, p2, 0, n, tau=1.0, precision=32)
    soft_lshape_cost(ctx, p2.detach(), 0, n, tau=1.0, precision=32)
    with pytest.raises(RuntimeError):
        first.backward()
    ctx.close()


def test_soft_batches_sum_to_stage(ga, ora):
    """Forward over two halves equals the whole (per-net values are independent)."""
    t, ctx, demand = _setup(ga, 3)
    n = t["nets"]
    whole, per, _ = ctx.soft_forward(0, n, *THETA, tau=1.0, precision=64, per_net=True)
    a, pa, _ = ctx.soft_forward(0, n // 2, *THETA, tau=1.0, precision=64, per_net=True)
    b, pb, _ = ctx.soft_forward(n // 2, n - n // 2, *THETA, tau=1.0, precision=64, per_net=True)
    assert np.array_equal(np.concatenate([pa, pb]), per)
    assert abs(a + b - whole) <= 1e-12 * abs(whole)
    ctx.close()


@pytest.mark.parametrize("kind", [0, 1])
def test_soft_dag_cost_gradients_match_finite_differences(ga, ora, kind):
    """SoftDagCost over the per-cell cost tensors, FP64: the autograd
    gradients equal the oracle's adjoint, and on cells the nets use they
    agree with central differences of the GPU forward (h = 1e-4) within 1e-4
    relative; a cell no net touches has gradient 0."""
    torch = pytest.importorskip("torch")
    from grotor_amd.soft import soft_dag_cost
    t, ctx, demand = _setup(ga, 4)
    # a slice of the nets keeps F small enough that the central difference's
    # rounding error (eps * |F| / h) stays far below the 1e-4 bound
    n = 64
    print(f"soft dag cost kind={kind} nets={n}", flush=True)
    grid = ora.Grid(t)
    w0, v0, *_ = grid.soft_costs(demand, *THETA)
    tau = 1.0
    wt = torch.tensor(w0, dtype=torch.float64, requires_grad=True)
    vt = torch.tensor(v0, dtype=torch.float64, requires_grad=True)
    total = soft_dag_cost(ctx, wt, vt, 0, n, tau=tau, precision=64, kind=kind)
    total.backward()
    gw, gv = wt.grad.numpy(), vt.grad.numpy()
    off = t["node_off"][:n + 1]
    F_o, gw_o, gv_o, _ = grid.soft_stage(demand, off, t["nodes"][:off[-1]], t["parents"][:off[-1]], tau, *THETA,
                                         grads=True, kind=kind)
    assert abs(total.item() - F_o) <= 1e-10 * abs(F_o)
    assert np.allclose(gw, gw_o, rtol=1e-8, atol=1e-10) and np.allclose(gv, gv_o, rtol=1e-8, atol=1e-10)
    rng = np.random.default_rng(9)
    h = 1e-4
    for name, base, grad in (("w", w0, gw), ("v", v0, gv)):
        used = np.flatnonzero(np.abs(grad) > 1e-2)
        for cell in rng.choice(used, size=min(8, len(used)), replace=False):
            a = base.copy()
            a[cell] += h
            fp = ctx.soft_forward_costs(0, n, a if name == "w" else w0, a if name == "v" else v0, tau, 64)[0]
            a[cell] -= 2 * h
            fm = ctx.soft_forward_costs(0, n, a if name == "w" else w0, a if name == "v" else v0, tau, 64)[0]
            fd = (fp - fm) / (2 * h)
            rounding = 8 * np.finfo(np.float64).eps * abs(F_o) / h
            assert abs(fd - grad[cell]) <= 1e-4 * abs(fd) + rounding, (name, cell, fd, grad[cell], rounding)
        unused = np.flatnonzero(grad == 0)
        assert len(unused) > 0
    ctx.close()


def _soft_trees(rng, L, X, Y):
    """Trees with long, short, straight and zero-length edges, every node
    degree, and one chain taller than 256 levels: (node_off, nodes, parents)."""
    off, nodes, parents = [0], [], []
    for n in (1, 2, 2, 3, 7, 20, 300):
        par = [-1] + [i - 1 if n == 300 else int(rng.integers(0, i)) for i in range(1, n)]
        x, y = rng.integers(0, X, n), rng.integers(0, Y, n)
        if n == 300:  # short steps, so that the oracle's Z-shape edges stay small
            x, y = np.arange(n) % 3 % X, np.arange(n) // 2 % Y
        x[1:][rng.random(n - 1) < 0.2] = x[0]
        if n > 3:
            x[2], y[2] = x[par[2]], y[par[2]]
        if n == 2:
            x[:], y[:] = (0, X - 1), (Y - 1, 0)  # the whole grid, falling
        layer = np.where(rng.random(n) < 0.5, L, rng.integers(0, L, n))
        nodes += ((layer * X + x) * Y + y).tolist()
        parents += par
        off.append(len(nodes))
    return np.array(off, np.int32), np.array(nodes, np.int32), np.array(parents, np.int32)


@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("L,X,Y", [(1, 5, 9), (2, 3, 40), (5, 37, 20), (9, 20, 70), (10, 18, 17)])
def test_soft_trees_of_every_form_match_oracle(ga, ora, L, X, Y, kind):
    """Every lane count (L lanes per node: 64, 32, 12, 7 and 6 nodes per
    wavefront), edges of more bends than they have lanes (16, or 64 on a level
    of few edges), a slot range that does not start at 0, given costs of either
    sign: FP64 equal to the oracle as on the generated instance above."""
    rng = np.random.default_rng(1000 * L + X)
    off, nodes, parents = _soft_trees(rng, L, X, Y)
    t = dict(L=L, X=X, Y=Y, DIR=L & 1, unit_length_wire_cost=0.01, unit_via_cost=0.5,
             unit_length_short_costs=np.full(L, 0.3), x_edge_len=np.full(X - 1, 30, np.int32),
             y_edge_len=np.full(Y - 1, 30, np.int32), capacity=rng.integers(0, 6, L * X * Y).astype(np.float32))
    n = len(off) - 1
    ctx = ga.Context(t)
    ctx.set_routes(off)
    ctx.lshape_upload(np.arange(n), off, nodes, parents)
    demand = random_demand(t, 3, high=4)
    ctx.upload_demand(demand)
    ctx.set_soft_kind(kind)
    grid = ora.Grid(t)
    print(f"soft trees L={L} {X}x{Y} kind={kind}", flush=True)
    for begin in (0, 2):
        o = off[begin:] - off[begin]
        F_o, gw_o, gv_o, gp_o = grid.soft_stage(demand, o, nodes[off[begin]:], parents[off[begin]:], 1.0, *THETA,
                                                grads=True, kind=kind)
        total, _, _ = ctx.soft_forward(begin, n - begin, *THETA, tau=1.0, precision=64)
        gp, _ = ctx.soft_backward()
        gw, gv = ctx.soft_edge_grads()
        assert abs(total - F_o) <= 1e-10 * abs(F_o)
        assert np.allclose(gw, gw_o, rtol=1e-8, atol=1e-10) and np.allclose(gv, gv_o, rtol=1e-8, atol=1e-10)
        assert np.allclose(gp, gp_o, rtol=1e-8, atol=1e-10)
    w, v = rng.normal(0.3, 0.5, L * X * Y), rng.normal(0.5, 0.5, L * X * Y)
    want = sum(np.array(grid.soft_net(w, v, nodes[off[k]:off[k + 1]], parents[off[k]:off[k + 1]], 0.5, kind=kind))
               for k in range(n))
    total, _, _ = ctx.soft_forward_costs(0, n, w, v, 0.5, 64)
    assert abs(total - want) <= 1e-10 * max(1.0, abs(want))
    ctx.close()


def _many_trees(rng, L, X, Y, nets, tall):
    """`nets` small trees in boxes of at most 14 x 14 cells and, next to each
    other in the middle, `tall` chains of 300 nodes: (node_off, nodes,
    parents)."""
    sizes = rng.choice([1, 2, 2, 3, 4, 7, 12], nets)
    sizes[nets // 2:nets // 2 + tall] = 300
    off, nodes, parents = [0], [], []
    for n in sizes:
        ox, oy = rng.integers(0, X - 14), rng.integers(0, Y - 14)
        x, y = ox + rng.integers(0, 14, n), oy + rng.integers(0, 14, n)
        par = [-1] + [int(rng.integers(0, i)) for i in range(1, n)]
        if n == 300:
            x, y, par = ox + np.arange(n) % 3, oy + np.arange(n) // 2 % 14, list(range(-1, n - 1))
        straight = rng.random(n) < 0.2
        x = np.where(straight, x[0], x)
        layer = np.where(rng.random(n) < 0.5, L, rng.integers(0, L, n))
        nodes += ((layer * X + x) * Y + y).tolist()
        parents += par
        off.append(len(nodes))
    return np.array(off, np.int32), np.array(nodes, np.int32), np.array(parents, np.int32)


@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("L,X,Y", [(4, 101, 87), (9, 70, 61)])
def test_soft_chunks_of_several_nets_match_oracle(ga, ora, L, X, Y, kind):
    """More nets than four times the compute units, so that a workgroup takes
    several (5 of 5,203 on 256 units, the last chunk fewer), three chains taller
    than the level bins in one chunk, on a grid whose arrays change their order
    on the device: values, per-cell gradients and given costs against the
    oracle, binary64 closely and binary32 within its rounding: a weight is
    a product over the levels of some eight factors exp(-(x - y) / tau), each
    off by two half units in the last place of a table entry, which on a net's
    routes of any weight is at most the net's value plus 30 tau."""
    rng = np.random.default_rng(10 * L + kind)
    n, tall, tau = 5203, 3, 1.0
    off, nodes, parents = _many_trees(rng, L, X, Y, n, tall)
    t = dict(L=L, X=X, Y=Y, DIR=L & 1, unit_length_wire_cost=0.01, unit_via_cost=0.5,
             unit_length_short_costs=np.full(L, 0.3), x_edge_len=np.full(X - 1, 30, np.int32),
             y_edge_len=np.full(Y - 1, 30, np.int32), capacity=rng.integers(1, 6, L * X * Y).astype(np.float32))
    assert L * X * Y >= 32768
    demand = random_demand(t, 3, high=4)
    ctx = ga.Context(t)
    ctx.set_routes(off)
    ctx.lshape_upload(np.arange(n), off, nodes, parents)
    ctx.upload_demand(demand)
    ctx.set_soft_kind(kind)
    grid = ora.Grid(t)
    print(f"soft chunks L={L} kind={kind}", flush=True)
    # every net in binary64; the nets before the chains in both
    for begin, count, precisions in ((0, n, (64,)), (3, n // 2 - 5, (64, 32))):
        end = begin + count
        o = off[begin:end + 1] - off[begin]
        part = slice(off[begin], off[end])
        F_o, gw_o, gv_o, gp_o = grid.soft_stage(demand, o, nodes[part], parents[part], tau, *THETA, grads=True, kind=kind)
        for precision in precisions:
            total, per_net, _ = ctx.soft_forward(begin, count, *THETA, tau=tau, precision=precision, per_net=True)
            gp, _ = ctx.soft_backward()
            gw, gv = ctx.soft_edge_grads()
            if precision == 64:
                values = per_net
                rel, rtol, atol = 1e-10, 1e-8, 1e-10
            else:
                levels = 12  # a tree of at most 12 nodes
                rel = 8 * levels * 2.0 ** -24
                rtol, atol = levels * 8 * 2 * 2.0 ** -24 * (np.abs(values).max() + 30 * tau) / tau, 1e-10
                assert rtol < 0.01
                assert np.allclose(per_net, values, rtol=rel, atol=rel)
            assert abs(total - F_o) <= rel * abs(F_o)
            assert np.allclose(gw, gw_o, rtol=rtol, atol=atol) and np.allclose(gv, gv_o, rtol=rtol, atol=atol)
            assert np.allclose(gp, gp_o, rtol=rtol, atol=atol)
            print(f"binary{precision} largest difference", np.abs(gw - gw_o).max(), np.abs(gv - gv_o).max(), flush=True)
    w, v = rng.gamma(2.0, 0.3, L * X * Y), rng.gamma(2.0, 0.3, L * X * Y)
    first = n // 2 - 20  # the chains among the nets before and after them
    total, per_net, _ = ctx.soft_forward_costs(first, n - first, w, v, 0.5, 64, per_net=True)
    for k in range(0, 60):
        part = slice(off[first + k], off[first + k + 1])
        want = grid.soft_net(w, v, nodes[part], parents[part], 0.5, kind=kind)
        assert abs(per_net[k] - want) <= 1e-10 * max(1.0, abs(want))
    ctx.close()
