// Soft (log-sum-exp) DP over L-shape or Z-shape edges, and its adjoint,
// for gfx950.
//
// No reference counterpart: a relaxation of the hard pattern-routing DPs in
// which every minimum becomes smin_tau(x) = -tau * log sum exp(-x / tau)
// over the finite entries.  Per net, with intervals lo <= hi of the L
// routing layers:
//   V_i[lo][hi]  via stack sum vcost(l), lo <= l < hi, infinite outside the pin layer
//   D_i          V_i + sum over children c of C_c
//   best_c[k]    smin over intervals containing k of D_c
//   diag_c[e]    smin over the edge's routes leaving the child on layer s
//                and arriving on layer e of best_c[s] + the route's cost
//   C_c[lo][hi]  smin over lo <= h <= hi of diag_c[h]
//   F            smin over all intervals of D_root
// Edge routes of kind 0, the L-shape DP (src/routing/lshape_warp.cuh:8-247,
// lshape.hip here): a straight edge is one wire on a layer of its direction
// (s = e); a bent edge a first leg on s, the corner vias strictly between s
// and e, a second leg on e.  Kind 1, the Z-shape route family
// (src/routing/zshape.cuh:62-288): straight as above (a column when the ends
// share both coordinates); bent: the two L-shapes and the Z-shapes whose
// middle leg runs on a row strictly between the ends' rows or a column
// strictly between their columns, each leg on one layer of its direction
// and a via stack vcost(k), lower <= k < upper layer, at each bend.  Nested
// soft minima compose exactly (smin_x(c_x + smin_y f_xy) = smin_xy(c_x +
// f_xy)), so F is the soft minimum over every route of the family.
//
// The costs are the smooth cost model (src/cost/full_update.cuh:9-83 with
// exact exp; F is differentiable in the overflow slopes and the via weight)
// or arrays the caller gives.  The forward pass checkpoints D, best and diag
// per node; the adjoint replays the tree from the root down, recomputing the
// edges' route costs, with d smin / d x_j = exp(-(x_j - smin) / tau), and
// scatters dF/dwcost (expected wire edge use) and dF/dvcost (expected via
// landings) into FP64 accumulators.
//
// Both passes run level by level over the nodes of a chunk of nets (see
// "chunks of nets" below), L lanes per node, and for kind 1 over the edges of
// a level, 16 lanes each, lane = bend position.  R, the type of the tables and
// of exp / log, is float or double; costs and gradients stay FP64.
#include "gr_kernels.hpp"

namespace grotor {

namespace {

constexpr double kSoftInf = 1e22;
constexpr double kSoftBig = 1e20;

__device__ __forceinline__ double soft_e(double cap, double dem, double s, double z, double& ds, double& dz) {
    ds = dz = 0.0;
    if (cap > 0.001) {
        const double e = exp(s * (dem - cap));
        ds = (dem - cap) * e;
        return e;
    }
    if (dem > 0) {
        const double e = exp(z * dem);
        dz = dem * e;
        return e;
    }
    return 0.0;
}

__device__ __forceinline__ double soft_incr(double cap, double dem, double inc, double sc, double s, double z,
                                            double& ds, double& dz) {
    double s0, z0, s1, z1;
    const double e0 = soft_e(cap, dem, s, z, s0, z0);
    const double e1 = soft_e(cap, dem + inc, s, z, s1, z1);
    const double v = (e1 - e0) * sc;
    if (v >= 1e12) {
        ds = dz = 0.0;
        return 1e12;
    }
    ds = (s1 - s0) * sc;
    dz = (z1 - z0) * sc;
    return v;
}

template <class R>
__device__ __forceinline__ R r_exp(R x);
template <>
__device__ __forceinline__ float r_exp<float>(float x) { return expf(x); }
template <>
__device__ __forceinline__ double r_exp<double>(double x) { return exp(x); }
template <class R>
__device__ __forceinline__ R r_log(R x);
template <>
__device__ __forceinline__ float r_log<float>(float x) { return logf(x); }
template <>
__device__ __forceinline__ double r_log<double>(double x) { return log(x); }

// A soft minimum in progress: value mn - tau * log(s), s = sum of
// exp(-(x - mn) / tau) over the entries so far (empty: mn infinite).
template <class R>
struct Lse {
    R mn, s;
};

template <class R>
__device__ __forceinline__ Lse<R> lse_empty() {
    return Lse<R>{R(kSoftInf), R(0)};
}

template <class R>
__device__ __forceinline__ Lse<R> lse_merge(const Lse<R>& a, const Lse<R>& b, R tau) {
    if (!(b.mn < R(kSoftBig))) return a;
    if (!(a.mn < R(kSoftBig))) return b;
    const R m = a.mn < b.mn ? a.mn : b.mn;
    return Lse<R>{m, a.s * r_exp<R>(-(a.mn - m) / tau) + b.s * r_exp<R>(-(b.mn - m) / tau)};
}

template <class R>
__device__ __forceinline__ R lse_value(const Lse<R>& a, R tau) {
    return a.mn < R(kSoftBig) ? a.mn - tau * r_log<R>(a.s) : R(kSoftInf);
}

template <class R>
__device__ __forceinline__ R soft_weight(R x, R y, R tau) {
    if (!(x < R(kSoftBig)) || !(y < R(kSoftBig))) return R(0);
    return r_exp<R>(-(x - y) / tau);
}

// Wire cost of layer l along its track between positions p0 and p1 of the
// track through `fixed` (x for along_y, else y), from the prefix sums.
__device__ __forceinline__ double leg(const SoftArgs& a, int l, int along_y, int fixed, int p0, int p1) {
    const int lo = min(p0, p1), hi = max(p0, p1);
    const int c0 = along_y ? cell_of(a.g, l, fixed, lo) : cell_of(a.g, l, lo, fixed);
    const int c1 = along_y ? cell_of(a.g, l, fixed, hi) : cell_of(a.g, l, hi, fixed);
    return a.presum[c1] - a.presum[c0];
}
// Checkpointed tables of the nodes [node0, node0 + table_nodes) of the call,
// node by node.
template <class R>
struct SoftTables {
    R *D, *best, *diag, *gdiag, *gbest;
};

template <class R>
__device__ __forceinline__ SoftTables<R> soft_tables(const SoftArgs& a) {
    const int L = a.g.L, T = L * (L + 1) / 2;
    const size_t N = size_t(a.table_nodes);
    SoftTables<R> t;
    t.D = reinterpret_cast<R*>(a.scratch);
    t.best = t.D + N * T;
    t.diag = t.best + N * L;
    t.gdiag = t.diag + N * L;
    t.gbest = t.gdiag + N * L;
    return t;
}

// Geometry of a tree edge from child (x, y) to parent (px, py).
struct Edge {
    int x, y, px, py;
};

}  // namespace

// Smooth costs per track (one workgroup per track): vcost, the exclusive
// prefix of wcost, and the partial derivatives in slope / zero_slope.
__global__ __launch_bounds__(256) void soft_costs_kernel(SoftCostArgs a) {
    const DeviceGrid& g = a.g;
    const int T = blockIdx.x;
    int l = 0;
#pragma unroll
    for (int i = 1; i < kMaxLayers; ++i)
        if (i < g.L && T >= g.track_begin[i]) l = i;
    const int dir = layer_dir(g, l);
    const int len = dir ? g.Y : g.X;
    const int base = l * g.XY + (T - g.track_begin[l]) * len;
    const int* elen = dir ? g.y_edge_len : g.x_edge_len;
    const double sc = g.short_cost[l];
    __shared__ double part[256];
    const int k = (len + blockDim.x - 1) / blockDim.x;
    const int p0 = threadIdx.x * k, p1 = min(len, p0 + k);
    double local = 0.0;
    for (int p = p0; p < p1; ++p) {
        const int i = base + p, q = p > 0 ? i - 1 : i;
        double ws, wz;
        double w = soft_incr(a.capacity[i], a.demand[i], 1.0, sc, a.slope, a.zero_slope, ws, wz);
        if (p < len - 1) w += g.unit_wire * (double)elen[p];
        double v, vs, vz;
        if (p == 0) {
            v = soft_incr(a.capacity[i], a.demand[i], 1.0, sc, a.slope, a.zero_slope, vs, vz);
        } else if (p == len - 1) {
            v = soft_incr(a.capacity[q], a.demand[q], 1.0, sc, a.slope, a.zero_slope, vs, vz);
        } else {
            double s1, z1, s2, z2;
            v = soft_incr(a.capacity[i], a.demand[i], 0.5, sc, a.slope, a.zero_slope, s1, z1) +
                soft_incr(a.capacity[q], a.demand[q], 0.5, sc, a.slope, a.zero_slope, s2, z2);
            vs = s1 + s2;
            vz = z1 + z2;
        }
        a.vcost[i] = v + a.via_weight * g.unit_via;
        a.dw_ds[i] = ws;
        a.dw_dz[i] = wz;
        a.dv_ds[i] = vs;
        a.dv_dz[i] = vz;
        a.wcost[i] = w;
        local += w;
    }
    part[threadIdx.x] = local;
    __syncthreads();
    if (threadIdx.x == 0) {
        double run = 0.0;
        for (int t = 0; t < (int)blockDim.x; ++t) {
            const double v = part[t];
            part[t] = run;
            run += v;
        }
    }
    __syncthreads();
    double run = part[threadIdx.x];
    for (int p = p0; p < p1; ++p) {
        a.presum[base + p] = run;
        run += a.wcost[base + p];
    }
}


// Level order: a node's level is its height in its tree, so a level's nodes
// depend on lower levels only (forward) or on higher ones only (adjoint).
constexpr int kLevelBins = 256;
constexpr int kLevelThreads = 256;

namespace {

// ---- a node on a group of L lanes ----
//
// Lane lo of a group holds row lo of an interval table in registers, entry m
// = interval [lo, lo + m]; entries past the last layer are absent.  What a
// layer needs of the rows that contain it comes by shuffles at distance m,
// so no table goes through LDS.
template <int L>
constexpr int kNodesPerWave = kWave / L;

template <class T>
__device__ __forceinline__ T from_lane(T v, int lane) {
    return __shfl(v, lane, kWave);
}

// an added entry, without a branch: one exponential
template <class R>
__device__ __forceinline__ void lse_push(Lse<R>& a, R x, R tau) {
    const R e = r_exp<R>(-(x < a.mn ? a.mn - x : x - a.mn) / tau);
    const bool fin = x < R(kSoftBig), less = x < a.mn;
    a.s = fin ? (less ? (a.mn < R(kSoftBig) ? a.s * e : R(0)) + R(1) : a.s + e) : a.s;
    a.mn = fin && less ? x : a.mn;
}

// C[lo][lo + m] = smin of diag[lo .. lo + m] for every m of the lane's row,
// handed to f(m, value) in ascending m; dl: the lane's own diag.
template <int L, class R, class F>
__device__ __forceinline__ void closure_row(R dl, int lane, int wl, R tau, F&& f) {
    Lse<R> st = lse_empty<R>();
#pragma unroll
    for (int m = 0; m < L; ++m) {
        const R x = from_lane(dl, lane + m < L ? wl + m : wl);
        if (lane + m < L) {
            lse_push(st, x, tau);
            f(m, lse_value(st, tau));
        }
    }
}

struct SoftNode {
    int x, y, fixed;
};
__device__ __forceinline__ SoftNode soft_node(const DeviceGrid& g, int v) { return SoftNode{v / g.Y % g.X, v % g.Y, v / g.XY}; }

// Kind 0 costs of the edge from (x, y) to (px, py) on lane l: the first leg
// (the whole of a straight edge) and the second leg of layer l, and the via
// costs of layer l at the corners (x, py) and (px, y).
struct EdgeCosts {
    double w1, w2, va, vb;
    bool straight, along;
};
__device__ __forceinline__ EdgeCosts edge_costs(const SoftArgs& a, int l, int x, int y, int px, int py) {
    const int d = layer_dir(a.g, l);
    EdgeCosts c{0.0, 0.0, 0.0, 0.0, x == px || y == py, false};
    c.along = d ? x == px : y == py;
    if (!c.straight || c.along) c.w1 = d ? leg(a, l, 1, x, y, py) : leg(a, l, 0, y, x, px);
    if (!c.straight) {
        c.w2 = d ? leg(a, l, 1, px, y, py) : leg(a, l, 0, py, x, px);
        c.va = a.vcost[cell_of(a.g, l, x, py)];
        c.vb = a.vcost[cell_of(a.g, l, px, y)];
    }
    return c;
}

// Visits the candidates of a bent kind 0 edge on lane pl (arriving layer):
// f(d, down, valid, cl, sum) for the leaving layers cl = pl - d (down) and pl
// + d, odd d, with sum = first leg + corner vias strictly between + second
// leg.  The corner column is (x, py) under a vertical first leg, else (px,
// y); its sums run upwards from the lower of the two layers.
template <int L, class F>
__device__ __forceinline__ void bent_candidates(const DeviceGrid& g, const EdgeCosts& c, int pl, int wl, F&& f) {
    const bool v = layer_dir(g, pl) != 0;
    const double own = v ? c.va : c.vb, other = v ? c.vb : c.va;  // columns of a first leg on pl, on pl +- 1
    double ua = 0.0, ub = 0.0;  // sums over the own / other column of layers pl + 1 .. pl + d - 1
#pragma unroll
    for (int d = 1; d < L; ++d) {
        const bool lo = pl >= d, hi = pl + d < L;
        const int below = lo ? wl - d : wl, above = hi ? wl + d : wl;
        if (d % 2) {
            // lane pl - d's own column is the one of its first leg
            const double fd = from_lane(ua, below), wd = from_lane(c.w1, below), wu = from_lane(c.w1, above);
            f(d, true, lo, pl - d, wd + fd + c.w2);
            f(d, false, hi, pl + d, wu + ub + c.w2);
        }
        // layer pl + d has pl's direction for even d: its own / other columns swap with the parity
        const double ad = from_lane(d % 2 ? other : own, above), bd = from_lane(d % 2 ? own : other, above);
        ua += hi ? ad : 0.0;
        ub += hi ? bd : 0.0;
    }
}

}  // namespace

// Nodes of one level of the forward pass: per node its intervals (via stack
// plus the closures of its children), the soft minima per layer, and for kind
// 0 the edge to its parent; a root's value.  L lanes per node.  Bound by the
// instruction issue of the exponentials and logarithms (about 4 L per lane)
// and the latency of the gathers.  Against one wavefront per net, 465k nodes
// of 8 layers in binary32: 1.61 -> 0.25 ms.
template <class R, int L, int K>
__device__ __forceinline__ void forward_nodes(const SoftArgs& a, const int4* order, int count, int first, int waves) {
    constexpr int T = L * (L + 1) / 2, G = kNodesPerWave<L>;
    const DeviceGrid& g = a.g;
    const R tau = R(a.tau);
    const int wl = threadIdx.x & (kWave - 1), grp = wl / L, lane = wl % L;
    const SoftTables<R> t = soft_tables<R>(a);
    for (int w = first; w * G < count; w += waves) {
        const int k = w * G + grp;
        if (grp >= G || k >= count) continue;  // whole groups: no shuffle crosses a group
        const int4 it = order[k];
        const int node = it.x, n0 = it.y;
        const SoftNode nd = soft_node(g, a.nodes[node]);
        const R via = R(a.vcost[cell_of(g, lane, nd.x, nd.y)]);
        R D[L];
        {
            R s = R(0);
#pragma unroll
            for (int m = 0; m < L; ++m) {
                if (m) s += from_lane(via, lane + m <= L ? wl + m - 1 : wl);
                const bool out = nd.fixed < L && (lane > nd.fixed || lane + m < nd.fixed);
                D[m] = out ? R(kSoftInf) : s;
            }
        }
        for (int c = (a.link[node] & 0xFFFF) - 1; c >= 0; c = (a.link[n0 + c] >> 16) - 1) {
            const R dl = t.diag[size_t(n0 + c - a.node0) * L + lane];
            closure_row<L>(dl, lane, wl, tau, [&](int m, R cv) {
                D[m] = (!(D[m] < R(kSoftBig)) || !(cv < R(kSoftBig))) ? R(kSoftInf) : D[m] + cv;
            });
        }
        R* Dn = t.D + size_t(node - a.node0) * T + (lane * (2 * L - lane + 1)) / 2;
#pragma unroll
        for (int m = 0; m < L; ++m)
            if (lane + m < L) Dn[m] = D[m];
        // S[m] = soft minimum over the row's intervals [lo, hi >= lo + m]
        Lse<R> S[L];
        {
            Lse<R> st = lse_empty<R>();
#pragma unroll
            for (int m = L - 1; m >= 0; --m) {
                if (lane + m < L) lse_push(st, D[m], tau);
                S[m] = st;
            }
        }
        if (it.w < 0) {  // root: over every interval
            Lse<R> st = S[0];
            for (int j = 1; j < L; ++j) {
                const int src = lane == 0 ? wl + j : wl;
                const Lse<R> o{from_lane(S[0].mn, src), from_lane(S[0].s, src)};
                if (lane == 0) st = lse_merge(st, o, tau);
            }
            if (lane == 0) a.value[it.z] = double(lse_value(st, tau));
            continue;
        }
        // layer k: rows k - m, intervals reaching at least k
        Lse<R> bs = S[0];
#pragma unroll
        for (int m = 1; m < L; ++m) {
            const int src = lane >= m ? wl - m : wl;
            const Lse<R> o{from_lane(S[m].mn, src), from_lane(S[m].s, src)};
            if (lane >= m) bs = lse_merge(bs, o, tau);
        }
        const R best = lse_value(bs, tau);
        const size_t row = size_t(node - a.node0) * L + lane;
        t.best[row] = best;
        if (K == 0) {
            const SoftNode pn = soft_node(g, a.nodes[n0 + it.w]);
            const EdgeCosts ec = edge_costs(a, lane, nd.x, nd.y, pn.x, pn.y);
            Lse<R> st = lse_empty<R>();
            if (ec.straight) {
                if (ec.along && best < R(kSoftBig)) lse_push(st, best + R(ec.w1), tau);
            } else {
                bent_candidates<L>(g, ec, lane, wl, [&](int d, bool down, bool valid, int, double sum) {
                    const R b = from_lane(best, valid ? (down ? wl - d : wl + d) : wl);
                    if (valid && b < R(kSoftBig)) lse_push(st, b + R(sum), tau);
                });
            }
            t.diag[row] = lse_value(st, tau);
        }
    }
}

namespace {

// ---- kind 1 edges on 16 lanes ----
constexpr int kZGroup = 16;

// Minimum / sum over a row of `lanes` lanes, the same in each of them.
template <class R, class Op>
__device__ __forceinline__ R row_reduce(R v, int lanes, Op&& op) {
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1)
        if (o < lanes) v = op(v, __shfl_xor(v, o, kWave));
    return v;
}

// sum[s][m] of the via stacks between every pair of layers of opposite
// direction at one place: f(lower, upper, sum), sums running upwards from
// the lower layer.
template <int L, class F>
__device__ __forceinline__ void stack_pairs(const double* v, F&& f) {
#pragma unroll
    for (int lo = 0; lo < L; ++lo) {
        double s = 0.0;
#pragma unroll
        for (int hi = lo + 1; hi < L; ++hi) {
            s += v[hi - 1];
            if ((hi - lo) & 1) f(lo, hi, s);
        }
    }
}

// One bend of an edge: the layers' legs and the two stacks' via costs.  P:
// parity of the layers of the first and last legs.  The corner bend (bend ==
// the child's own row or column) has no first leg and no first stack: the
// middle leg starts at the child.
template <int V>
struct ZParity {
    static constexpr int value = V;
};
template <int L>
struct ZBend {
    double legs[L];  // first leg on layers of parity P, middle leg on the others
    double last[L];  // last leg (parity P)
    double va[L], vb[L];
    bool corner;
};
template <int L, int P>
__device__ __forceinline__ void load_bend(const SoftArgs& a, const Edge& E, int d1, int b, ZBend<L>& z) {
    const int ax = d1 ? E.x : b, ay = d1 ? b : E.y, bx = d1 ? E.px : b, by = d1 ? b : E.py;
    const bool along = d1 ? E.py > E.y : E.px > E.x, across = d1 ? E.px > E.x : E.py > E.y;
    z.corner = b == (d1 ? E.y : E.x);
#pragma unroll
    for (int l = 0; l < L; ++l) {
        const int ca = cell_of(a.g, l, ax, ay), cb = cell_of(a.g, l, bx, by);
        const double pa = a.presum[ca], pb = a.presum[cb];
        if ((l & 1) == P) {
            const double pc = a.presum[cell_of(a.g, l, E.x, E.y)], pp = a.presum[cell_of(a.g, l, E.px, E.py)];
            z.legs[l] = along ? pa - pc : pc - pa;
            z.last[l] = along ? pp - pb : pb - pp;
        } else {
            z.legs[l] = across ? pb - pa : pa - pb;
            z.last[l] = 0.0;
        }
        z.va[l] = a.vcost[ca];
        z.vb[l] = a.vcost[cb];
    }
}

// Soft minima of a bend's routes from the leaving layers: f1[m] per middle
// layer (before the middle leg), mv[e] per arriving layer (before the last
// leg).
template <class R, int L, int P>
__device__ __forceinline__ void bend_minima(const ZBend<L>& z, const R* best, R tau, R* f1, R* mv) {
    Lse<R> s1[L], s2[L];
#pragma unroll
    for (int l = 0; l < L; ++l) s1[l] = s2[l] = lse_empty<R>();
    stack_pairs<L>(z.va, [&](int lo, int hi, double s) {
        const int from = (lo & 1) == P ? lo : hi, to = (lo & 1) == P ? hi : lo;
        if (best[from] < R(kSoftBig)) lse_push(s1[to], best[from] + R(z.legs[from] + s), tau);
    });
#pragma unroll
    for (int m = 0; m < L; ++m)
        if ((m & 1) != P) f1[m] = z.corner ? best[m] : lse_value(s1[m], tau);
    stack_pairs<L>(z.vb, [&](int lo, int hi, double s) {
        const int e = (lo & 1) == P ? lo : hi, m = (lo & 1) == P ? hi : lo;
        if (f1[m] < R(kSoftBig)) lse_push(s2[e], f1[m] + R(z.legs[m] + s), tau);
    });
#pragma unroll
    for (int e = 0; e < L; ++e)
        if ((e & 1) == P) mv[e] = lse_value(s2[e], tau);
}

// The bends of one orientation (d1 = direction of the first leg) of an edge,
// `lanes` at a time: the child's own row (column) and those strictly between.
template <int L, int P, class F>
__device__ __forceinline__ void for_each_bend(const SoftArgs& a, const Edge& E, int d1, int lane, int lanes, F&& f) {
    const int from = d1 ? E.y : E.x, to = d1 ? E.py : E.px, n = abs(to - from);
    for (int b0 = 0; b0 < n; b0 += lanes) {
        const int k = b0 + lane;
        const bool live = k < n;
        ZBend<L> z;
        const int b = to > from ? from + (live ? k : 0) : from - (live ? k : 0);
        load_bend<L, P>(a, E, d1, b, z);
        f(z, b, live, b0);
    }
}

}  // namespace

// Kind 1: edges of one level, 16 lanes each: lane = bend, the lanes' soft
// minima per arriving layer merged over the row (the minimum first, then one
// exponential per lane and layer).  Every via cost and prefix sum of a bend is
// loaded once into registers, where the one-wavefront-per-net form read each
// stack's costs again for every pair of layers.  Bound by the exponentials
// (about L^2 / 2 per bend) at three wavefronts per SIMD.  16 lanes an edge:
// 8 and 4 lanes leave fewer idle on the usual box of 5 x 5 cells but make the
// long edges the tail (forward over 188k nodes, 8 layers, binary32, tau =
// 0.1: 0.66 ms at 16, 0.80 at 8, 0.97 at 4, one launch per level; 0.53 by
// chunks; before, 1.33).  A level of no more edges than the workgroup has
// wavefronts gives each a whole one: with 16 lanes a few long edges leave the
// rest idle (8 chains of 8 nodes across 512 x 512 cells, binary64: 4.51 ms, 1.14
// here, 3.66 with one wavefront per net).
template <class R, int L>
__device__ __forceinline__ void forward_zedges(const SoftArgs& a, const int4* order, int count) {
    const DeviceGrid& g = a.g;
    const R tau = R(a.tau);
    const int group = count <= 256 / kWave ? kWave : kZGroup;
    const SoftTables<R> t = soft_tables<R>(a);
    for (int k = threadIdx.x / group; k < count; k += 256 / group) {
        const int4 it = order[k];
        if (it.w < 0) continue;
        const SoftNode c = soft_node(g, a.nodes[it.x]), p = soft_node(g, a.nodes[it.y + it.w]);
        const Edge E{c.x, c.y, p.x, p.y};
        // short edges keep rows of 16, all four of the wavefront the same
        const int lanes = max(abs(E.x - E.px), abs(E.y - E.py)) <= kZGroup ? kZGroup : group;
        const int lane = threadIdx.x % lanes;
        const R* bn = t.best + size_t(it.x - a.node0) * L;
        R* out = t.diag + size_t(it.x - a.node0) * L;
        if (E.x == E.px || E.y == E.py) {
            const int d = E.x == E.px;  // a column (also when both coordinates agree)
            if (lane < L) {
                R v = R(kSoftInf);
                if (layer_dir(g, lane) == d && bn[lane] < R(kSoftBig))
                    v = bn[lane] + R(d ? leg(a, lane, 1, E.x, E.y, E.py) : leg(a, lane, 0, E.y, E.x, E.px));
                out[lane] = v;
            }
            continue;
        }
        R best[L];
        Lse<R> st[L];
#pragma unroll
        for (int l = 0; l < L; ++l) best[l] = bn[l], st[l] = lse_empty<R>();
        auto pass = [&](auto par, int d1) {
            constexpr int P = decltype(par)::value;
            for_each_bend<L, P>(a, E, d1, lane, lanes, [&](const ZBend<L>& z, int, bool live, int) {
                R f1[L], mv[L];
                bend_minima<R, L, P>(z, best, tau, f1, mv);
#pragma unroll
                for (int e = 0; e < L; ++e)
                    if ((e & 1) == P && live && mv[e] < R(kSoftBig)) lse_push(st[e], mv[e] + R(z.last[e]), tau);
            });
        };
        // layer l runs along y (direction 1) where its parity differs from DIR
        if (g.DIR) {
            pass(ZParity<0>{}, 1);
            pass(ZParity<1>{}, 0);
        } else {
            pass(ZParity<1>{}, 1);
            pass(ZParity<0>{}, 0);
        }
#pragma unroll
        for (int e = 0; e < L; ++e) {
            const R mn = row_reduce(st[e].mn, lanes, [](R u, R v) { return v < u ? v : u; });
            const R s = st[e].mn < R(kSoftBig) ? st[e].s * r_exp<R>(-(st[e].mn - mn) / tau) : R(0);
            const Lse<R> m{mn, row_reduce(s, lanes, [](R u, R v) { return u + v; })};
            if (lane == e) out[e] = lse_value(m, tau);
        }
    }
}

namespace {

// gr added to the wire cells [lo, hi) of layer l's track through `fixed`,
// spread over `width` lanes: consecutive lanes take consecutive cells, which
// is one 64-byte segment for eight of them (scattered atomics run at 24 G/s
// here, eight to a segment at 180 G/s).  Every lane of the group calls it.
__device__ __forceinline__ void spread_leg(const SoftArgs& a, int l, int along_y, int fixed, int p0, int p1, double gr,
                                           int lane, int width) {
    if (gr == 0.0) return;
    const int lo = min(p0, p1), hi = max(p0, p1);
    double* base = a.gw + (along_y ? cell_of(a.g, l, fixed, 0) : cell_of(a.g, l, 0, fixed));
    for (int p = lo + lane; p < hi; p += width) atomicAdd(base + p, gr);
}

// Layer k's sum over the rows that contain it: v[m] of lane k - m, m = 0 ..
// k (row k - m, intervals reaching at least k).
template <int L, class R>
__device__ __forceinline__ R gather_rows(const R (&v)[L], int lane, int wl) {
    R s = v[0];
#pragma unroll
    for (int m = 1; m < L; ++m) {
        const R o = from_lane(v[m], lane >= m ? wl - m : wl);
        s += lane >= m ? o : R(0);
    }
    return s;
}

}  // namespace

// Nodes of one level of the adjoint: for kind 0 the edge of each node to its parent
// (gdiag -> gbest, wires and corner vias), then the node itself: dF/dD of its
// intervals in registers, its via stack, and its children's gdiag.  A root
// starts from its value.  L lanes per node, as in the forward pass.
//  - gD[lo][hi] = sum over k in [lo, hi] of gbest[k] exp(-(D - best[k]) / tau)
//    runs along hi with the terms scaled by the largest best so far (two
//    exponentials an entry instead of one per layer of the interval), and
//    gdiag of a child along hi downwards, its closures growing: every factor
//    stays within (0, 1].
//  - a layer's first legs of all its routes end in one weight, so a leg's
//    cells are added once per layer, by the group's lanes side by side.
// Bound by the atomics' 64-byte segments and the latency of the gathers.
// Against one wavefront per net with an atomic per route and cell from one
// lane, 465k nodes of 8 layers in binary32: 1.78 -> 0.48 ms.
template <class R, int L, int K>
__device__ __forceinline__ void backward_nodes(const SoftArgs& a, const int4* order, int count, int first, int waves) {
    constexpr int T = L * (L + 1) / 2, G = kNodesPerWave<L>;
    const DeviceGrid& g = a.g;
    const R tau = R(a.tau);
    const int wl = threadIdx.x & (kWave - 1), grp = wl / L, lane = wl % L;
    const SoftTables<R> t = soft_tables<R>(a);
    for (int w = first; w * G < count; w += waves) {
        const int k = w * G + grp;
        if (grp >= G || k >= count) continue;  // whole groups: no shuffle crosses a group
        const int4 it = order[k];
        const int node = it.x, n0 = it.y;
        const SoftNode nd = soft_node(g, a.nodes[node]);
        const size_t row = size_t(node - a.node0) * L + lane;
        const R* Dn = t.D + size_t(node - a.node0) * T + (lane * (2 * L - lane + 1)) / 2;
        R D[L], gD[L];
#pragma unroll
        for (int m = 0; m < L; ++m) D[m] = lane + m < L ? Dn[m] : R(kSoftInf);
        if (it.w < 0) {
            const R F = R(a.value[it.z]);
#pragma unroll
            for (int m = 0; m < L; ++m) gD[m] = soft_weight<R>(D[m], F, tau);
        } else {
            const R best = t.best[row];
            R gbest;
            if (K == 0) {
                const R diag = t.diag[row], gdiag = t.gdiag[row];
                const SoftNode pn = soft_node(g, a.nodes[n0 + it.w]);
                const int x = nd.x, y = nd.y, px = pn.x, py = pn.y;
                const EdgeCosts ec = edge_costs(a, lane, x, y, px, py);
                double g1 = 0.0, g2 = 0.0;  // weights of this layer's first and second legs
                if (ec.straight) {
                    g1 = ec.along ? double(gdiag) : 0.0;
                } else {
                    // corner vias of layer l lie strictly inside the candidates
                    // between a lane below and a lane above it; their column
                    // follows the leaving layer's direction, which is l's own
                    // for an arriving layer at odd distance
                    double same = 0.0, other = 0.0;
                    bent_candidates<L>(g, ec, lane, wl, [&](int d, bool down, bool valid, int, double sum) {
                        const R b = from_lane(best, valid ? (down ? wl - d : wl + d) : wl);
                        double gr = 0.0;
                        if (valid && b < R(kSoftBig) && gdiag != R(0))
                            gr = double(gdiag * soft_weight<R>(b + R(sum), diag, tau));
                        g2 += gr;
                        // the leaving lane takes the weight of its first leg
                        const bool has = down ? lane + d < L : lane >= d;
                        const double in = from_lane(gr, has ? (down ? wl + d : wl - d) : wl);
                        g1 += has ? in : 0.0;
#pragma unroll
                        for (int j = 1; j < L; ++j) {
                            if (j >= d) continue;
                            // arriving lane j above (down) or below, reaching past this layer
                            const bool in_range = down ? lane + j < L && lane + j >= d : lane >= j && lane - j + d < L;
                            const double v = from_lane(gr, in_range ? (down ? wl + j : wl - j) : wl);
                            if (j % 2) same += in_range ? v : 0.0;
                            else other += in_range ? v : 0.0;
                        }
                    });
                    const bool v = layer_dir(g, lane) != 0;
                    const double ga = v ? same : other, gb = v ? other : same;  // corners (x, py), (px, y)
                    if (ga != 0.0) atomicAdd(a.gv + cell_of(g, lane, x, py), ga);
                    if (gb != 0.0) atomicAdd(a.gv + cell_of(g, lane, px, y), gb);
                }
#pragma unroll
                for (int l = 0; l < L; ++l) {
                    const int src = wl - lane + l, d = layer_dir(g, l);
                    const double v1 = from_lane(g1, src), v2 = from_lane(g2, src);
                    spread_leg(a, l, d, d ? x : y, d ? y : x, d ? py : px, v1, lane, L);
                    spread_leg(a, l, d, d ? px : py, d ? y : x, d ? py : px, v2, lane, L);
                }
                gbest = R(g1);
            } else {
                gbest = t.gbest[row];
            }
            R mx = -R(kSoftInf), run = R(0);
#pragma unroll
            for (int m = 0; m < L; ++m) {
                const int src = lane + m < L ? wl + m : wl;
                const R b = from_lane(best, src), gb = from_lane(gbest, src);
                gD[m] = R(0);
                if (lane + m < L && b < R(kSoftBig)) {
                    if (gb != R(0)) {
                        const R e = r_exp<R>(-(b < mx ? mx - b : b - mx) / tau);
                        run = b > mx ? run * e + gb : run + gb * e;
                        mx = b > mx ? b : mx;
                    }
                }
                if (lane + m < L && run != R(0) && D[m] < R(kSoftBig)) gD[m] = run * r_exp<R>(-(D[m] - mx) / tau);
            }
        }
        // via stacks: D[lo][hi] holds vcost(l) for lo <= l < hi
        {
            R Q[L], s = R(0);
#pragma unroll
            for (int m = L - 1; m >= 0; --m) {
                Q[m] = s;
                s += gD[m];
            }
            const R v = gather_rows<L>(Q, lane, wl);
            if (lane < L - 1 && v != R(0)) atomicAdd(a.gv + cell_of(g, lane, nd.x, nd.y), double(v));
        }
        // children: dF/d diag[h] = sum over the intervals containing h of
        // gD exp(-(diag[h] - C) / tau)
        for (int c = (a.link[node] & 0xFFFF) - 1; c >= 0; c = (a.link[n0 + c] >> 16) - 1) {
            const size_t crow = size_t(n0 + c - a.node0) * L + lane;
            const R dl = t.diag[crow];
            R C[L], P[L];
#pragma unroll
            for (int m = 0; m < L; ++m) C[m] = R(kSoftInf);
            closure_row<L>(dl, lane, wl, tau, [&](int m, R v) { C[m] = v; });
            R run = R(0), ref = R(kSoftInf);
#pragma unroll
            for (int m = L - 1; m >= 0; --m) {
                const R d = from_lane(dl, lane + m < L ? wl + m : wl);
                P[m] = R(0);
                if (lane + m >= L || !(C[m] < R(kSoftBig))) continue;
                run = (ref < R(kSoftBig) ? run * r_exp<R>(-(C[m] - ref) / tau) : R(0)) + gD[m];
                ref = C[m];
                if (run != R(0) && d < R(kSoftBig)) P[m] = run * r_exp<R>(-(d - C[m]) / tau);
            }
            t.gdiag[crow] = gather_rows<L>(P, lane, wl);
        }
    }
}

namespace {

// Over a row of 16 lanes: the sum up to and including the lane, the sum of
// the lanes after it, and the total.
__device__ __forceinline__ double prefix_sum16(double v, int lane, double& total) {
#pragma unroll
    for (int o = 1; o < kZGroup; o <<= 1) {
        const double u = __shfl_up(v, o, kZGroup);
        v += lane >= o ? u : 0.0;
    }
    total = __shfl(v, kZGroup - 1, kZGroup);
    return v;
}
__device__ __forceinline__ double suffix_sum16(double v, int lane, double& total) {
#pragma unroll
    for (int o = 1; o < kZGroup; o <<= 1) {
        const double u = __shfl_down(v, o, kZGroup);
        v += lane + o < kZGroup ? u : 0.0;
    }
    total = __shfl(v, 0, kZGroup);
    const double after = __shfl_down(v, 1, kZGroup);
    return lane + 1 < kZGroup ? after : 0.0;
}

}  // namespace

// Kind 1: edges of one level of the adjoint, 16 lanes each, lane = bend:
// gdiag -> gbest, and the weights of every route's cells.  The first and last
// legs of the bends cover nested runs of one track per layer, so a cell's
// weight is a running sum over the bends, taken across the lanes, and each
// cell of those tracks is added once per layer by consecutive lanes; a bend's
// middle leg is added by the whole row, bend after bend; a via cell's weight is
// summed over the pairs of layers that pass it before it is added.  Bound by
// latency at two wavefronts per SIMD (binary32; one in binary64) and, on large
// boxes, by the middle legs' atomics.  Against one wavefront per net with an
// atomic per route and cell (8 layers, binary32): 188k nodes, tau = 0.1 1.91
// -> 0.87 ms; 465k nodes, tau = 10 8.0 -> 2.2 ms.
template <class R, int L>
__device__ __forceinline__ void backward_zedges(const SoftArgs& a, const int4* order, int count, int first, int groups) {
    const DeviceGrid& g = a.g;
    const R tau = R(a.tau);
    const int lane = threadIdx.x % kZGroup;
    const SoftTables<R> t = soft_tables<R>(a);
    for (int k = first; k < count; k += groups) {
        const int4 it = order[k];
        if (it.w < 0) continue;
        const SoftNode c = soft_node(g, a.nodes[it.x]), p = soft_node(g, a.nodes[it.y + it.w]);
        const Edge E{c.x, c.y, p.x, p.y};
        const size_t base = size_t(it.x - a.node0) * L;
        if (E.x == E.px || E.y == E.py) {
            const int d = E.x == E.px;
#pragma unroll
            for (int l = 0; l < L; ++l) {
                R w = R(0);
                if (layer_dir(g, l) == d) {
                    w = t.gdiag[base + l];
                    spread_leg(a, l, d, d ? E.x : E.y, d ? E.y : E.x, d ? E.py : E.px, double(w), lane, kZGroup);
                }
                if (lane == l) t.gbest[base + l] = w;
            }
            continue;
        }
        const R *diag = t.diag + base, *gdiag = t.gdiag + base;  // read at their use: registers are short here
        R best[L];
        double gb[L];  // this lane's share of dF/d best
        bool any = false;
#pragma unroll
        for (int l = 0; l < L; ++l) {
            best[l] = t.best[base + l];
            gb[l] = 0.0;
            any |= gdiag[l] != R(0);
        }
        auto pass = [&](auto par, int d1) {
            constexpr int P = decltype(par)::value;
            const int from = d1 ? E.y : E.x, to = d1 ? E.py : E.px, n = abs(to - from);
            const bool up = to > from;
            double before[L];  // last-leg weights of the bends nearer the child
#pragma unroll
            for (int l = 0; l < L; ++l) before[l] = 0.0;
            for_each_bend<L, P>(a, E, d1, lane, kZGroup, [&](const ZBend<L>& z, int b, bool live, int b0) {
                const int ax = d1 ? E.x : b, ay = d1 ? b : E.y, bx = d1 ? E.px : b, by = d1 ? b : E.py;
                const int cell = up ? b : b - 1;  // this lane's cell of the first and last legs' tracks
                R f1[L], mv[L];
                bend_minima<R, L, P>(z, best, tau, f1, mv);
                double gm[L], gf[L], gs[L], via[L];
#pragma unroll
                for (int l = 0; l < L; ++l) {
                    gm[l] = gf[l] = gs[l] = via[l] = 0.0;
                    if ((l & 1) != P) continue;
                    const R gd = gdiag[l], dg = diag[l];
                    if (live && mv[l] < R(kSoftBig) && gd != R(0))
                        gm[l] = double(gd * soft_weight<R>(mv[l] + R(z.last[l]), dg, tau));
                }
                // second bend: the middle layers' weights and its via cells
                stack_pairs<L>(z.vb, [&](int lo, int hi, double s) {
                    const int e = (lo & 1) == P ? lo : hi, m = (lo & 1) == P ? hi : lo;
                    double w = 0.0;
                    if (gm[e] != 0.0 && f1[m] < R(kSoftBig))
                        w = gm[e] * double(soft_weight<R>(f1[m] + R(z.legs[m] + s), mv[e], tau));
                    gf[m] += w;
#pragma unroll
                    for (int l = 0; l < L; ++l)
                        if (l >= lo && l < hi) via[l] += w;
                });
#pragma unroll
                for (int l = 0; l < L; ++l) {
                    if (via[l] != 0.0) atomicAdd(a.gv + cell_of(g, l, bx, by), via[l]);
                    via[l] = 0.0;
                }
                // first bend: the leaving layers' weights and its via cells
                stack_pairs<L>(z.va, [&](int lo, int hi, double s) {
                    const int f = (lo & 1) == P ? lo : hi, m = (lo & 1) == P ? hi : lo;
                    double w = 0.0;
                    if (!z.corner && gf[m] != 0.0 && best[f] < R(kSoftBig))
                        w = gf[m] * double(soft_weight<R>(best[f] + R(z.legs[f] + s), f1[m], tau));
                    gs[f] += w;
#pragma unroll
                    for (int l = 0; l < L; ++l)
                        if (l >= lo && l < hi) via[l] += w;
                });
#pragma unroll
                for (int l = 0; l < L; ++l) {
                    if (via[l] != 0.0) atomicAdd(a.gv + cell_of(g, l, ax, ay), via[l]);
                    gb[l] += (l & 1) == P ? gs[l] : z.corner ? gf[l] : 0.0;
                }
                const int bends = min(kZGroup, n - b0);
#pragma unroll
                for (int l = 0; l < L; ++l) {
                    if ((l & 1) == P) {
                        // cell k of the last leg's track is passed by the bends
                        // up to k, cell k of the first leg's by those after k
                        double total;
                        const double w2 = before[l] + prefix_sum16(gm[l], lane, total);
                        before[l] += total;
                        const double w1 = suffix_sum16(gs[l], lane, total);
                        if (live && w2 != 0.0)
                            atomicAdd(a.gw + (d1 ? cell_of(g, l, E.px, cell) : cell_of(g, l, cell, E.py)), w2);
                        if (live && w1 != 0.0)
                            atomicAdd(a.gw + (d1 ? cell_of(g, l, E.x, cell) : cell_of(g, l, cell, E.y)), w1);
                        // the cells before these 16 bends
                        if (b0) spread_leg(a, l, d1, d1 ? E.x : E.y, from, up ? from + b0 : from - b0, total, lane, kZGroup);
                    } else {
                        for (int q = 0; q < bends; ++q) {
                            const double w = __shfl(gf[l], q, kZGroup);
                            const int bq = __shfl(b, q, kZGroup);
                            spread_leg(a, l, d1 ^ 1, bq, d1 ? E.x : E.y, d1 ? E.px : E.py, w, lane, kZGroup);
                        }
                    }
                }
            });
        };
        if (any) {
            if (g.DIR) {
                pass(ZParity<0>{}, 1);
                pass(ZParity<1>{}, 0);
            } else {
                pass(ZParity<1>{}, 1);
                pass(ZParity<0>{}, 0);
            }
        }
#pragma unroll
        for (int l = 0; l < L; ++l) {
            const double s = row_reduce(gb[l], kZGroup, [](double u, double v) { return u + v; });
            if (lane == l) t.gbest[base + l] = R(s);
        }
    }
}

// ---- chunks of nets ----
//
// Each pass is one launch: a workgroup of four wavefronts takes a chunk of
// nets through their levels, a level's nodes of all its nets at a time, with
// barriers between the levels.  One wavefront per net, its nodes one after
// another, kept 8 of 64 lanes busy; one launch per level over all nets fills
// the chip on the low levels but pays a launch for each of the few nodes of
// the high ones (forward and adjoint of 2k nets, 6k nodes, Z-shape, binary64:
// 0.53 ms against 0.21 here; of 96k nets, 465k nodes, L-shape, binary32 0.86
// against 0.72; before, 0.37 and 3.47).  Nets per chunk: four workgroups a CU
// where the call has that many nets (at least one net, at most 64), between
// the small calls, which want every net on its own (eight a CU: 0.21 ms there
// too), and the large, which want full levels (11k nets, Z-shape, binary32:
// 0.77 ms at four a CU, 1.00 at eight, 1.18 at two).

// The order of a chunk: its nodes by height; those of height kLevelBins - 1
// and above net by net (each net's by height), which the passes take one at a
// time.  start: a row of bins + 1 per chunk.
__global__ __launch_bounds__(kLevelThreads) void soft_chunk_order_kernel(SoftLevelArgs a) {
    __shared__ int s_off[kSoftChunkNets + 1], s_bin[kLevelBins + 1];
    const int k0 = blockIdx.x * a.chunk, nets = min(a.chunk, a.count - k0);
    const int bins = min(a.levels, kLevelBins);
    for (int i = threadIdx.x; i <= nets; i += kLevelThreads) s_off[i] = a.node_off[a.begin + k0 + i];
    for (int h = threadIdx.x; h <= kLevelBins; h += kLevelThreads) s_bin[h] = 0;
    __syncthreads();
    const int q0 = s_off[0], q1 = s_off[nets];
    for (int q = q0 + threadIdx.x; q < q1; q += kLevelThreads) atomicAdd(s_bin + min(a.lvl[q] >> 16, kLevelBins - 1), 1);
    __syncthreads();
    if (threadIdx.x == 0) {
        int run = 0;
        for (int h = 0; h < bins; ++h) {
            const int v = s_bin[h];
            s_bin[h] = run;
            run += v;
        }
        s_bin[bins] = run;
    }
    __syncthreads();
    int* row = a.start + size_t(blockIdx.x) * (bins + 1);
    for (int h = threadIdx.x; h <= bins; h += kLevelThreads) row[h] = s_bin[h];
    __syncthreads();
    int4* order = a.order + (q0 - a.node_off[a.begin]);
    for (int q = q0 + threadIdx.x; q < q1; q += kLevelThreads) {
        const int h = a.lvl[q] >> 16, v = a.lvl[q] & 0xFFFF;
        if (h >= kLevelBins - 1) continue;
        int lo = 0, hi = nets - 1;  // last net that starts at or before q
        while (lo < hi) {
            const int m = (lo + hi + 1) >> 1;
            if (s_off[m] <= q) lo = m;
            else hi = m - 1;
        }
        const int n0 = s_off[lo];
        order[atomicAdd(s_bin + h, 1)] = make_int4(n0 + v, n0, k0 + lo, a.parents[n0 + v]);
    }
    if (threadIdx.x == 0 && bins == kLevelBins) {
        int at = s_bin[kLevelBins - 1];
        for (int i = 0; i < nets; ++i) {
            const int n0 = s_off[i], n = s_off[i + 1] - n0;
            int q = n;  // a net's level order is by height: its tall nodes end it
            while (q > 0 && a.lvl[n0 + q - 1] >> 16 >= kLevelBins - 1) --q;
            for (; q < n; ++q) {
                const int v = a.lvl[n0 + q] & 0xFFFF;
                order[at++] = make_int4(n0 + v, n0, k0 + i, a.parents[n0 + v]);
            }
        }
    }
}

template <class R, int L, int K>
__global__ __launch_bounds__(256) void soft_forward_chunk_kernel(SoftArgs a, SoftLevels lv) {
    const int* start = lv.dstart + size_t(blockIdx.x) * (lv.bins + 1);
    const int4* order = lv.order + (a.node_off[a.begin + blockIdx.x * lv.chunk] - a.node0);
    const int wave = threadIdx.x / kWave;
    const int bins = min(lv.bins, kLevelBins - 1), tall = lv.bins == kLevelBins ? start[bins + 1] - start[bins] : 0;
    for (int h = 0; h < bins + tall; ++h) {
        const int b = h < bins ? start[h] : start[bins] + h - bins, e = h < bins ? start[h + 1] : b + 1;
        if (b == e) break;  // heights are contiguous
        forward_nodes<R, L, K>(a, order + b, e - b, wave, 256 / kWave);
        __syncthreads();
        if (K) {
            forward_zedges<R, L>(a, order + b, e - b);
            __syncthreads();
        }
    }
}

template <class R, int L, int K>
__global__ __launch_bounds__(256, sizeof(R) == 4 ? 2 : 1) void soft_backward_chunk_kernel(SoftArgs a, SoftLevels lv) {
    const int* start = lv.dstart + size_t(blockIdx.x) * (lv.bins + 1);
    const int4* order = lv.order + (a.node_off[a.begin + blockIdx.x * lv.chunk] - a.node0);
    const int wave = threadIdx.x / kWave, group = threadIdx.x / kZGroup;
    const int bins = min(lv.bins, kLevelBins - 1), tall = lv.bins == kLevelBins ? start[bins + 1] - start[bins] : 0;
    for (int h = bins + tall - 1; h >= 0; --h) {
        const int b = h < bins ? start[h] : start[bins] + h - bins, e = h < bins ? start[h + 1] : b + 1;
        if (b == e) continue;
        if (K) {
            backward_zedges<R, L>(a, order + b, e - b, group, 256 / kZGroup);
            __syncthreads();
        }
        backward_nodes<R, L, K>(a, order + b, e - b, wave, 256 / kWave);
        __syncthreads();
    }
}

// Exclusive prefix of given wire costs along each track (one workgroup per
// track), for soft passes over caller-supplied costs.
__global__ __launch_bounds__(256) void soft_prefix_kernel(DeviceGrid g, const double* wcost, double* presum) {
    const int T = blockIdx.x;
    int l = 0;
#pragma unroll
    for (int i = 1; i < kMaxLayers; ++i)
        if (i < g.L && T >= g.track_begin[i]) l = i;
    const int len = layer_dir(g, l) ? g.Y : g.X;
    const int base = l * g.XY + (T - g.track_begin[l]) * len;
    __shared__ double part[256];
    const int k = (len + blockDim.x - 1) / blockDim.x;
    const int p0 = threadIdx.x * k, p1 = min(len, p0 + k);
    double local = 0.0;
    for (int p = p0; p < p1; ++p) local += wcost[base + p];
    part[threadIdx.x] = local;
    __syncthreads();
    if (threadIdx.x == 0) {
        double run = 0.0;
        for (int t = 0; t < (int)blockDim.x; ++t) {
            const double v = part[t];
            part[t] = run;
            run += v;
        }
    }
    __syncthreads();
    double run = part[threadIdx.x];
    for (int p = p0; p < p1; ++p) {
        presum[base + p] = run;
        run += wcost[base + p];
    }
}

// dF/d(slope, zero_slope, via_weight) = sum over cells of the per-cell
// gradients times the cost model's partial derivatives.
__global__ __launch_bounds__(256) void soft_params_kernel(SoftCostArgs c, const double* gw, const double* gv,
                                                          long long cells, double* out) {
    __shared__ double red[3][256];
    double s = 0.0, z = 0.0, u = 0.0;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < cells; i += (long long)gridDim.x * blockDim.x) {
        s += gw[i] * c.dw_ds[i] + gv[i] * c.dv_ds[i];
        z += gw[i] * c.dw_dz[i] + gv[i] * c.dv_dz[i];
        u += gv[i] * c.g.unit_via;
    }
    red[0][threadIdx.x] = s;
    red[1][threadIdx.x] = z;
    red[2][threadIdx.x] = u;
    __syncthreads();
    for (int w = blockDim.x / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w)
            for (int j = 0; j < 3; ++j) red[j][threadIdx.x] += red[j][threadIdx.x + w];
        __syncthreads();
    }
    // three sums per 128-byte stripe, stripes summed by the host
    if (threadIdx.x < 3) atomicAdd(out + (blockIdx.x % kStatStripes) * kCounterStride + threadIdx.x, red[threadIdx.x][0]);
}


size_t soft_scratch_bytes(int L, long long nodes, int precision) {
    const int T = L * (L + 1) / 2;
    return size_t(nodes) * size_t(T + 4 * L) * (precision == 64 ? 8 : 4);
}

void launch_soft_chunks(const SoftLevelArgs& a, hipStream_t st) {
    hipLaunchKernelGGL(soft_chunk_order_kernel, dim3((a.count + a.chunk - 1) / a.chunk), dim3(kLevelThreads), 0, st, a);
}

int soft_level_bins(int levels) { return std::min(levels, kLevelBins); }

namespace {
template <class R, int L>
void forward_chunks(const SoftArgs& a, const SoftLevels& lv, int kind, hipStream_t st) {
    const dim3 grid((a.count + lv.chunk - 1) / lv.chunk);
    if (kind) hipLaunchKernelGGL((soft_forward_chunk_kernel<R, L, 1>), grid, dim3(256), 0, st, a, lv);
    else hipLaunchKernelGGL((soft_forward_chunk_kernel<R, L, 0>), grid, dim3(256), 0, st, a, lv);
}
template <class R, int L>
void backward_chunks(const SoftArgs& a, const SoftLevels& lv, int kind, hipStream_t st) {
    const dim3 grid((a.count + lv.chunk - 1) / lv.chunk);
    if (kind) hipLaunchKernelGGL((soft_backward_chunk_kernel<R, L, 1>), grid, dim3(256), 0, st, a, lv);
    else hipLaunchKernelGGL((soft_backward_chunk_kernel<R, L, 0>), grid, dim3(256), 0, st, a, lv);
}
}  // namespace

void launch_soft_forward(const SoftArgs& a, const SoftLevels& lv, int precision, int kind, hipStream_t st) {
    switch (a.g.L) {
#define GR_SOFT_CASE(n)                                                        \
    case n:                                                                    \
        if (precision == 64) forward_chunks<double, n>(a, lv, kind, st);  \
        else forward_chunks<float, n>(a, lv, kind, st);                   \
        break;
        GR_SOFT_CASE(1) GR_SOFT_CASE(2) GR_SOFT_CASE(3) GR_SOFT_CASE(4) GR_SOFT_CASE(5)
        GR_SOFT_CASE(6) GR_SOFT_CASE(7) GR_SOFT_CASE(8) GR_SOFT_CASE(9) GR_SOFT_CASE(10)
#undef GR_SOFT_CASE
        default: break;
    }
}

void launch_soft_backward(const SoftArgs& a, const SoftLevels& lv, int precision, int kind, hipStream_t st) {
    switch (a.g.L) {
#define GR_SOFT_CASE(n)                                                         \
    case n:                                                                     \
        if (precision == 64) backward_chunks<double, n>(a, lv, kind, st);  \
        else backward_chunks<float, n>(a, lv, kind, st);                   \
        break;
        GR_SOFT_CASE(1) GR_SOFT_CASE(2) GR_SOFT_CASE(3) GR_SOFT_CASE(4) GR_SOFT_CASE(5)
        GR_SOFT_CASE(6) GR_SOFT_CASE(7) GR_SOFT_CASE(8) GR_SOFT_CASE(9) GR_SOFT_CASE(10)
#undef GR_SOFT_CASE
        default: break;
    }
}

}  // namespace grotor
