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
// The forward pass runs level by level over the nodes of all nets (see "level
// order" below), L lanes per node, and for kind 1 over the edges of a level,
// 16 lanes each, lane = bend position; the adjoint one wavefront per net.  R,
// the type of the tables and of exp / log, is float or double; costs and
// gradients stay FP64.
#include "gr_kernels.hpp"

namespace grotor {

namespace {

constexpr double kSoftInf = 1e22;
constexpr double kSoftBig = 1e20;
constexpr int kSoftMaxT = kSoftLayers * (kSoftLayers + 1) / 2;

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
__device__ __forceinline__ void lse_add(Lse<R>& a, R x, R tau) {
    if (!(x < R(kSoftBig))) return;
    if (x < a.mn) {
        a.s = (a.mn < R(kSoftBig) ? a.s * r_exp<R>(-(a.mn - x) / tau) : R(0)) + R(1);
        a.mn = x;
    } else {
        a.s += r_exp<R>(-(x - a.mn) / tau);
    }
}

template <class R>
__device__ __forceinline__ Lse<R> lse_merge(const Lse<R>& a, const Lse<R>& b, R tau) {
    if (!(b.mn < R(kSoftBig))) return a;
    if (!(a.mn < R(kSoftBig))) return b;
    const R m = a.mn < b.mn ? a.mn : b.mn;
    return Lse<R>{m, a.s * r_exp<R>(-(a.mn - m) / tau) + b.s * r_exp<R>(-(b.mn - m) / tau)};
}

// every lane receives the merge of all lanes' states (the butterfly adds
// the same two terms on both partners, so all lanes agree bit for bit)
template <class R>
__device__ __forceinline__ Lse<R> lse_wave(Lse<R> a, R tau) {
    for (int off = kWave / 2; off; off >>= 1) {
        const Lse<R> b{__shfl_xor(a.mn, off, kWave), __shfl_xor(a.s, off, kWave)};
        a = lse_merge(a, b, tau);
    }
    return a;
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

__device__ __forceinline__ double wave_sum(double v) {
    for (int off = kWave / 2; off; off >>= 1) v += __shfl_xor(v, off, kWave);
    return v;
}

__device__ __forceinline__ int tri_index(int L, int lo, int hi) { return lo * (2 * L - lo + 1) / 2 + (hi - lo); }

// Wire cost of layer l along its track between positions p0 and p1 of the
// track through `fixed` (x for along_y, else y), from the prefix sums; the
// gradient variant adds gr to each edge cell [min, max) of the leg.
__device__ __forceinline__ double leg(const SoftArgs& a, int l, int along_y, int fixed, int p0, int p1) {
    const int lo = min(p0, p1), hi = max(p0, p1);
    const int c0 = along_y ? cell_of(a.g, l, fixed, lo) : cell_of(a.g, l, lo, fixed);
    const int c1 = along_y ? cell_of(a.g, l, fixed, hi) : cell_of(a.g, l, hi, fixed);
    return a.presum[c1] - a.presum[c0];
}
__device__ __forceinline__ void leg_grad(const SoftArgs& a, int l, int along_y, int fixed, int p0, int p1, double gr) {
    if (gr == 0.0) return;
    const int lo = min(p0, p1), hi = max(p0, p1);
    for (int p = lo; p < hi; ++p) atomicAdd(a.gw + (along_y ? cell_of(a.g, l, fixed, p) : cell_of(a.g, l, p, fixed)), gr);
}
// via stack at (x, y) between layers l0 and l1: vcost(k), min <= k < max
__device__ __forceinline__ double stack(const SoftArgs& a, int x, int y, int l0, int l1) {
    double s = 0.0;
    for (int k = min(l0, l1); k < max(l0, l1); ++k) s += a.vcost[cell_of(a.g, k, x, y)];
    return s;
}
__device__ __forceinline__ void stack_grad(const SoftArgs& a, int x, int y, int l0, int l1, double gr) {
    if (gr == 0.0) return;
    for (int k = min(l0, l1); k < max(l0, l1); ++k) atomicAdd(a.gv + cell_of(a.g, k, x, y), gr);
}

// Checkpointed tables of the nodes [node0, node0 + table_nodes) of the call,
// node by node.
template <class R>
struct SoftTables {
    R *D, *gD, *best, *diag;
};

template <class R>
__device__ __forceinline__ SoftTables<R> soft_tables(const SoftArgs& a) {
    const int L = a.g.L, T = L * (L + 1) / 2;
    const size_t N = size_t(a.table_nodes);
    SoftTables<R> t;
    t.D = reinterpret_cast<R*>(a.scratch);
    t.gD = t.D + N * T;
    t.best = t.gD + N * T;
    t.diag = t.best + N * L;
    return t;
}

template <class R>
__device__ __forceinline__ SoftTables<R> net_tables(const SoftArgs& a, int slot) {
    const int L = a.g.L, T = L * (L + 1) / 2;
    const size_t n0 = size_t(a.node_off[slot] - a.node0);
    SoftTables<R> t = soft_tables<R>(a);
    t.D += n0 * T;
    t.gD += n0 * T;
    t.best += n0 * L;
    t.diag += n0 * L;
    return t;
}

// Interval table of a workgroup: s_lo[e], s_hi[e] for e = tri_index(L, lo, hi).
__device__ __forceinline__ void interval_table(int L, unsigned char* s_lo, unsigned char* s_hi) {
    const int T = L * (L + 1) / 2;
    for (int e = threadIdx.x; e < T; e += blockDim.x) {
        int lo = 0, rem = e;
        while (rem >= L - lo) rem -= L - lo, ++lo;
        s_lo[e] = (unsigned char)lo;
        s_hi[e] = (unsigned char)(lo + rem);
    }
}

// Geometry of a tree edge from child (x, y) to parent (px, py).
struct Edge {
    int x, y, px, py;
};

// ---- kind 1: the Z-shape route family ----
//
// zedge() visits every route of the edge as (leaving layer s, arriving
// layer e, cost): straight and L-shape routes are split over the lanes by
// arriving layer, the Z-shapes by bend position.  Visit(s, e, cost,
// scatter) is called with the route's cost; in the adjoint pass it returns
// the route's weight and then scatter(w) adds w to the route's cells.  The
// Z-shapes are visited through their nested soft minima: per bend, F1 over
// the leaving layer, M over the middle layer, then the arriving layer.

// Adjoint of zedge_forward: gdiag[e] = dF/d diag[e]; adds each route's
// weight to gb[s] (this lane's share of dF/d best[s]) and its cells.
template <class R>
__device__ __forceinline__ void zedge_backward(const SoftArgs& a, const Edge& E, const R* best, const R* diag,
                                               const R* gdiag, R tau, double* gb) {
    const DeviceGrid& g = a.g;
    const int L = g.L, lane = threadIdx.x;
    const int x = E.x, y = E.y, px = E.px, py = E.py;
    if (x == px || y == py) {
        const int e = lane;
        const int dv = x == px;
        if (e < L && layer_dir(g, e) == dv && gdiag[e] != R(0) && best[e] < R(kSoftBig)) {
            const double c = dv ? leg(a, e, 1, x, y, py) : leg(a, e, 0, y, x, px);
            const double w = double(gdiag[e] * soft_weight<R>(best[e] + R(c), diag[e], tau));
            gb[e] += w;
            if (dv) leg_grad(a, e, 1, x, y, py, w);
            else leg_grad(a, e, 0, y, x, px, w);
        }
        return;
    }
    {
        const int e = lane;
        if (e < L && gdiag[e] != R(0)) {
            const int h = layer_dir(g, e) == 0;  // arriving horizontal: first leg vertical through (x, py)
            const double last = h ? leg(a, e, 0, py, x, px) : leg(a, e, 1, px, y, py);
            double wl = 0.0;
            for (int s = 0; s < L; ++s) {
                if (layer_dir(g, s) != (h ? 1 : 0) || !(best[s] < R(kSoftBig))) continue;
                const double first = h ? leg(a, s, 1, x, y, py) : leg(a, s, 0, y, x, px);
                const double c = first + (h ? stack(a, x, py, s, e) : stack(a, px, y, s, e)) + last;
                const double w = double(gdiag[e] * soft_weight<R>(best[s] + R(c), diag[e], tau));
                if (w == 0.0) continue;
                gb[s] += w;
                wl += w;
                if (h) {
                    leg_grad(a, s, 1, x, y, py, w);
                    stack_grad(a, x, py, s, e, w);
                } else {
                    leg_grad(a, s, 0, y, x, px, w);
                    stack_grad(a, px, y, s, e, w);
                }
            }
            if (h) leg_grad(a, e, 0, py, x, px, wl);
            else leg_grad(a, e, 1, px, y, py, wl);
        }
    }
    for (int pass = 0; pass < 2; ++pass) {
        const int lo = pass == 0 ? min(y, py) : min(x, px), hi = pass == 0 ? max(y, py) : max(x, px);
        const int d1 = pass == 0 ? 1 : 0;
        for (int b0 = lo + 1; b0 < hi; b0 += kWave) {
            const int b = b0 + lane;
            if (b >= hi) continue;
            const int ax = pass == 0 ? x : b, ay = pass == 0 ? b : y;
            const int bx = pass == 0 ? px : b, by = pass == 0 ? b : py;
            R f1[kSoftLayers], mv[kSoftLayers];
            double gf1[kSoftLayers], gm[kSoftLayers];
            for (int m = 0; m < L; ++m) {
                Lse<R> s1 = lse_empty<R>();
                if (layer_dir(g, m) != d1)
                    for (int s = 0; s < L; ++s)
                        if (layer_dir(g, s) == d1 && best[s] < R(kSoftBig)) {
                            const double c = (pass == 0 ? leg(a, s, 1, x, y, b) : leg(a, s, 0, y, x, b)) +
                                             stack(a, ax, ay, s, m);
                            lse_add(s1, best[s] + R(c), tau);
                        }
                f1[m] = lse_value(s1, tau);
                gf1[m] = 0.0;
            }
            for (int e = 0; e < L; ++e) {
                gm[e] = 0.0;
                mv[e] = R(kSoftInf);
                if (layer_dir(g, e) != d1) continue;
                Lse<R> s2 = lse_empty<R>();
                for (int m = 0; m < L; ++m)
                    if (layer_dir(g, m) != d1 && f1[m] < R(kSoftBig)) {
                        const double c = (pass == 0 ? leg(a, m, 0, b, x, px) : leg(a, m, 1, b, y, py)) +
                                         stack(a, bx, by, m, e);
                        lse_add(s2, f1[m] + R(c), tau);
                    }
                mv[e] = lse_value(s2, tau);
                if (mv[e] < R(kSoftBig) && gdiag[e] != R(0)) {
                    const double c = pass == 0 ? leg(a, e, 1, px, b, py) : leg(a, e, 0, py, b, px);
                    gm[e] = double(gdiag[e] * soft_weight<R>(mv[e] + R(c), diag[e], tau));
                    if (pass == 0) leg_grad(a, e, 1, px, b, py, gm[e]);
                    else leg_grad(a, e, 0, py, b, px, gm[e]);
                }
            }
            // middle legs and the second bend's stacks
            for (int m = 0; m < L; ++m) {
                if (layer_dir(g, m) == d1 || !(f1[m] < R(kSoftBig))) continue;
                const double mid = pass == 0 ? leg(a, m, 0, b, x, px) : leg(a, m, 1, b, y, py);
                for (int e = 0; e < L; ++e) {
                    if (layer_dir(g, e) != d1 || gm[e] == 0.0) continue;
                    const double c = mid + stack(a, bx, by, m, e);
                    const double w = gm[e] * double(soft_weight<R>(f1[m] + R(c), mv[e], tau));
                    gf1[m] += w;
                    stack_grad(a, bx, by, m, e, w);
                }
                if (pass == 0) leg_grad(a, m, 0, b, x, px, gf1[m]);
                else leg_grad(a, m, 1, b, y, py, gf1[m]);
            }
            // first legs and the first bend's stacks
            for (int s = 0; s < L; ++s) {
                if (layer_dir(g, s) != d1 || !(best[s] < R(kSoftBig))) continue;
                const double first = pass == 0 ? leg(a, s, 1, x, y, b) : leg(a, s, 0, y, x, b);
                double ws = 0.0;
                for (int m = 0; m < L; ++m) {
                    if (layer_dir(g, m) == d1 || gf1[m] == 0.0) continue;
                    const double c = first + stack(a, ax, ay, s, m);
                    const double w = gf1[m] * double(soft_weight<R>(best[s] + R(c), f1[m], tau));
                    ws += w;
                    stack_grad(a, ax, ay, s, m, w);
                }
                gb[s] += ws;
                if (pass == 0) leg_grad(a, s, 1, x, y, b, ws);
                else leg_grad(a, s, 0, y, x, b, ws);
            }
        }
    }
}

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


// ---- level order ----
//
// Both passes run over the nodes of all nets of the call level by level: a
// node's level is its height in its tree, so a level's nodes depend on lower
// levels only (forward) or on higher ones only (adjoint), and every launch
// has the whole batch's nodes of a level to fill the chip with.  One
// wavefront per net, its nodes one after another, kept 8 of 64 lanes busy and
// every table a dependent round trip away.
//
// The order is three small kernels per (stage, slot range): count the nodes
// per height, scan, place.  Blocks gather their counts in LDS (heights below
// kLevelBins), one atomic per block and height.
constexpr int kLevelBins = 256;
constexpr int kLevelThreads = 256;

__global__ __launch_bounds__(kLevelThreads) void soft_level_count_kernel(SoftLevelArgs a) {
    __shared__ int s_bin[kLevelBins];
    for (int h = threadIdx.x; h < kLevelBins; h += kLevelThreads) s_bin[h] = 0;
    __syncthreads();
    const int q0 = a.node_off[a.begin], q1 = a.node_off[a.begin + a.count];
    for (int q = q0 + blockIdx.x * kLevelThreads + threadIdx.x; q < q1; q += gridDim.x * kLevelThreads) {
        const int h = a.lvl[q] >> 16;
        atomicAdd(h < kLevelBins ? s_bin + h : a.cursor + h, 1);
    }
    __syncthreads();
    for (int h = threadIdx.x; h < min(kLevelBins, a.levels); h += kLevelThreads)
        if (s_bin[h]) atomicAdd(a.cursor + h, s_bin[h]);
}

// cursor[h]: counts in, exclusive prefix out; start[0 .. levels] the same
// with the total at the end.  One workgroup.
__global__ __launch_bounds__(kLevelThreads) void soft_level_scan_kernel(SoftLevelArgs a) {
    __shared__ int s_part[kLevelThreads];
    const int k = (a.levels + kLevelThreads - 1) / kLevelThreads;
    const int p0 = min(a.levels, int(threadIdx.x) * k), p1 = min(a.levels, p0 + k);
    int sum = 0;
    for (int p = p0; p < p1; ++p) sum += a.cursor[p];
    s_part[threadIdx.x] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        int run = 0;
        for (int t = 0; t < kLevelThreads; ++t) {
            const int v = s_part[t];
            s_part[t] = run;
            run += v;
        }
        a.start[a.levels] = run;
    }
    __syncthreads();
    int run = s_part[threadIdx.x];
    for (int p = p0; p < p1; ++p) {
        const int v = a.cursor[p];
        a.cursor[p] = a.start[p] = run;
        run += v;
    }
}

// order[...] = {node, first node of its net, slot - begin, parent (-1: root)};
// one thread per slot
__global__ __launch_bounds__(kLevelThreads) void soft_level_place_kernel(SoftLevelArgs a) {
    __shared__ int s_bin[kLevelBins];
    const int k = blockIdx.x * kLevelThreads + threadIdx.x;
    const int n0 = k < a.count ? a.node_off[a.begin + k] : 0;
    const int n = k < a.count ? a.node_off[a.begin + k + 1] - n0 : 0;
    for (int h = threadIdx.x; h < kLevelBins; h += kLevelThreads) s_bin[h] = 0;
    __syncthreads();
    for (int i = 0; i < n; ++i) {
        const int h = a.lvl[n0 + i] >> 16;
        if (h < kLevelBins) atomicAdd(s_bin + h, 1);
    }
    __syncthreads();
    for (int h = threadIdx.x; h < min(kLevelBins, a.levels); h += kLevelThreads)
        if (s_bin[h]) s_bin[h] = atomicAdd(a.cursor + h, s_bin[h]);
    __syncthreads();
    for (int i = 0; i < n; ++i) {
        const int q = a.lvl[n0 + i], h = q >> 16, v = q & 0xFFFF;
        const int at = atomicAdd(h < kLevelBins ? s_bin + h : a.cursor + h, 1);
        a.order[at] = make_int4(n0 + v, n0, k, a.parents[n0 + v]);
    }
}

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

// One level of the forward pass: per node its intervals (via stack plus the
// closures of its children), the soft minima per layer, and for kind 0 the
// edge to its parent; a root's value.  L lanes per node.  Bound by the
// instruction issue of the exponentials and logarithms (about 4 L per lane)
// and, on the upper levels, by the launch itself.  Against one wavefront per
// net, forward over 465k nodes of 8 layers in binary32: 1.61 -> 0.33 ms.
template <class R, int L, int K>
__global__ __launch_bounds__(256) void soft_forward_level_kernel(SoftArgs a, const int4* order, int count) {
    constexpr int T = L * (L + 1) / 2, G = kNodesPerWave<L>;
    const DeviceGrid& g = a.g;
    const R tau = R(a.tau);
    const int wl = threadIdx.x & (kWave - 1), grp = wl / L, lane = wl % L;
    const SoftTables<R> t = soft_tables<R>(a);
    const int waves = gridDim.x * (256 / kWave);
    for (int w = blockIdx.x * (256 / kWave) + threadIdx.x / kWave; w * G < count; w += waves) {
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

// Minimum / sum over a row of 16 lanes, the same in each of them.
template <class R, class Op>
__device__ __forceinline__ R row_reduce(R v, Op&& op) {
#pragma unroll
    for (int o = 1; o < kZGroup; o <<= 1) v = op(v, __shfl_xor(v, o, kWave));
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
// kZGroup at a time: the child's own row (column) and those strictly between.
template <int L, int P, class F>
__device__ __forceinline__ void for_each_bend(const SoftArgs& a, const Edge& E, int d1, int lane, F&& f) {
    const int from = d1 ? E.y : E.x, to = d1 ? E.py : E.px, n = abs(to - from);
    for (int b0 = 0; b0 < n; b0 += kZGroup) {
        const int k = b0 + lane;
        const bool live = k < n;
        ZBend<L> z;
        const int b = to > from ? from + (live ? k : 0) : from - (live ? k : 0);
        load_bend<L, P>(a, E, d1, b, z);
        f(z, b, live, b0);
    }
}

}  // namespace

// Kind 1: one level's edges, 16 lanes each: lane = bend, the lanes' soft
// minima per arriving layer merged over the row (the minimum first, then one
// exponential per lane and layer).  Every via cost and prefix sum of a bend is
// loaded once into registers, where the one-wavefront-per-net form read each
// stack's costs again for every pair of layers.  Bound by the exponentials
// (about L^2 / 2 per bend) at three wavefronts per SIMD.  16 lanes an edge:
// 8 and 4 lanes leave fewer idle on the usual box of 5 x 5 cells but make the
// long edges the tail (forward over 188k nodes, 8 layers, binary32, tau =
// 0.1: 0.66 ms at 16, 0.80 at 8, 0.97 at 4; before, 1.33).
template <class R, int L>
__global__ __launch_bounds__(256) void soft_zedge_level_kernel(SoftArgs a, const int4* order, int count) {
    const DeviceGrid& g = a.g;
    const R tau = R(a.tau);
    const int lane = threadIdx.x % kZGroup;
    const SoftTables<R> t = soft_tables<R>(a);
    const int groups = gridDim.x * (256 / kZGroup);
    for (int k = blockIdx.x * (256 / kZGroup) + threadIdx.x / kZGroup; k < count; k += groups) {
        const int4 it = order[k];
        if (it.w < 0) continue;
        const SoftNode c = soft_node(g, a.nodes[it.x]), p = soft_node(g, a.nodes[it.y + it.w]);
        const Edge E{c.x, c.y, p.x, p.y};
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
            for_each_bend<L, P>(a, E, d1, lane, [&](const ZBend<L>& z, int, bool live, int) {
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
            const R mn = row_reduce(st[e].mn, [](R u, R v) { return v < u ? v : u; });
            const R s = st[e].mn < R(kSoftBig) ? st[e].s * r_exp<R>(-(st[e].mn - mn) / tau) : R(0);
            const Lse<R> m{mn, row_reduce(s, [](R u, R v) { return u + v; })};
            if (lane == e) out[e] = lse_value(m, tau);
        }
    }
}

// One wavefront per net (grid-stride over the slots [begin, begin + count)).
template <class R, int K>
__global__ __launch_bounds__(kWave) void soft_backward_kernel(SoftArgs a) {
    __shared__ unsigned char s_lo[kSoftMaxT], s_hi[kSoftMaxT];
    __shared__ R s_C[kSoftMaxT], s_gC[kSoftMaxT];
    __shared__ R s_best[kSoftLayers], s_diag[kSoftLayers], s_gdiag[kSoftLayers], s_gbest[kSoftLayers];
    const int lane = threadIdx.x;
    const DeviceGrid& g = a.g;
    const int L = g.L, X = g.X, Y = g.Y, T = L * (L + 1) / 2;
    const R tau = R(a.tau);
    interval_table(L, s_lo, s_hi);
    __syncthreads();
    for (int slot = a.begin + blockIdx.x; slot < a.begin + a.count; slot += gridDim.x) {
        const int n0 = a.node_off[slot], n = a.node_off[slot + 1] - n0;
        const int* nodes = a.nodes + n0;
        const int* parents = a.parents + n0;
        const SoftTables<R> t = net_tables<R>(a, slot);
        const R F = R(a.value[slot - a.begin]);
        if (!(F < R(kSoftBig))) continue;  // uniform over the wave
        for (int e = lane; e < T; e += kWave) t.gD[e] = soft_weight<R>(t.D[e], F, tau);
        __syncthreads();
        for (int c = 1; c < n; ++c) {
            const int p = parents[c];
            const Edge E{nodes[c] / Y % X, nodes[c] % Y, nodes[p] / Y % X, nodes[p] % Y};
            const R* dg = t.diag + size_t(c) * L;
            const R* gC = t.gD + size_t(p) * T;
            for (int e = lane; e < T; e += kWave) {
                Lse<R> st = lse_empty<R>();
                for (int h = s_lo[e]; h <= s_hi[e]; ++h) lse_add(st, dg[h], tau);
                s_C[e] = lse_value(st, tau);
                s_gC[e] = gC[e];
            }
            if (lane < L) {
                s_best[lane] = t.best[size_t(c) * L + lane];
                s_diag[lane] = dg[lane];
            }
            __syncthreads();
            if (lane < L) {
                const int h = lane;
                R s = 0;
                for (int lo = 0; lo <= h; ++lo)
                    for (int hi = h; hi < L; ++hi) {
                        const int e = tri_index(L, lo, hi);
                        if (s_gC[e] != R(0)) s += s_gC[e] * soft_weight<R>(s_diag[h], s_C[e], tau);
                    }
                s_gdiag[h] = s;
            }
            __syncthreads();
            double gb[kSoftLayers];
#pragma unroll
            for (int k = 0; k < kSoftLayers; ++k) gb[k] = 0.0;
            if (K == 0) {
                const int x = E.x, y = E.y, px = E.px, py = E.py;
                const bool straight = x == px || y == py;
                if (lane < L && s_gdiag[lane] != R(0)) {
                    const int pl = lane, d = layer_dir(g, pl);
                    if (straight) {
                        if (d ? x == px : y == py) {
                            gb[pl] += double(s_gdiag[pl]);
                            if (d) leg_grad(a, pl, 1, x, y, py, double(s_gdiag[pl]));
                            else leg_grad(a, pl, 0, y, x, px, double(s_gdiag[pl]));
                        }
                    } else {
                        // the forward's candidate values, recomputed the same way
                        const double wpl = d ? leg(a, pl, 1, px, y, py) : leg(a, pl, 0, py, x, px);
                        double w2 = 0.0;
                        for (int cl = (pl & 1) ^ 1; cl < L; cl += 2) {
                            if (!(s_best[cl] < R(kSoftBig))) continue;
                            const int lo = min(cl, pl), hi = max(cl, pl);
                            const int dcl = layer_dir(g, cl);
                            double f = 0.0;
                            for (int l = lo + 1; l < hi; ++l)
                                f += dcl ? a.vcost[cell_of(g, l, x, py)] : a.vcost[cell_of(g, l, px, y)];
                            const double wcl = dcl ? leg(a, cl, 1, x, y, py) : leg(a, cl, 0, y, x, px);
                            const R tc = s_best[cl] + R(wcl + f + wpl);
                            const double gr = double(s_gdiag[pl] * soft_weight<R>(tc, s_diag[pl], tau));
                            if (gr == 0.0) continue;
                            gb[cl] += gr;
                            w2 += gr;
                            if (dcl) leg_grad(a, cl, 1, x, y, py, gr);
                            else leg_grad(a, cl, 0, y, x, px, gr);
                            for (int l = lo + 1; l < hi; ++l)
                                atomicAdd(a.gv + (dcl ? cell_of(g, l, x, py) : cell_of(g, l, px, y)), gr);
                        }
                        if (d) leg_grad(a, pl, 1, px, y, py, w2);
                        else leg_grad(a, pl, 0, py, x, px, w2);
                    }
                }
            } else {
                zedge_backward<R>(a, E, s_best, s_diag, s_gdiag, tau, gb);
            }
            for (int k = 0; k < L; ++k) {
                const double v = wave_sum(gb[k]);
                if (lane == k) s_gbest[k] = R(v);
            }
            __syncthreads();
            const R* Dc = t.D + size_t(c) * T;
            R* gDc = t.gD + size_t(c) * T;
            for (int e = lane; e < T; e += kWave) {
                R s = 0;
                const R d = Dc[e];
                for (int k = s_lo[e]; k <= s_hi[e]; ++k)
                    if (s_gbest[k] != R(0)) s += s_gbest[k] * soft_weight<R>(d, s_best[k], tau);
                gDc[e] = s;
            }
            __syncthreads();
        }
        // via stacks: D_i[lo][hi] holds vcost(l) for lo <= l < hi
        for (int q = lane; q < n * (L - 1); q += kWave) {
            const int i = q / (L - 1), l = q % (L - 1);
            const int x = nodes[i] / Y % X, y = nodes[i] % Y;
            R s = 0;
            for (int lo = 0; lo <= l; ++lo)
                for (int hi = l + 1; hi < L; ++hi) s += t.gD[size_t(i) * T + tri_index(L, lo, hi)];
            if (s != R(0)) atomicAdd(a.gv + cell_of(g, l, x, y), double(s));
        }
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
    return size_t(nodes) * size_t(2 * T + 2 * L) * (precision == 64 ? 8 : 4);
}

void launch_soft_levels(const SoftLevelArgs& a, int nodes, int cus, hipStream_t st) {
    const int blocks = std::max(1, std::min((nodes + kLevelThreads - 1) / kLevelThreads, std::max(1, cus) * 4));
    hipLaunchKernelGGL(fill_int_kernel, dim3((a.levels + 255) / 256), dim3(256), 0, st, a.cursor, 0, (long long)a.levels);
    hipLaunchKernelGGL(soft_level_count_kernel, dim3(blocks), dim3(kLevelThreads), 0, st, a);
    hipLaunchKernelGGL(soft_level_scan_kernel, dim3(1), dim3(kLevelThreads), 0, st, a);
    hipLaunchKernelGGL(soft_level_place_kernel, dim3((a.count + kLevelThreads - 1) / kLevelThreads), dim3(kLevelThreads),
                       0, st, a);
}

namespace {
int soft_grid(const SoftArgs& a, int cus) { return std::max(1, std::min(a.count, std::max(1, cus) * 32)); }

// workgroups for `count` items of `per` items a workgroup, at most 16 a CU
int level_grid(int count, int per, int cus) { return std::max(1, std::min((count + per - 1) / per, std::max(1, cus) * 16)); }

template <class R, int L>
void forward_levels(const SoftArgs& a, const SoftLevels& lv, int kind, int cus, hipStream_t st) {
    for (int h = 0; h + 1 < int(lv.start.size()); ++h) {
        const int count = lv.start[h + 1] - lv.start[h];
        if (!count) continue;
        const int4* order = lv.order + lv.start[h];
        const dim3 grid(level_grid(count, 256 / kWave * kNodesPerWave<L>, cus));
        if (kind) {
            hipLaunchKernelGGL((soft_forward_level_kernel<R, L, 1>), grid, dim3(256), 0, st, a, order, count);
            hipLaunchKernelGGL((soft_zedge_level_kernel<R, L>), dim3(level_grid(count, 256 / kZGroup, cus)), dim3(256), 0,
                               st, a, order, count);
        } else {
            hipLaunchKernelGGL((soft_forward_level_kernel<R, L, 0>), grid, dim3(256), 0, st, a, order, count);
        }
    }
}
}  // namespace

void launch_soft_forward(const SoftArgs& a, const SoftLevels& lv, int precision, int kind, int cus, hipStream_t st) {
    switch (a.g.L) {
#define GR_SOFT_CASE(n)                                                        \
    case n:                                                                    \
        if (precision == 64) forward_levels<double, n>(a, lv, kind, cus, st);  \
        else forward_levels<float, n>(a, lv, kind, cus, st);                   \
        break;
        GR_SOFT_CASE(1) GR_SOFT_CASE(2) GR_SOFT_CASE(3) GR_SOFT_CASE(4) GR_SOFT_CASE(5)
        GR_SOFT_CASE(6) GR_SOFT_CASE(7) GR_SOFT_CASE(8) GR_SOFT_CASE(9) GR_SOFT_CASE(10)
#undef GR_SOFT_CASE
        default: break;
    }
}

void launch_soft_backward(const SoftArgs& a, int precision, int kind, int cus, hipStream_t st) {
    const dim3 grid(soft_grid(a, cus));
    if (precision == 64) {
        if (kind) hipLaunchKernelGGL((soft_backward_kernel<double, 1>), grid, dim3(kWave), 0, st, a);
        else hipLaunchKernelGGL((soft_backward_kernel<double, 0>), grid, dim3(kWave), 0, st, a);
    } else {
        if (kind) hipLaunchKernelGGL((soft_backward_kernel<float, 1>), grid, dim3(kWave), 0, st, a);
        else hipLaunchKernelGGL((soft_backward_kernel<float, 0>), grid, dim3(kWave), 0, st, a);
    }
}

}  // namespace grotor
