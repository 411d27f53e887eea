// Z-shape pattern routing (GGR) for gfx950.
//
// Reference: zshape::solve<Warps>, viaSweep and reset_nodes
// (src/routing/zshape.cuh:42-404), convert_routes
// (src/routing/zshape_topology.hpp:233-289).
//
// Two forms.  zshape_net_kernel (end of this file) routes a net with its DP
// in LDS and takes every net that fits; the general kernels take the rest
// (large trees, nodes with two parents, and whole plans with a record whose
// words rest on what earlier nets left on the shared map).  In the
// general form one 64-lane wavefront routes one tree (the reference uses a
// 32-lane warp).  Nets of a batch have disjoint bounding boxes, so they share one
// map of LAYER = L + 1 planes of n x n cells (n = max(X, Y)) without
// touching each other's cells; map layer i is routing layer i - 1 and its
// second index runs along the layer's tracks.  Per tree edge (child -> node)
// the phases are: clear the box's two rows and two columns on plane 4; first
// leg along the child's row/column; via sweeps at every cell of that leg;
// middle leg across the box; via sweeps on the node's row/column; last leg
// into child slot j of the node.  Lanes take disjoint cells in every phase,
// so the values equal a sequential run; the last leg's per-layer first
// minimum is a wavefront reduction.  Each cell's via sweep, the child's
// value in the first leg and the node's interval combination work on values
// loaded once into registers instead of chains of dependent global accesses.
// The node's interval combination and the traceback run on lane 0, as in
// the reference.  Costs are integers:
// int(min(|presum(a) - presum(b)|, 5e8)) per wire, int(clamp(vcost, 1, 1e6))
// per via landing.  Indices decoded from the traceback tables are checked
// against the map before use; a bad one sets the error word.
#include "gr_kernels.hpp"

namespace grotor {

namespace {

constexpr int kZInf = 1000000000;

struct Z {
    const ZshapeArgs& a;
    long long nn, P;
    __device__ Z(const ZshapeArgs& args) : a(args), nn((long long)args.n * args.n), P(args.layers * nn) {}
    __device__ __forceinline__ bool vert(int i) const { return ((i & 1) ^ a.dirv) != 0; }
    __device__ __forceinline__ long long cell(int i, int x, int y) const {
        return i * nn + (vert(i) ? (long long)x * a.n + y : (long long)y * a.n + x);
    }
    // the same (x, y) in the orientation of the layer next to i
    __device__ __forceinline__ long long cell_swapped(int i_other, int i, int x, int y) const {
        return i_other * nn + (vert(i) ? (long long)y * a.n + x : (long long)x * a.n + y);
    }
    __device__ __forceinline__ double wire_sum(long long index) const {
        const int layer = int(index / nn) - 1;
        if (layer < 0 || layer >= a.g.L) return 0.0;
        const int p = int(index / a.n % a.n), q = int(index % a.n);
        const bool along_y = layer_dir(a.g, layer);
        return a.presum[cell_of(a.g, layer, along_y ? p : q, along_y ? q : p)];
    }
    __device__ __forceinline__ int via(long long index) const {
        const int layer = int(index / nn) - 1;
        if (layer < 0 || layer >= a.g.L) return kZInf;
        const int p = int(index / a.n % a.n), q = int(index % a.n);
        const bool along_y = layer_dir(a.g, layer);
        return (int)fminf(fmaxf(a.vcost[cell_of(a.g, layer, along_y ? p : q, along_y ? q : p)], 1.f), 1.e6f);
    }
    __device__ __forceinline__ int wire(long long p, long long q) const {
        return (int)fmin(fabs(wire_sum(p) - wire_sum(q)), double(kZInf / 2));
    }
    // wire(p, q) with wire_sum(p) already loaded
    __device__ __forceinline__ int wire_from(double wp, long long q) const {
        return (int)fmin(fabs(wp - wire_sum(q)), double(kZInf / 2));
    }
};

// The via sweeps at one (x, y) of plane 4: upwards then downwards through
// the layer stack, each step taking the neighbour's value plus the via cost
// when it is smaller.  The stack is loaded once and swept in registers, in
// the reference's order (zshape.cuh viaSweep); only this lane touches it.
__device__ void via_sweep(const Z& z, int x, int y) {
    int* m = z.a.map + 4 * z.P;
    int* pr = z.a.prev + 4 * z.P;
    const int L1 = z.a.layers;
    long long idx[kMaxLayers];
    int mv[kMaxLayers], pv[kMaxLayers], pl[kMaxLayers], vc[kMaxLayers];
#pragma unroll
    for (int i = 1; i < kMaxLayers; i++) {
        if (i >= L1) continue;
        idx[i] = z.cell(i, x, y);
        mv[i] = m[idx[i]];
        pv[i] = pr[idx[i]];
        pl[i] = (int)idx[i];
        vc[i] = i < L1 - 1 ? z.via(idx[i]) : 0;
    }
#pragma unroll
    for (int i = 2; i < kMaxLayers; i++) {
        if (i >= L1) continue;
        const int v = mv[i - 1] + vc[i - 1];
        if (mv[i] > v) {
            mv[i] = v;
            pv[i] = pv[i - 1];
            pl[i] = (int)idx[i - 1];
        }
    }
#pragma unroll
    for (int i = kMaxLayers - 2; i >= 1; i--) {
        if (i > L1 - 2) continue;
        const int v = mv[i + 1] + vc[i];
        if (mv[i] > v) {
            mv[i] = v;
            pv[i] = pv[i + 1];
            pl[i] = (int)idx[i + 1];
        }
    }
#pragma unroll
    for (int i = 1; i < kMaxLayers; i++) {
        if (i >= L1) continue;
        m[idx[i]] = mv[i];
        pr[idx[i]] = pv[i];
        pr[idx[i] + z.P] = pl[i];
    }
}

__device__ void zedge(const Z& z, int lane, int j, int fromx, int fromy, int tox, int toy) {
    const ZshapeArgs& a = z.a;
    const long long nn = z.nn, P = z.P;
    const int L1 = a.layers, n = a.n;
    int* map = a.map;
    int* prev = a.prev;
    int* prev2 = a.prev + 10 * P;
    int* m4 = map + 4 * P;
    int* p4 = prev + 4 * P;
    const int x0 = min(fromx, tox), x1 = max(fromx, tox), y0 = min(fromy, toy), y1 = max(fromy, toy);
    if (fromx != tox && fromy != toy) {
        for (int q = x0 + lane; q <= x1; q += kWave)
            for (int i = 1; i < L1; i++) {
                if (z.vert(i)) {
                    m4[i * nn + (long long)q * n + toy] = kZInf;
                    m4[i * nn + (long long)q * n + fromy] = kZInf;
                } else {
                    m4[i * nn + (long long)toy * n + q] = kZInf;
                    m4[i * nn + (long long)fromy * n + q] = kZInf;
                }
            }
        __syncthreads();
        for (int q = y0 + lane; q <= y1; q += kWave)
            for (int i = 1; i < L1; i++) {
                if (z.vert(i)) {
                    m4[i * nn + (long long)tox * n + q] = kZInf;
                    m4[i * nn + (long long)fromx * n + q] = kZInf;
                } else {
                    m4[i * nn + (long long)q * n + tox] = kZInf;
                    m4[i * nn + (long long)q * n + fromx] = kZInf;
                }
            }
        __syncthreads();
        // first leg along the child's column (vertical layers) or row
        // (horizontal layers); the child's value and prefix sum per layer are
        // loaded once, and the layers need no barrier between them
        {
            int cv[kMaxLayers];
            double cw[kMaxLayers];
#pragma unroll
            for (int i = 1; i < kMaxLayers; i++) {
                if (i >= L1) continue;
                const long long last = z.vert(i) ? i * nn + (long long)fromx * n + fromy : i * nn + (long long)fromy * n + fromx;
                cv[i] = map[last];
                cw[i] = z.wire_sum(last);
            }
            for (int q = y0 + lane; q <= y1; q += kWave) {
                if (q == fromy) continue;
#pragma unroll
                for (int i = 1; i < kMaxLayers; i++) {
                    if (i >= L1 || !z.vert(i)) continue;
                    const long long cur = i * nn + (long long)fromx * n + q;
                    m4[cur] = cv[i] + z.wire_from(cw[i], cur);
                    p4[cur] = (int)(i * nn + (long long)fromx * n + fromy);
                }
            }
            for (int q = x0 + lane; q <= x1; q += kWave) {
                if (q == fromx) continue;
#pragma unroll
                for (int i = 1; i < kMaxLayers; i++) {
                    if (i >= L1 || z.vert(i)) continue;
                    const long long cur = i * nn + (long long)fromy * n + q;
                    m4[cur] = cv[i] + z.wire_from(cw[i], cur);
                    p4[cur] = (int)(i * nn + (long long)fromy * n + fromx);
                }
            }
            __syncthreads();
        }
        for (int q = y0 + lane; q <= y1; q += kWave)
            if (q != fromy) via_sweep(z, fromx, q);
        __syncthreads();
        for (int q = x0 + lane; q <= x1; q += kWave)
            if (q != fromx) via_sweep(z, q, fromy);
        __syncthreads();
        // middle leg across the box: vertical layers from row fromy to row
        // toy, horizontal layers from column fromx to column tox; cells of
        // different layers and lanes are disjoint, so one barrier suffices
        for (int q = x0 + lane; q <= x1; q += kWave) {
#pragma unroll
            for (int i = 1; i < kMaxLayers; i++) {
                if (i >= L1 || !z.vert(i)) continue;
                const long long last = i * nn + (long long)q * n + fromy, cur = i * nn + (long long)q * n + toy;
                const int cost = z.wire(last, cur), ml = m4[last], mc = m4[cur], pl = p4[last];
                if (ml + cost < mc) {
                    m4[cur] = ml + cost;
                    p4[cur] = pl;
                }
            }
        }
        for (int q = y0 + lane; q <= y1; q += kWave) {
#pragma unroll
            for (int i = 1; i < kMaxLayers; i++) {
                if (i >= L1 || z.vert(i)) continue;
                const long long last = i * nn + (long long)q * n + fromx, cur = i * nn + (long long)q * n + tox;
                const int cost = z.wire(last, cur), ml = m4[last], mc = m4[cur], pl = p4[last];
                if (ml + cost < mc) {
                    m4[cur] = ml + cost;
                    p4[cur] = pl;
                }
            }
        }
        __syncthreads();
        for (int q = y0 + lane; q <= y1; q += kWave)
            if (q != toy) via_sweep(z, tox, q);
        __syncthreads();
        for (int q = x0 + lane; q <= x1; q += kWave)
            if (q != tox) via_sweep(z, q, toy);
        __syncthreads();
        // last leg into child slot j of the node, per layer the first
        // minimum over the leg's cells in ascending order: each lane takes
        // every 64th cell, then a wavefront reduction keeps the smallest
        // value and, among equal values, the smallest cell
#pragma unroll 1
        for (int i = 1; i < L1; i++) {
            const bool v = z.vert(i);
            const long long cur = v ? i * nn + (long long)tox * n + toy : i * nn + (long long)toy * n + tox;
            const int lo = v ? y0 : x0, hi = v ? y1 : x1, skip = v ? toy : tox;
            const double wc = z.wire_sum(cur);
            int best = kZInf * 2, bq = -1;  // above every candidate (at most kZInf + kZInf / 2)
            for (int q = lo + lane; q <= hi; q += kWave) {
                if (q == skip) continue;
                const long long last = v ? i * nn + (long long)tox * n + q : i * nn + (long long)toy * n + q;
                const int cand = m4[last] + (int)fmin(fabs(z.wire_sum(last) - wc), double(kZInf / 2));
                if (cand < best) {
                    best = cand;
                    bq = q;
                }
            }
            for (int o = kWave / 2; o; o >>= 1) {
                const int ob = __shfl_xor(best, o, kWave), oq = __shfl_xor(bq, o, kWave);
                if (ob < best || (ob == best && oq >= 0 && (bq < 0 || oq < bq))) {
                    best = ob;
                    bq = oq;
                }
            }
            if (lane == 0 && bq >= 0 && best < map[cur + j * P]) {
                const long long last = v ? i * nn + (long long)tox * n + bq : i * nn + (long long)toy * n + bq;
                map[cur + j * P] = best;
                prev[cur + j * P] = p4[last];
                prev2[cur + j * P] = prev[5 * P + last];
            }
        }
    } else if (fromx == tox) {
        for (int i = 1 + lane; i < L1; i += kWave) {
            if (z.vert(i)) {
                const long long last = i * nn + (long long)fromx * n + fromy, cur = i * nn + (long long)tox * n + toy;
                const int cost = z.wire(last, cur);
                if (map[cur + j * P] > map[last] + cost) {
                    map[cur + j * P] = map[last] + cost;
                    prev[cur + j * P] = (int)last;
                }
            } else {
                map[i * nn + (long long)toy * n + tox + j * P] = kZInf;
            }
        }
    } else {
        for (int i = 1 + lane; i < L1; i += kWave) {
            if (!z.vert(i)) {
                const long long last = i * nn + (long long)fromy * n + fromx, cur = i * nn + (long long)toy * n + tox;
                const int cost = z.wire(last, cur);
                if (map[cur + j * P] > map[last] + cost) {
                    map[cur + j * P] = map[last] + cost;
                    prev[cur + j * P] = (int)last;
                }
            } else {
                map[i * nn + (long long)tox * n + toy + j * P] = kZInf;
            }
        }
    }
    __syncthreads();
}

// The node's interval combination (zshape.cuh, lane 0 as in the
// reference): for every layer interval [lower, upper] the cheapest entry of
// each child slot inside it plus the vias of the interval, kept where it
// lowers the node's plane-0 value.  The node's cells are loaded once and
// combined in registers in the reference's order.
__device__ void znode(const Z& z, const int* rec) {
    const ZshapeArgs& a = z.a;
    const int tox = rec[0] / a.n, toy = rec[0] % a.n, minlayer = rec[1], maxlayer = rec[2];
    const int L1 = a.layers;
    const bool has[3] = {rec[3] != -1, rec[4] != -1, rec[5] != -1};
    long long idx[kMaxLayers];
    int slot[3][kMaxLayers], mv[kMaxLayers], pv[kMaxLayers], via[kMaxLayers];
#pragma unroll
    for (int i = 0; i < kMaxLayers; i++) {
        if (i >= L1) continue;
        idx[i] = z.cell(i, tox, toy);
#pragma unroll
        for (int j = 0; j < 3; j++) slot[j][i] = has[j] ? a.map[idx[i] + (j + 1) * z.P] : 0;
        mv[i] = a.map[idx[i]];
        pv[i] = a.prev[idx[i]];
        via[i] = z.via(idx[i]);
    }
#pragma unroll 1
    for (int lower = 0; lower < L1; lower++) {
        int via_sum = 0, min_cost = kZInf, bestpos[3] = {0, 0, 0};
        int costs[3] = {has[0] ? kZInf : 0, has[1] ? kZInf : 0, has[2] ? kZInf : 0};
#pragma unroll
        for (int upper = 0; upper < kMaxLayers; upper++) {
            if (upper < lower || upper >= L1) continue;
#pragma unroll
            for (int j = 0; j < 3; j++)
                if (has[j] && slot[j][upper] < costs[j]) {
                    costs[j] = slot[j][upper];
                    bestpos[j] = upper;
                }
            if (1LL * costs[0] + costs[1] + costs[2] < min_cost) min_cost = costs[0] + costs[1] + costs[2];
            if (minlayer == -1 || (lower <= minlayer && maxlayer <= upper)) {
                const int code = (((lower * L1 + upper) * L1 + bestpos[2]) * L1 + bestpos[1]) * L1 + bestpos[0];
#pragma unroll
                for (int i = 0; i < kMaxLayers; i++) {
                    if (i < lower || i > upper) continue;
                    if (mv[i] > min_cost + via_sum) {
                        mv[i] = min_cost + via_sum;
                        pv[i] = code;
                    }
                }
            }
            via_sum += via[upper];
        }
    }
#pragma unroll
    for (int i = 0; i < kMaxLayers; i++) {
        if (i >= L1) continue;
        a.map[idx[i]] = mv[i];
        a.prev[idx[i]] = pv[i];
    }
}

struct Emitter {
    int* routes;
    int cap;
    int* error;
    __device__ __forceinline__ void operator()(long long p, long long q) {
        if (routes[0] + 1 >= cap) {
            atomicExch(error, (int)kDevRouteOverflow);
            return;
        }
        routes[routes[0]++] = (int)p;
        routes[routes[0]++] = (int)q;
    }
};

__device__ __forceinline__ bool in_map(const Z& z, long long idx) { return idx >= 0 && idx < z.P; }

__device__ void ztrace(const Z& z, const int* pts, int node_cnt, int* routes, int cap) {
    const ZshapeArgs& a = z.a;
    const long long nn = z.nn, P = z.P;
    const int L1 = a.layers, n = a.n;
    int* map = a.map;
    const int* prev = a.prev;
    const int* prev2 = a.prev + 10 * P;
    Emitter emit{routes, cap, a.error};
    int min_total = kZInf;
    for (int i = 0; i < L1; i++) {
        const long long idx = z.cell(i, pts[0] / n, pts[0] % n);
        if (map[idx] < min_total) {
            min_total = map[idx];
            map[5 * P + pts[0]] = i;
        }
    }
    if (min_total == kZInf || min_total < 0) {
        routes[0] = -1;
        return;
    }
    for (int t = 0; t < 6 * node_cnt; t += 6) {
        const int x = pts[t] / n, y = pts[t] % n, layer = map[5 * P + pts[t]];
        if (layer < 0 || layer >= L1) {
            atomicExch(a.error, (int)kDevNoSolution);
            return;
        }
        const long long idx = z.cell(layer, x, y);
        const int code = prev[idx];
        const int minl = code / L1 / L1 / L1 / L1, maxl = code / L1 / L1 / L1 % L1;
        for (int i = minl; i < maxl && i < L1; i++) emit(z.cell(i, x, y), -1);
        int bestpos = code;
        for (int j = 0; j < 3; j++) {
            if (pts[t + 3 + j] == -1) break;
            const int child = pts[pts[t + 3 + j]];
            const int entry_layer = bestpos % L1;
            const long long entry = z.cell(entry_layer, x, y);
            bestpos /= L1;
            const long long last = prev[(j + 1) * P + entry];
            if (!in_map(z, last)) {
                atomicExch(a.error, (int)kDevNoSolution);
                return;
            }
            const int last_layer = int(last / nn);
            int lastx = int(last / n % n), lasty = int(last % n);
            if (!z.vert(last_layer)) {
                const int s = lastx;
                lastx = lasty;
                lasty = s;
            }
            if (lastx != x && lasty != y) {
                const long long mid = prev2[(j + 1) * P + entry];
                if (!in_map(z, mid)) {
                    atomicExch(a.error, (int)kDevNoSolution);
                    return;
                }
                const int mid_layer = int(mid / nn);
                int midx = int(mid / n % n), midy = int(mid % n);
                if (!z.vert(mid_layer)) {
                    const int s = midx;
                    midx = midy;
                    midy = s;
                }
                const long long p1 = z.vert(entry_layer) ? entry - y + midy : entry - x + midx;
                const long long p3 = z.vert(mid_layer) ? mid - midy + lasty : mid - midx + lastx;
                const long long p4 = z.vert(last_layer) ? last - lasty + midy : last - lastx + midx;
                if (entry != p1) emit(min(entry, p1), entry < p1 ? p1 - entry : entry - p1);
                if (p1 != mid)
                    for (int i = min(entry_layer, mid_layer); i < max(entry_layer, mid_layer); i++)
                        emit(z.cell(i, midx, midy), -1);
                if (mid != p3) emit(min(mid, p3), mid < p3 ? p3 - mid : mid - p3);
                if (p3 != p4) {
                    int tx = int(p3 / n % n), ty = int(p3 % n);
                    if (!z.vert(int(p3 / nn))) {
                        const int s = tx;
                        tx = ty;
                        ty = s;
                    }
                    for (int i = min(mid_layer, last_layer); i < max(mid_layer, last_layer); i++)
                        emit(z.cell(i, tx, ty), -1);
                }
                if (p4 != last) emit(min(p4, last), p4 < last ? last - p4 : p4 - last);
            } else {
                emit(min(entry, last), entry < last ? last - entry : entry - last);
            }
            map[5 * P + child] = last_layer;
        }
    }
}

}  // namespace

__global__ __launch_bounds__(kWave) void zshape_solve_kernel(ZshapeArgs a) {
    if (int(blockIdx.x) >= a.count) return;
    const int k = a.list[blockIdx.x];
    const int lane = threadIdx.x;
    const Z z(a);
    const int* pts = a.points + a.points[k];
    int* routes = a.raw + pts[0];
    const int cap = a.raw_cap[k];
    if (lane == 0) routes[0] = 1;
    __syncthreads();
    const int node_cnt = pts[1];
    pts += 2;
    for (int t = 6 * (node_cnt - 1); t >= 0; t -= 6) {
        const int tox = pts[t] / a.n, toy = pts[t] % a.n;
        for (int j = 1; j <= 3; j++) {
            if (pts[t + 2 + j] == -1) continue;
            const int child = pts[pts[t + 2 + j]];
            zedge(z, lane, j, child / a.n, child % a.n, tox, toy);
        }
        if (lane == 0) znode(z, pts + t);
        __syncthreads();
    }
    if (lane == 0) ztrace(z, pts, node_cnt, routes, cap);
}

__global__ __launch_bounds__(256) void zshape_reset_kernel(ZshapeArgs a) {
    if (int(blockIdx.x) >= a.count) return;
    const int k = a.list[blockIdx.x];
    const Z z(a);
    const int* rec = a.points + a.points[k];
    const int nodes = rec[1];
    rec += 2;
    for (int i = threadIdx.x; i < nodes * a.layers; i += blockDim.x) {
        const int layer = i % a.layers, point = rec[(i / a.layers) * 6];
        const long long index = z.cell(layer, point / a.n, point % a.n);
        for (int plane = 0; plane < 4; ++plane) a.map[plane * z.P + index] = kZInf;
    }
}

// Raw words [map start, length or -1 for a via] into route words
// (src/routing/zshape_topology.hpp:233-289).
__global__ __launch_bounds__(256) void zshape_convert_kernel(ZshapeArgs a, const int* net_ids, RouteStore rs) {
    const int at = blockIdx.x * blockDim.x + threadIdx.x;
    if (at >= a.count) return;
    const int k = a.list[at];
    const DeviceGrid& g = a.g;
    const int n = a.n, X = g.X, Y = g.Y, L = g.L, XY = g.XY;
    const int id = net_ids[k];
    const int* src = a.raw + a.points[a.points[k]];
    int* dst = rs.routes + (size_t)rs.pin_acc_num[id] * rs.per_pin;
    const int cap = rs.per_pin * (rs.pin_acc_num[id + 1] - rs.pin_acc_num[id]);
    int out = 1;
    for (int p = 1; p + 1 < src[0]; p += 2) {
        const int start = src[p], len = src[p + 1];
        const int layer = start / (n * n) - 1;
        const int u = start / n % n, v = start % n;
        const bool vert = layer >= 0 && layer_dir(g, layer);
        const int x = vert ? u : v, y = vert ? v : u;
        if (layer < 0 || layer >= L || x >= X || y >= Y) {
            atomicExch(a.error, (int)kDevBadCoordinate);
            continue;
        }
        const int pos0 = (layer * X + x) * Y + y;
        int pos1 = pos0;
        if (len == -1) {
            if (layer + 1 >= L) {
                atomicExch(a.error, (int)kDevBadCoordinate);
                continue;
            }
            pos1 += XY;
        } else {
            const int end = start + len, eu = end / n % n, ev = end % n;
            const int ex = vert ? eu : ev, ey = vert ? ev : eu;
            if (ex >= X || ey >= Y) {
                atomicExch(a.error, (int)kDevBadCoordinate);
                continue;
            }
            pos1 = (layer * X + ex) * Y + ey;
        }
        if (out + 1 < cap) {
            dst[out++] = pos0;
            dst[out++] = pos1;
        } else {
            atomicExch(a.error, (int)kDevRouteOverflow);
        }
    }
    if (src[0] <= 0) atomicExch(a.error, (int)kDevNoSolution);
    dst[0] = out;
}

// ---- nets whose tree fits in LDS ----
//
// One workgroup routes one net with its whole DP in LDS.  Every value the
// reference keeps on the shared map is a pure function of the child's values
// and the costs, so nothing but prefix sums, via costs and the route words
// touches memory:
//  - a node's plane-0 cell of layer i is one 64-bit key, cost << 32 | code
//    (interval and best layer per child slot).  The code grows with (lower,
//    upper), so the least key is the reference's first strict minimum;
//  - a child slot's cell of layer e is one key, cost << 32 | bend << 8 |
//    leaving layer << 4 | middle layer: the least key is the reference's first
//    minimum over the last leg's cells in ascending order, and the traceback
//    needs no more of its two map indices than those three values.
// An edge's routes bend on one row or one column of its box each, and routes
// of different bends meet only in that minimum: one lane carries one bend's
// L values through first leg, via sweep, middle leg, via sweep and last leg
// in registers.  The nodes of one height are independent; their intervals
// (lane = node and lower layer), then their edges to the parents (lane =
// edge and bend, flattened over the level's edges) run over the whole
// workgroup with one barrier after each.  The corner of the box that is
// reached straight from the child (bend == the child's own row or column)
// skips the first via sweep; its second sweep changes nothing in the
// reference (the values are already closed under via steps), hence its
// middle layer is the arriving one.
//
// Bound by latency: a batch holds at most a few hundred nets, one workgroup
// each, and a net's levels follow one another.  Four wavefronts per net
// (a level of a 10 x 10 box holds 20 items per edge) and every load of an item
// in flight at once.  Against one wavefront per net with the shared map in
// global memory (the general kernels above), 128x128x5 with 20k nets:
// the DP takes 23 us per batch instead of 232 (136 batches of at most 250
// nets, batch loop 33.5 -> 5.3 ms).
namespace {

constexpr unsigned long long kZNone = (unsigned long long)kZInf << 32;

struct ZnetTables {
    unsigned long long *val, *slot;
    int4* node;
    int *via, *ipre, *ls, *pre, *lay, *woff, *wst, *wedge;
};

__host__ __device__ inline size_t znet_bytes(int L, int n) {
    const size_t L1 = size_t(L) + 1, N = size_t(n);
    return (N * (32 * L1 + 16 + 4 * L1 + 4 * 7) + 4 * 4 + 15) & ~size_t(15);
}

__device__ __forceinline__ ZnetTables znet_carve(char* base, int L, int n) {
    const size_t L1 = size_t(L) + 1, N = size_t(n);
    ZnetTables t;
    t.node = reinterpret_cast<int4*>(base);
    t.val = reinterpret_cast<unsigned long long*>(t.node + N);
    t.slot = t.val + N * L1;
    t.via = reinterpret_cast<int*>(t.slot + N * 3 * L1);
    t.ipre = t.via + N * L1;
    t.ls = t.ipre + N + 1;
    t.pre = t.ls + N + 2;
    t.lay = t.pre + N;
    t.woff = t.lay + N;
    t.wst = t.woff + N + 1;
    t.wedge = t.wst + N;
    return t;
}

__device__ __forceinline__ int zvia_of(float v) { return (int)fminf(fmaxf(v, 1.f), 1.e6f); }
__device__ __forceinline__ int zwire_of(double p, double q) { return (int)fmin(fabs(p - q), double(kZInf / 2)); }

// The reference's via sweep (upwards, then downwards) over one cell's
// layers; src follows the value, mid becomes the layer a value came from.
template <int L>
__device__ __forceinline__ void zsweep(int (&m)[L], int (&src)[L], int (&mid)[L], const int (&vc)[L]) {
#pragma unroll
    for (int l = 1; l < L; ++l) {
        const int v = m[l - 1] + vc[l - 1];
        const bool up = m[l] > v;
        m[l] = up ? v : m[l];
        src[l] = up ? src[l - 1] : src[l];
        mid[l] = up ? l - 1 : mid[l];
    }
#pragma unroll
    for (int l = L - 2; l >= 0; --l) {
        const int v = m[l + 1] + vc[l];
        const bool down = m[l] > v;
        m[l] = down ? v : m[l];
        src[l] = down ? src[l + 1] : src[l];
        mid[l] = down ? l + 1 : mid[l];
    }
}

// One bend of the edge from node c at (fx, fy) to its parent's slot at (tx,
// ty): row != 0 bends on row q (first leg vertical), else on column q.
template <int L>
__device__ __forceinline__ void zbend(const ZnetArgs& a, const unsigned long long* cval, unsigned long long* slot, int fx,
                                      int fy, int tx, int ty, int row, int q) {
    const DeviceGrid& g = a.g;
    const int d1 = row ? 1 : 0;  // direction of the first and last legs
    const bool corner = q == (row ? fy : fx);
    const int ax = row ? fx : q, ay = row ? q : fy, bx = row ? tx : q, by = row ? q : ty;
    double pa[L], pb[L], pc[L], pt[L];
    float va[L], vb[L];
#pragma unroll
    for (int l = 0; l < L; ++l) {
        const bool first = layer_dir(g, l) == d1;
        const int ca = cell_of(g, l, ax, ay), cb = cell_of(g, l, bx, by);
        pa[l] = a.presum[ca];
        pb[l] = a.presum[cb];
        pc[l] = a.presum[first ? cell_of(g, l, fx, fy) : ca];
        pt[l] = a.presum[first ? cell_of(g, l, tx, ty) : cb];
        va[l] = a.vcost[ca];
        vb[l] = a.vcost[cb];
    }
    int m[L], src[L], mid[L], vc[L], cv[L];
#pragma unroll
    for (int l = 0; l < L; ++l) {
        cv[l] = int(cval[l + 1] >> 32);
        m[l] = layer_dir(g, l) == d1 ? cv[l] + zwire_of(pc[l], pa[l]) : kZInf;
        src[l] = l;
        mid[l] = l;
        vc[l] = zvia_of(va[l]);
    }
    zsweep<L>(m, src, mid, vc);
#pragma unroll
    for (int l = 0; l < L; ++l) {
        const bool middle = layer_dir(g, l) != d1;
        m[l] = middle ? (corner ? cv[l] : m[l]) + zwire_of(pa[l], pb[l]) : kZInf;
        src[l] = corner ? l : src[l];
        mid[l] = l;
        vc[l] = zvia_of(vb[l]);
    }
    zsweep<L>(m, src, mid, vc);
#pragma unroll
    for (int l = 0; l < L; ++l) {
        if (layer_dir(g, l) != d1) continue;
        const int cost = m[l] + zwire_of(pb[l], pt[l]);
        const int via = corner ? l : mid[l];
        if (cost < kZInf)
            atomicMin(slot + l + 1, (unsigned long long)cost << 32 | unsigned(q << 8 | (src[l] + 1) << 4 | (via + 1)));
    }
}

// A straight edge: one wire on each layer along it.
template <int L>
__device__ __forceinline__ void zstraight(const ZnetArgs& a, const unsigned long long* cval, unsigned long long* slot,
                                          int fx, int fy, int tx, int ty) {
    const DeviceGrid& g = a.g;
    const int d = fx == tx ? 1 : 0;
    double pc[L], pt[L];
#pragma unroll
    for (int l = 0; l < L; ++l) {
        pc[l] = a.presum[cell_of(g, l, fx, fy)];
        pt[l] = a.presum[cell_of(g, l, tx, ty)];
    }
#pragma unroll
    for (int l = 0; l < L; ++l) {
        if (layer_dir(g, l) != d) continue;
        const int cost = int(cval[l + 1] >> 32) + zwire_of(pc[l], pt[l]);
        if (cost < kZInf) slot[l + 1] = (unsigned long long)cost << 32 | unsigned((l + 1) << 4 | (l + 1));
    }
}

// The intervals [lower, upper] of one node for one lower layer (0..L, layer
// 0 below the first routing layer): the cheapest entry of every child slot
// inside the interval plus its vias, offered to every layer it covers.
template <int L>
__device__ __forceinline__ void zintervals(const ZnetTables& s, int i, int lower) {
    constexpr int L1 = L + 1;
    const int4 nd = s.node[i];
    const int minl = (nd.y & 0xFF) - 1, maxl = (nd.y >> 8 & 0xFF) - 1, nchild = nd.y >> 16;
    unsigned long long key[L1];
    int via_sum = 0, min_cost = kZInf, pos[3] = {0, 0, 0};
    int costs[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) costs[j] = j < nchild ? kZInf : 0;
#pragma unroll
    for (int upper = 0; upper < L1; ++upper) {
        key[upper] = kZNone;
        if (upper < lower) continue;
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const int v = int(s.slot[(size_t(i) * 3 + j) * L1 + upper] >> 32);
            if (j < nchild && v < costs[j]) {
                costs[j] = v;
                pos[j] = upper;
            }
        }
        const long long sum = 1LL * costs[0] + costs[1] + costs[2];
        if (sum < min_cost) min_cost = int(sum);
        const int cost = min_cost + via_sum;
        if (cost < kZInf && (minl == -1 || (lower <= minl && maxl <= upper)))
            key[upper] = (unsigned long long)cost << 32 |
                         unsigned((((lower * L1 + upper) * L1 + pos[2]) * L1 + pos[1]) * L1 + pos[0]);
        via_sum += s.via[i * L1 + upper];
    }
    unsigned long long best = kZNone;
#pragma unroll
    for (int l = L; l >= 0; --l) {
        if (l < lower) continue;
        best = key[l] < best ? key[l] : best;
        if (best < kZNone) atomicMin(s.val + i * L1 + l, best);
    }
}

// The words of the edge from node c to its parent, in the reference's order
// (zshape.cuh:288-345): emit(layer, x, y, layer2, x2, y2) per pair.
template <int L, class Emit>
__device__ __forceinline__ void zedge_words(const ZnetTables& s, int c, int dirv, Emit&& emit) {
    constexpr int L1 = L + 1;
    const int4 cn = s.node[c];
    const int p = cn.z & 0xFFFF, j = cn.z >> 16;
    const int pxy = s.node[p].x;
    const int fx = cn.x & 0xFFFF, fy = cn.x >> 16, x = pxy & 0xFFFF, y = pxy >> 16;
    int code = int(unsigned(s.val[p * L1 + s.lay[p]]));
    for (int k = 0; k < j; ++k) code /= L1;
    const int entry = code % L1;
    const unsigned w = unsigned(s.slot[(size_t(p) * 3 + j) * L1 + entry]);
    const int last = w >> 4 & 15, mid = w & 15, q = int(w >> 8);
    auto wire = [&](int l, int x0, int y0, int x1, int y1) {
        emit(l, min(x0, x1), min(y0, y1), l, max(x0, x1), max(y0, y1));
    };
    if (fx == x || fy == y) {
        wire(entry, x, y, fx, fy);
        return;
    }
    auto vert = [&](int l) { return ((l & 1) ^ dirv) != 0; };
    const bool ve = vert(entry), vm = vert(mid), vl = vert(last);
    const int mx = ve ? x : q, my = ve ? q : y;
    if (mx != x || my != y) wire(entry, x, y, mx, my);
    for (int l = min(entry, mid); l < max(entry, mid); ++l) emit(l, mx, my, l + 1, mx, my);
    const int x3 = vm ? mx : fx, y3 = vm ? fy : my;  // the middle leg's end
    if (x3 != mx || y3 != my) wire(mid, mx, my, x3, y3);
    for (int l = min(mid, last); l < max(mid, last); ++l) emit(l, x3, y3, l + 1, x3, y3);
    const int x4 = vl ? fx : mx, y4 = vl ? my : fy;  // the last leg's start
    if (x4 != fx || y4 != fy) wire(last, x4, y4, fx, fy);
}

}  // namespace

namespace {

// The wires among a net's `pairs` route pairs committed by its workgroup (what
// commit_wires_kernel adds at K = 1): a batch's nets have their costs from the
// refresh before it, so their demand can go up while others are being solved.
// One lane per pair, long wires shared by the wavefront (commit_cells).
// It saves the commit's launch, 6 us of a batch whose DP takes 23 (136
// batches: loop 5.33 -> 4.84 ms).
__device__ __forceinline__ void commit_words(const ZnetArgs& a, const int* out, int pairs) {
    const DeviceGrid& g = a.g;
    const WireCommit& c = a.wires;
    long long length = 0;
    int edges = 0;
    const int lane = threadIdx.x % kWave;
    for (int t0 = threadIdx.x - lane; t0 < pairs; t0 += kZnetThreads) {
        const int t = t0 + lane;
        int c0 = 0, step = 0, len = 0;
        bool one_track = false;
        const int ra = t < pairs ? out[1 + 2 * t] : 0, rb = t < pairs ? out[2 + 2 * t] : 0;
        const int l = ra / g.XY;
        if (t < pairs && l == rb / g.XY) {
            const int x0 = ra / g.Y % g.X, y0 = ra % g.Y, x1 = rb / g.Y % g.X, y1 = rb % g.Y;
            const bool along_y = x0 == x1;
            const int lo = along_y ? min(y0, y1) : min(x0, x1), hi = along_y ? max(y0, y1) : max(x0, x1);
            c0 = along_y ? cell_of(g, l, x0, lo) : cell_of(g, l, lo, y0);
            one_track = along_y == (layer_dir(g, l) != 0);
            step = one_track ? 1 : (along_y ? g.X : g.Y);
            len = hi - lo;
            c.timestamp[cell_of(g, l, x0, y0)] = c.stamp;
            c.timestamp[cell_of(g, l, x1, y1)] = c.stamp;
            if (one_track && len) c.track_dirty[track_of_cell(g, c0)] = 1u;
            const long long* sum = along_y ? c.y_len_sum : c.x_len_sum;
            length += sum[hi] - sum[lo];
            edges += len;
        }
        commit_cells(g, c, c0, step, one_track, len, lane, kWave);
    }
    for (int o = kWave / 2; o; o >>= 1) {
        length += __shfl_xor(length, o, kWave);
        edges += __shfl_xor(edges, o, kWave);
    }
    Stats* st = c.stats + blockIdx.x % kStatStripes;
    if (lane == 0 && length) atomicAdd(&st->total_wirelength, double(length));
    if (lane == 0 && edges) atomicAdd(&st->wire_edges, (unsigned long long)edges);
}

}  // namespace

// Workgroup k routes net k of the list; see above.
template <int L>
__global__ __launch_bounds__(kZnetThreads) void zshape_net_kernel(ZnetArgs a) {
    constexpr int L1 = L + 1;
    extern __shared__ __align__(16) char smem[];
    __shared__ int s_root, s_short;
    const DeviceGrid& g = a.g;
    const int tid = threadIdx.x;
    const int4 d = a.desc[blockIdx.x];  // record, nodes, height, raw capacity
    const int n = d.y, H = d.z, dirv = g.DIR ^ 1;
    const ZnetTables s = znet_carve(smem, L, n);
    // record: nodes (4 words each, by height), item prefix, level starts, preorder
    const int* rec = a.recs + d.x;
    for (int i = tid; i < n; i += kZnetThreads) {
        const int4 nd = make_int4(rec[4 * i], rec[4 * i + 1], rec[4 * i + 2], rec[4 * i + 3]);
        s.node[i] = nd;
        s.pre[i] = rec[5 * n + 1 + H + 2 + i];
    }
    for (int i = tid; i <= n; i += kZnetThreads) s.ipre[i] = rec[4 * n + i];
    for (int i = tid; i < H + 2; i += kZnetThreads) s.ls[i] = rec[5 * n + 1 + i];
    for (int i = tid; i < 4 * n * L1; i += kZnetThreads) s.val[i] = kZNone;  // val and slot adjoin
    for (int q = tid; q < n * L1; q += kZnetThreads) {
        const int xy = rec[4 * (q / L1)], l = q % L1 - 1;
        s.via[q] = l < 0 ? kZInf : zvia_of(a.vcost[cell_of(g, l, xy & 0xFFFF, xy >> 16)]);
    }
    __syncthreads();
    for (int h = 0; h <= H; ++h) {
        const int b = s.ls[h], e = s.ls[h + 1];
        for (int q = tid; q < (e - b) * L1; q += kZnetThreads) zintervals<L>(s, b + q / L1, q % L1);
        __syncthreads();
        if (h == H) break;  // the root
        const int t0 = s.ipre[b], t1 = s.ipre[e];
        for (int t = t0 + tid; t < t1; t += kZnetThreads) {
            int lo = b, hi = e - 1;  // last node whose items start at or before t
            while (lo < hi) {
                const int m = (lo + hi + 1) >> 1;
                if (s.ipre[m] <= t) lo = m;
                else hi = m - 1;
            }
            const int4 nd = s.node[lo];
            const int p = nd.z & 0xFFFF, j = nd.z >> 16, pxy = s.node[p].x;
            const int fx = nd.x & 0xFFFF, fy = nd.x >> 16, tx = pxy & 0xFFFF, ty = pxy >> 16;
            const unsigned long long* cval = s.val + lo * L1;
            unsigned long long* slot = s.slot + (size_t(p) * 3 + j) * L1;
            if (fx == tx || fy == ty) {
                zstraight<L>(a, cval, slot, fx, fy, tx, ty);
            } else {
                // the |dy| rows of the box but the parent's, then its |dx| columns
                int k = t - s.ipre[lo];
                const int rows = abs(ty - fy), row = k < rows;
                if (!row) k -= rows;
                const int from = row ? fy : fx, to = row ? ty : tx;
                zbend<L>(a, cval, slot, fx, fy, tx, ty, row, to < from ? to + 1 + k : from + k);
            }
        }
        __syncthreads();
    }
    // traceback: the root's first cheapest layer, then level by level
    const int root = n - 1;
    if (tid == 0) {
        unsigned long long best = kZNone;
        int at = -1;
        for (int l = 0; l < L1; ++l)
            if (s.val[root * L1 + l] >> 32 < best >> 32) best = s.val[root * L1 + l], at = l;
        s.lay[root] = at;
        s_root = at;
    }
    __syncthreads();
    int* out = a.rs.routes + (size_t)a.rs.pin_acc_num[a.net_ids[blockIdx.x]] * a.rs.per_pin;
    if (s_root < 0) {
        if (tid == 0) {
            atomicExch(a.error, (int)kDevNoSolution);
            out[0] = 1;
        }
        return;
    }
    for (int h = H - 1; h >= 0; --h) {
        for (int c = s.ls[h] + tid; c < s.ls[h + 1]; c += kZnetThreads) {
            const int p = s.node[c].z & 0xFFFF, j = s.node[c].z >> 16;
            int code = int(unsigned(s.val[p * L1 + s.lay[p]]));
            for (int k = 0; k < j; ++k) code /= L1;
            s.lay[c] = int(unsigned(s.slot[(size_t(p) * 3 + j) * L1 + code % L1]) >> 4 & 15);
        }
        __syncthreads();
    }
    // pairs per node (its via stack) and per edge, then their places: the
    // reference emits a node's stack and its children's edges in preorder
    for (int i = tid; i < n; i += kZnetThreads) {
        const int code = int(unsigned(s.val[i * L1 + s.lay[i]]));
        s.wst[i] = code / (L1 * L1 * L1) % L1 - code / (L1 * L1 * L1 * L1);
        int w = 0;
        if (i != root) zedge_words<L>(s, i, dirv, [&](int, int, int, int, int, int) { ++w; });
        s.wedge[i] = w;
    }
    __syncthreads();
    if (tid < kWave) {
        int carry = 0;
        for (int b = 0; b < n; b += kWave) {
            const int i = b + tid < n ? s.pre[b + tid] : 0;
            int w = 0;
            if (b + tid < n) {
                const int ch = s.node[i].w;
                w = s.wst[i];
                for (int k = 0; k < 3; ++k) {
                    const int c = (ch >> (10 * k) & 1023) - 1;
                    if (c >= 0) w += s.wedge[c];
                }
            }
            int incl = w;
            for (int o = 1; o < kWave; o <<= 1) {
                const int v = __shfl_up(incl, o, kWave);
                if (tid >= o) incl += v;
            }
            if (b + tid < n) s.woff[i] = carry + incl - w;
            carry += __shfl(incl, kWave - 1, kWave);
        }
        if (tid == 0) {
            const int id = a.net_ids[blockIdx.x];
            const int cap = min(a.rs.per_pin * (a.rs.pin_acc_num[id + 1] - a.rs.pin_acc_num[id]), d.w);
            const int fit = max(0, (cap - 1) / 2);
            if (carry > fit) atomicExch(a.error, (int)kDevRouteOverflow);
            s_short = min(carry, fit);
            out[0] = 1 + 2 * s_short;
        }
    }
    __syncthreads();
    const int fit = s_short;
    for (int i = tid; i < n; i += kZnetThreads) {
        int at = s.woff[i];
        auto put = [&](int l, int x, int y, int l2, int x2, int y2) {
            if (at < fit) {
                out[1 + 2 * at] = ((l - 1) * g.X + x) * g.Y + y;
                out[2 + 2 * at] = ((l2 - 1) * g.X + x2) * g.Y + y2;
            }
            ++at;
        };
        const int4 nd = s.node[i];
        const int x = nd.x & 0xFFFF, y = nd.x >> 16;
        const int low = int(unsigned(s.val[i * L1 + s.lay[i]])) / (L1 * L1 * L1 * L1);
        for (int k = 0; k < s.wst[i]; ++k) put(low + k, x, y, low + k + 1, x, y);
        for (int k = 0; k < 3; ++k) {
            const int c = (nd.w >> (10 * k) & 1023) - 1;
            if (c >= 0) zedge_words<L>(s, c, dirv, put);
        }
    }
    if (a.wires.demand) {
        __syncthreads();  // the words above, read back from this workgroup's stores
        commit_words(a, out, fit);
    }
}

size_t znet_lds_bytes(int L, int n) { return znet_bytes(L, n); }

void launch_zshape_nets(const ZnetArgs& a, int count, int nmax, hipStream_t st) {
    switch (a.g.L) {
#define GR_Z_CASE(k)                                                                                              \
    case k:                                                                                                       \
        hipLaunchKernelGGL(zshape_net_kernel<k>, dim3(count), dim3(kZnetThreads), znet_bytes(k, nmax), st, a); \
        break;
        GR_Z_CASE(1) GR_Z_CASE(2) GR_Z_CASE(3) GR_Z_CASE(4) GR_Z_CASE(5) GR_Z_CASE(6) GR_Z_CASE(7) GR_Z_CASE(8)
        GR_Z_CASE(9) GR_Z_CASE(10) GR_Z_CASE(11) GR_Z_CASE(12) GR_Z_CASE(13) GR_Z_CASE(14) GR_Z_CASE(15)
#undef GR_Z_CASE
        default: break;
    }
}

}  // namespace grotor
