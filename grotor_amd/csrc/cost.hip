// Cost refresh for gfx950: wire/via costs and the Fenwick-ordered prefix.
//
// Reference: update_single_wcost_ispd24 / update_single_vcost_ispd24
// (src/cost/full_update.cuh:34-83), refresh_fenwick_tracks
// (src/cost/fenwick.cuh:129-168) driven by graph::refresh_cost
// (src/cost/incremental_update.cuh:98-132).
//
// All three outputs are pure functions of (capacity, demand) along one
// routing track: wcost and vcost read the cell and its predecessor on the
// track, presum reads the track's wcost.  The reference tracks dirtiness per
// cell plus per Fenwick node; here one flag per track suffices and a dirty
// track is recomputed whole, which yields the same values bit for bit.
//
// One workgroup per track.  With the track-major layout a track is one
// contiguous run, so thread t owns the k consecutive positions
// [t*k, t*k + k) and every global access is a unit-stride vector access.
// Fenwick nodes are built level by level in LDS in the reference's exact
// addition order; wcost itself never leaves the chip unless requested.
#include "gr_kernels.hpp"

namespace grotor {

__global__ __launch_bounds__(kRefreshThreads) void refresh_tracks_kernel(
    DeviceGrid g, const float* __restrict__ capacity, const float* __restrict__ demand,
    float* __restrict__ vcost, double* __restrict__ presum, float* __restrict__ wcost_out,
    unsigned* __restrict__ track_dirty, int force, CostParams cp, unsigned long long* __restrict__ refreshed) {
    const int T = blockIdx.x;
    if (!force && !track_dirty[T]) return;
    int l = 0;
#pragma unroll
    for (int i = 1; i < kMaxLayers; ++i)
        if (i < g.L && T >= g.track_begin[i]) l = i;
    const int dir = layer_dir(g, l);
    const int len = dir ? g.Y : g.X;
    const int base = l * g.XY + (T - g.track_begin[l]) * len;
    const int* elen = dir ? g.y_edge_len : g.x_edge_len;
    const double sc = g.short_cost[l];
    extern __shared__ double fv[];  // Fenwick values, index = BIT position

    // increments of each thread's last cell: the via cost of the next
    // thread's first cell needs them
    __shared__ double last_h[kRefreshThreads], last_1[kRefreshThreads];
    const int k = (len + blockDim.x - 1) / blockDim.x;
    const int p0 = threadIdx.x * k;
    const int p1 = min(len, p0 + k);
    double first_h = 0.0, first_1 = 0.0;  // increments of cell p0
    if (p0 < len) {
        double prev_h = 0.0, prev_1 = 0.0;
        for (int p = p0; p < p1; ++p) {
            const float c = capacity[base + p], d = demand[base + p];
            double e0, eh, e1;
            of_cost3(c, d, cp.slope, cp.zero_slope, e0, eh, e1);
            const double inc_h = incr_from(e0, eh, sc);
            const double inc_1 = incr_from(e0, e1, sc);
            // wcost: src/cost/full_update.cuh:44-46
            float w = (float)inc_1;
            if (p < len - 1) w = (float)((double)w + g.unit_wire * (double)elen[p]);
            if (cp.integer_wire) w = (float)(long long)fminf(fmaxf(w, 0.f), 1.e7f);
            if (wcost_out) wcost_out[base + p] = w;
            if (p < len - 1) fv[p + 1] = (double)w;
            if (p == p0) {
                first_h = inc_h;
                first_1 = inc_1;
            } else {
                // vcost: src/cost/full_update.cuh:67-82
                const double v = p == len - 1 ? prev_1 : inc_h + prev_h;
                float vf = (float)v;
                vf = (float)((double)vf + cp.via_weight * g.unit_via);
                vcost[base + p] = vf;
            }
            prev_h = inc_h;
            prev_1 = inc_1;
        }
        last_h[threadIdx.x] = prev_h;
        last_1[threadIdx.x] = prev_1;
    }
    if (threadIdx.x == 0) fv[0] = 0.0;
    __syncthreads();
    if (p0 < len) {
        double v;
        if (p0 == 0) v = first_1;
        else if (p0 == len - 1) v = last_1[threadIdx.x - 1];
        else v = first_h + last_h[threadIdx.x - 1];
        float vf = (float)v;
        vf = (float)((double)vf + cp.via_weight * g.unit_via);
        vcost[base + p0] = vf;
    }
    // Fenwick nodes: node(i) = leaf(i) + node(i-1) + node(i-2) + ... +
    // node(i - width/2) for i = (2s+1)*width - 1 (src/cost/fenwick.cuh:149-159)
    for (int width = 2; width <= len; width <<= 1) {
        for (int i = (2 * threadIdx.x + 1) * width - 1; i < len; i += 2 * blockDim.x * width) {
            double value = fv[i];
            for (int off = 1; off < width; off <<= 1) value += fv[i - off];
            fv[i] = value;
        }
        __syncthreads();
    }
    // exclusive prefix along the Fenwick path (src/cost/fenwick.cuh:160-166)
    for (int p = p0; p < p1; ++p) {
        double sum = 0.0;
        for (int j = p; j >= 0; j = (j & (j + 1)) - 1) sum += fv[j];
        presum[base + p] = sum;
    }
    if (threadIdx.x == 0) {
        track_dirty[T] = 0;
        // refreshed cells, striped like the stage statistics
        if (refreshed) atomicAdd(refreshed + (T % kStatStripes) * kCounterStride, (unsigned long long)len);
    }
}

// Grid arrays between the ABI's IDX order (l * X + x) * Y + y and the
// track-major order: layers running along y agree in both, the others are
// transposed in 32 x 32 tiles through LDS so that reads and writes are
// unit-stride.  Bound by the link the array crosses before or after; on the
// host, one cell at a time with a stride of a track, the same took 2.3 of the
// 2.9 ms of a cost download (1M cells: 4 + 4 + 8 bytes a cell).
constexpr int kLayoutTile = 32;
template <class T>
__global__ __launch_bounds__(256) void layout_kernel(DeviceGrid g, LayoutArrays<T> arrays, int to_track) {
    __shared__ T tile[kLayoutTile][kLayoutTile + 1];
    const unsigned layers = unsigned(arrays.layers);
    const T* __restrict__ src = blockIdx.z < layers ? arrays.src[0] : arrays.src[1];
    T* __restrict__ dst = blockIdx.z < layers ? arrays.dst[0] : arrays.dst[1];
    const int l = blockIdx.z % layers, tx = threadIdx.x % kLayoutTile, ty = threadIdx.x / kLayoutTile;
    const size_t base = size_t(l) * g.XY;
    // rows of the source: x (IDX) or the track y of a horizontal layer
    const bool copy = layer_dir(g, arrays.first + l), by_x = to_track || copy;
    const int rows = by_x ? g.X : g.Y, cols = by_x ? g.Y : g.X;
    // tiles along the source's rows first
    const int ctiles = (cols + kLayoutTile - 1) / kLayoutTile;
    const int r0 = int(blockIdx.x) / ctiles * kLayoutTile, c0 = int(blockIdx.x) % ctiles * kLayoutTile;
    for (int r = ty; r < kLayoutTile; r += 256 / kLayoutTile)
        if (r0 + r < rows && c0 + tx < cols) {
            const T v = src[base + size_t(r0 + r) * cols + c0 + tx];
            if (copy) dst[base + size_t(r0 + r) * cols + c0 + tx] = v;
            else tile[r][tx] = v;
        }
    if (copy) return;  // uniform over the workgroup
    __syncthreads();
    for (int c = ty; c < kLayoutTile; c += 256 / kLayoutTile)
        if (c0 + c < cols && r0 + tx < rows) dst[base + size_t(c0 + c) * rows + r0 + tx] = tile[tx][c];
}

template <class T>
void launch_layout(const DeviceGrid& g, const LayoutArrays<T>& a, bool to_track, hipStream_t st) {
    if (!a.count) return;
    const int xtiles = (g.X + kLayoutTile - 1) / kLayoutTile, ytiles = (g.Y + kLayoutTile - 1) / kLayoutTile;
    const dim3 grid(unsigned(xtiles * ytiles), 1, unsigned(a.layers * a.count));
    hipLaunchKernelGGL(layout_kernel<T>, grid, dim3(256), 0, st, g, a, to_track ? 1 : 0);
}
template void launch_layout<float>(const DeviceGrid&, const LayoutArrays<float>&, bool, hipStream_t);
template void launch_layout<int>(const DeviceGrid&, const LayoutArrays<int>&, bool, hipStream_t);
template void launch_layout<double>(const DeviceGrid&, const LayoutArrays<double>&, bool, hipStream_t);

}  // namespace grotor
