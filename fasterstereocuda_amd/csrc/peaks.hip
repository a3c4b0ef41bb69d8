// Peak removal on the GPU: small connected segments of a disparity map are
// set invalid.
//
// The reference (SgmStereoCuda/StereoCudaImpl.cpp:32-97, 463-498) runs, on
// the host after the map has been copied back, a breadth-first search per
// horizontal strip: strip i of `strips` covers rows [i r, (i + 1) r) with
// r = H / strips (rows from strips * r on are left as they are); within a
// strip, valid 4-neighbours join one segment when |d - d'| <= 1 (float
// arithmetic), and a segment of fewer than (int)((float)(W r) * ratio)
// pixels becomes invalid.  The reference takes `strips` from the host's core
// count (hardware_concurrency() * 3 / 4), which makes its result depend on
// the machine; here it is a parameter (default 1, the whole image).
//
// The segments are the connected components of the symmetric relation
// above, so any method that finds components gives the same answer.  This
// one labels 64 x 16 tiles in LDS first and then joins the tiles' components
// through device memory, with a lock-free union-find in both places: parents
// only ever decrease (parent[x] <= x), every union retry strictly lowers one
// of its two indices and every find strictly lowers its index, so all loops
// end.  A map is mostly a few large segments, so one union per pixel edge and
// one count per pixel all land on the same few roots (640x359 pixels: 390 us
// of unions and 1070 us of counts, against 5-20 us a pass of the map); with
// tiles, device memory sees one union per run of crossing edges (of edges, a
// 13th part of the pixels) and one count per tile and component.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <mutex>

#include "sgm_internal.h"

namespace fsgm {
namespace {

// relaxed read of a parent link another lane may be lowering
__device__ __forceinline__ int parent_of(const int* p, int x) {
    return __hip_atomic_load(p + x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ int find_root(const int* p, int x) {
    int q = parent_of(p, x);
    while (q != x) {
        x = q;
        q = parent_of(p, x);
    }
    return x;
}

// links the roots of a and b (in device memory or in LDS)
__device__ __forceinline__ void unite(int* p, int a, int b) {
    while (true) {
        a = find_root(p, a);
        b = find_root(p, b);
        if (a == b) return;
        if (a > b) { const int t = a; a = b; b = t; }
        const int old = atomicMin(p + b, a);   // link root b under a
        if (old == b) return;                  // b was still a root
        b = old;                               // b moved meanwhile: retry from its new parent
    }
}

__device__ __forceinline__ bool joins(float a, float b) {
    return a != kInvalidDisp && b != kInvalidDisp && fabsf(a - b) <= 1.0f;
}

// One workgroup labels a tile: a wave takes 4 of its rows, a lane one column.
// A row's runs of joined pixels come from one ballot, so labels start as run
// starts and only vertical edges are united, once per stretch of columns
// joined on both rows.  Writes parent (the tile root's pixel; tile order and
// pixel order agree, so parent[x] <= x) and size (the component's pixels in
// the tile at its root, 0 elsewhere) of every pixel of the tile.
constexpr int kTileW = 64, kTileH = 16;
__global__ __launch_bounds__(256) void peaks_tile_kernel(const float* __restrict__ disp,
                                                         int* __restrict__ parent,
                                                         int* __restrict__ size, int W, int rows,
                                                         int strip_rows) {
    __shared__ float sd[kTileH][kTileW];
    __shared__ int label[kTileH * kTileW], cnt[kTileH * kTileW];
    __shared__ uint64_t srun[kTileH];   // bit x: pixel x joins pixel x - 1
    const int tiles_x = (W + kTileW - 1) / kTileW;
    const int x0 = (int)(blockIdx.x % tiles_x) * kTileW, y0 = (int)(blockIdx.x / tiles_x) * kTileH;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int x = x0 + lane;
    float v[4];
    uint64_t run[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int r = wave + 4 * k, y = y0 + r;
        v[k] = (x < W && y < rows) ? disp[(int64_t)y * W + x] : kInvalidDisp;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int r = wave + 4 * k;
        const float left = __shfl_up(v[k], 1);
        run[k] = __ballot(lane > 0 && joins(left, v[k]));
        // the run's start: the last lane up to this one that joins no left pixel
        const uint64_t starts = ~run[k] & ((2ull << lane) - 1ull);
        label[r * kTileW + lane] = r * kTileW + 63 - __clzll((long long)starts);
        cnt[r * kTileW + lane] = 0;
        sd[r][lane] = v[k];
        if (lane == 0) srun[r] = run[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int r = wave + 4 * k;
        if (r == 0 || (y0 + r) % strip_rows == 0) continue;   // no edge up (wave-uniform)
        const bool up = joins(sd[r - 1][lane], v[k]);
        const uint64_t ups = __ballot(up);
        const uint64_t same = run[k] & srun[r - 1] & (ups << 1);   // the left edge joins these two
        if (up && !((same >> lane) & 1ull)) unite(label, (r - 1) * kTileW + lane, r * kTileW + lane);
    }
    __syncthreads();
    int root[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        root[k] = find_root(label, (wave + 4 * k) * kTileW + lane);
        if (v[k] != kInvalidDisp && !((run[k] >> lane) & 1ull)) {   // one count per run
            const uint64_t after = lane < 63 ? ~run[k] >> (lane + 1) : 0ull;
            const int len = after ? __ffsll((unsigned long long)after) : kTileW - lane;
            atomicAdd(cnt + root[k], len);
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int r = wave + 4 * k, y = y0 + r;
        if (x >= W || y >= rows) continue;
        const int64_t i = (int64_t)y * W + x;
        parent[i] = (y0 + root[k] / kTileW) * W + x0 + root[k] % kTileW;
        size[i] = cnt[r * kTileW + lane];
    }
}

// unions over the edges that cross tiles: first the `rows` edges of every
// tile column boundary, then the W edges of every tile row boundary.  An edge
// is skipped where the one before it on the same boundary joins the same two
// components (both its ends join this edge's ends inside their tiles).
__global__ __launch_bounds__(256) void peaks_border_kernel(const float* __restrict__ disp,
                                                           int* __restrict__ parent, int W,
                                                           int rows, int strip_rows, int64_t n_col,
                                                           int64_t n) {
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (int64_t)gridDim.x * 256) {
        if (e < n_col) {
            const int x = (int)(e / rows + 1) * kTileW, y = (int)(e % rows);
            const int i = y * W + x;
            const float a = disp[i - 1], b = disp[i];
            if (!joins(a, b)) continue;
            if (y % kTileH != 0 && y % strip_rows != 0) {
                const float pa = disp[i - W - 1], pb = disp[i - W];
                if (joins(pa, pb) && joins(pa, a) && joins(pb, b)) continue;
            }
            unite(parent, i - 1, i);
        } else {
            const int64_t f = e - n_col;
            const int y = (int)(f / W + 1) * kTileH, x = (int)(f % W);
            if (y % strip_rows == 0) continue;
            const int i = y * W + x;
            const float a = disp[i - W], b = disp[i];
            if (!joins(a, b)) continue;
            if (x % kTileW != 0) {
                const float pa = disp[i - W - 1], pb = disp[i - 1];
                if (joins(pa, pb) && joins(pa, a) && joins(pb, b)) continue;
            }
            unite(parent, i - W, i);
        }
    }
}

// segment sizes: every tile root that is not its segment's root adds its
// tile's count there and is linked to it directly
__global__ __launch_bounds__(256) void peaks_count_kernel(int* __restrict__ parent,
                                                          int* __restrict__ size, int n) {
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        const int c = size[i];
        if (c == 0) continue;
        const int r = find_root(parent, i);
        if (r == i) continue;
        atomicAdd(size + r, c);
        __hip_atomic_store(parent + i, r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// a pixel's parent is its tile root, whose parent is the segment's root
__global__ __launch_bounds__(256) void peaks_remove_kernel(float* __restrict__ disp,
                                                           const int* __restrict__ parent,
                                                           const int* __restrict__ size, int n,
                                                           int threshold) {
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        if (disp[i] == kInvalidDisp) continue;
        if (size[parent[parent[i]]] < threshold) disp[i] = kInvalidDisp;
    }
}

}  // namespace

int peaks_threshold(int W, int strip_rows, float ratio) {
    // StereoCudaImpl.cpp:476: int * int, times a float, truncated to int
    return (int)((float)(W * strip_rows) * ratio);
}

// Scratch of the allocation-free peak removal (sgm_stage_remove_peaks_noalloc):
// parent links and segment sizes of up to kPeaksNoAllocMaxPixels pixels,
// 2 * 4 B per pixel (16 MiB).  Each device holds its own copy for the life of
// the process.  Host code never uses this name as an address: it passes the
// per-device pointer from hipGetSymbolAddress.
static __device__ __align__(256) int scratch[2 * (size_t)kPeaksNoAllocMaxPixels];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
int* g_scratch_ptr[kMaxDevices] = {};
}  // namespace

hipError_t peaks_noalloc_scratch(int** out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        // once per device, with that device current: its copy's address
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        g_scratch_ptr[dev] = static_cast<int*>(p);
    }
    *out = g_scratch_ptr[dev];
    return hipSuccess;
}

hipError_t launch_remove_peaks(float* disp, int* work, int W, int H, int strips, float ratio,
                               hipStream_t s) {
    if (W <= 0 || H <= 0 || strips <= 0) return hipErrorInvalidValue;
    const int strip_rows = H / strips;
    const int rows = strip_rows * strips;   // rows past the last strip are left alone
    if (strip_rows == 0) return hipSuccess;
    const int threshold = peaks_threshold(W, strip_rows, ratio);
    const int n = W * rows;
    int* parent = work;
    int* size = work + (size_t)W * H;
    const unsigned blocks = (unsigned)std::min((n + 255) / 256, 65535);
    const int tiles_x = (W + kTileW - 1) / kTileW, tiles_y = (rows + kTileH - 1) / kTileH;
    const int64_t n_col = (int64_t)(tiles_x - 1) * rows, n_edges = n_col + (int64_t)(tiles_y - 1) * W;
    hipLaunchKernelGGL(peaks_tile_kernel, dim3((unsigned)(tiles_x * tiles_y)), dim3(256), 0, s, disp,
                       parent, size, W, rows, strip_rows);
    if (n_edges > 0)
        hipLaunchKernelGGL(peaks_border_kernel,
                           dim3((unsigned)std::min<int64_t>((n_edges + 255) / 256, 65535)), dim3(256),
                           0, s, disp, parent, W, rows, strip_rows, n_col, n_edges);
    hipLaunchKernelGGL(peaks_count_kernel, dim3(blocks), dim3(256), 0, s, parent, size, n);
    hipLaunchKernelGGL(peaks_remove_kernel, dim3(blocks), dim3(256), 0, s, disp, parent, size, n,
                       threshold);
    return hipGetLastError();
}

}  // namespace fsgm
