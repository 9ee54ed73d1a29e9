// lbvh.hip — the TLAS fast path (cudaBVH_buildTLASFast) on the GPU: the
// reference's LBVH (layer/cuda_bvh_backend.cu:257-389, :1620-1698) — 10-bit
// per axis Morton codes of the box centroids normalised by their bounds, a
// stable sort by code, a median split of the sorted order with one box per
// leaf, and the stackless DFS export of the nodes.
//
// The tree's shape depends only on n: the node of range [s, e) with
// pre-order index i has its left child at i + 1 ([s, m), m = s + (e-s)/2)
// and its right child at i + 2(m - s), and its subtree holds 2(e-s) - 1
// nodes. So every node finds its range by descending from the root (O(log n)
// steps) and writes its 32-byte DFS record (box, leaf code, skip = i + size,
// -1 past the end) in place. Box merges reproduce the host builder's fminf /
// fmaxf exactly (x86-64 libm: equal operands, e.g. -0 and +0, give the second
// operand; a NaN operand gives the other), so the output is byte-identical to
// a host build of the same algorithm.
//
// A small TLAS is all launch and round trip: 4,096 boxes took some 35 launches
// of 3-5 us, an allocation and a read back of the tree's depth, 320 us in all.
// So up to kSmallBoxes boxes are sorted by one launch in which every workgroup
// computes all keys for itself and the ranks of its 64 boxes by comparison,
// and one launch finds every node's box by a wave of its own straight from its
// range of sorted boxes (each box is then read once per level, from L2).
// That takes 109 us for 4,096 boxes. Both launches grow faster than n: for
// 8,192 boxes they still took half the time of the general path, but for
// 20,000 the wave per node 75 us more than a launch per level.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "rt_internal.h"
#include "trace_launch.h"

namespace rtl {

constexpr int kT = 256;
constexpr int kSmallBoxes = 8192;

__device__ __forceinline__ int f2o(float f) {
    const int i = __float_as_int(f);
    return i >= 0 ? i : i ^ 0x7fffffff;
}
__device__ __forceinline__ float o2f(int i) { return __int_as_float(i >= 0 ? i : i ^ 0x7fffffff); }

__device__ __forceinline__ float host_fminf(float x, float y) {
    if (y != y) return x;
    if (x != x) return y;
    return x < y ? x : y;
}
__device__ __forceinline__ float host_fmaxf(float x, float y) {
    if (y != y) return x;
    if (x != x) return y;
    return x > y ? x : y;
}

__device__ __forceinline__ uint32_t spread10(uint32_t v) {
    v &= 0x3ffu;
    v = (v | (v << 16)) & 0x030000ffu;
    v = (v | (v << 8)) & 0x0300f00fu;
    v = (v | (v << 4)) & 0x030c30c3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}
__device__ __forceinline__ uint32_t morton3d(float x, float y, float z) {
    x = fminf(fmaxf(x * 1024.0f, 0.0f), 1023.0f);
    y = fminf(fmaxf(y * 1024.0f, 0.0f), 1023.0f);
    z = fminf(fmaxf(z * 1024.0f, 0.0f), 1023.0f);
    return spread10((uint32_t)x) * 4u + spread10((uint32_t)y) * 2u + spread10((uint32_t)z);
}

// Centroids (mn + mx) * 0.5 and their bounds (ordered-int atomics; NaN
// centroids are left out, as the host's fminf / fmaxf ignore them). The sign
// of a zero bound does not matter: only c - min and max - min use it.
__global__ __launch_bounds__(kT) void k_centroids(const float* __restrict__ aabbs, int n, float* cen, int* bnd) {
    __shared__ int s[6];
    if (threadIdx.x < 6) s[threadIdx.x] = threadIdx.x < 3 ? 0x7fffffff : (int)0x80000000;
    __syncthreads();
    int lo[3] = {0x7fffffff, 0x7fffffff, 0x7fffffff}, hi[3] = {(int)0x80000000, (int)0x80000000, (int)0x80000000};
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        for (int a = 0; a < 3; a++) {
            const float c = (aabbs[6 * (size_t)i + a] + aabbs[6 * (size_t)i + 3 + a]) * 0.5f;
            cen[3 * (size_t)i + a] = c;
            if (c == c) { lo[a] = min(lo[a], f2o(c)); hi[a] = max(hi[a], f2o(c)); }
        }
    }
    for (int a = 0; a < 3; a++) { atomicMin(&s[a], lo[a]); atomicMax(&s[3 + a], hi[a]); }
    __syncthreads();
    if (threadIdx.x < 3) atomicMin(&bnd[threadIdx.x], s[threadIdx.x]);
    else if (threadIdx.x < 6) atomicMax(&bnd[threadIdx.x], s[threadIdx.x]);
}

__global__ void k_init_bounds(int* bnd) {
    if (threadIdx.x < 6) bnd[threadIdx.x] = threadIdx.x < 3 ? 0x7fffffff : (int)0x80000000;
}

// Morton key of a box from its centroid; lo / inv as the host computes them.
__device__ __forceinline__ uint32_t box_key(const float* cen, const int* bnd) {
    float q[3];
    for (int a = 0; a < 3; a++) {
        // with no finite centroid the host keeps its initial bounds (1e30, -1e30)
        const float lo = bnd[a] == 0x7fffffff ? 1e30f : o2f(bnd[a]);
        const float hi = bnd[3 + a] == (int)0x80000000 ? -1e30f : o2f(bnd[3 + a]);
        const float inv = (hi - lo > 1e-8f) ? 1.0f / (hi - lo) : 0.0f;
        q[a] = (cen[a] - lo) * inv;
    }
    return morton3d(q[0], q[1], q[2]);
}

// Key and index of every box.
__global__ __launch_bounds__(kT) void k_keys(const float* cen, int n, const int* bnd, uint32_t* keys, int* vals) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    keys[i] = box_key(cen + 3 * (size_t)i, bnd);
    vals[i] = i;
}

// Range [s, e) and tree level of pre-order node `id` of an n-leaf median tree.
__device__ __forceinline__ void node_range(int n, int id, int& s, int& e, int& level) {
    s = 0; e = n; level = 0;
    int cur = 0;
    while (cur != id) {
        const int m = s + (e - s) / 2;
        const int right = cur + 2 * (m - s);
        if (id < right) { cur = cur + 1; e = m; }
        else { cur = right; s = m; }
        level++;
    }
}

__global__ __launch_bounds__(kT) void k_levels(int n, int total, int* level) {
    const int id = blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= total) return;
    int s, e, l;
    node_range(n, id, s, e, l);
    level[id] = l;
}

// Sort of at most kSmallBoxes boxes by Morton code: box i goes to the position
// that is the number of boxes with a lower code, or an equal one and a lower
// index. One workgroup per 64 boxes, one box per lane; each wave compares them
// with every 16th tile of 64 codes. Also leaves the boxes themselves in sorted
// order, so that the nodes' waves wait for one load, not two, per box.
constexpr int kRankT = 1024;

__global__ __launch_bounds__(kRankT) void k_rank_sort(const float* __restrict__ aabbs, int n, int* ordered,
                                                       float2* __restrict__ sorted) {
    __shared__ int s_bnd[6];
    __shared__ __align__(16) uint32_t s_key[kSmallBoxes];
    __shared__ int s_rank[64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (tid < 6) s_bnd[tid] = tid < 3 ? 0x7fffffff : (int)0x80000000;
    if (tid < 64) s_rank[tid] = 0;
    __syncthreads();
    // centroids (kept in registers, all boxes in flight at once) and their
    // bounds, as k_centroids
    constexpr int kPer = kSmallBoxes / kRankT;
    float cen[kPer][3];
#pragma unroll
    for (int j = 0; j < kPer; j++) {
        const int i = tid + j * kRankT;
        if (i < n)
            for (int a = 0; a < 3; a++) cen[j][a] = (aabbs[6 * i + a] + aabbs[6 * i + 3 + a]) * 0.5f;
    }
    int lo[3] = {0x7fffffff, 0x7fffffff, 0x7fffffff}, hi[3] = {(int)0x80000000, (int)0x80000000, (int)0x80000000};
#pragma unroll
    for (int j = 0; j < kPer; j++)
        if (tid + j * kRankT < n)
            for (int a = 0; a < 3; a++) {
                const float c = cen[j][a];
                if (c == c) { lo[a] = min(lo[a], f2o(c)); hi[a] = max(hi[a], f2o(c)); }
            }
    for (int a = 0; a < 3; a++) {
        for (int o = 32; o > 0; o >>= 1) {
            lo[a] = min(lo[a], __shfl_xor(lo[a], o, 64));
            hi[a] = max(hi[a], __shfl_xor(hi[a], o, 64));
        }
        if (lane == 0) { atomicMin(&s_bnd[a], lo[a]); atomicMax(&s_bnd[3 + a], hi[a]); }
    }
    __syncthreads();
    const int tiles = (n + 63) >> 6;
#pragma unroll
    for (int j = 0; j < kPer; j++) {
        const int i = tid + j * kRankT;
        // (a code past the end comes after every other)
        if (i < tiles * 64) s_key[i] = i < n ? box_key(cen[j], s_bnd) : 0xffffffffu;
    }
    __syncthreads();
    const int own = blockIdx.x, i = own * 64 + lane;
    const uint32_t key = s_key[i];
    int rank = 0;
    for (int t = wave; t < tiles; t += kRankT / 64) {
        const uint4* k4 = reinterpret_cast<const uint4*>(s_key + 64 * t);
        if (t < own) {
            for (int j = 0; j < 16; j++) {
                const uint4 k = k4[j];
                rank += (k.x <= key) + (k.y <= key) + (k.z <= key) + (k.w <= key);
            }
        } else if (t > own) {
            for (int j = 0; j < 16; j++) {
                const uint4 k = k4[j];
                rank += (k.x < key) + (k.y < key) + (k.z < key) + (k.w < key);
            }
        } else {
            for (int j = 0; j < 64; j++) {
                const uint32_t k = s_key[64 * t + j];
                rank += k < key || (k == key && j < lane);
            }
        }
    }
    atomicAdd(&s_rank[lane], rank);
    __syncthreads();
    if (wave == 0 && i < n) {
        const int r = s_rank[lane];
        ordered[r] = i;
        const float2* b = reinterpret_cast<const float2*>(aabbs) + 3 * i;
        for (int k = 0; k < 3; k++) sorted[3 * r + k] = b[k];
    }
}

// Writes node id's DFS record: box, leaf code, skip.
__device__ __forceinline__ void put_node(uint32_t* out, int id, int s, int e, int total, const float* mn, const float* mx) {
    const int size = 2 * (e - s) - 1;
    uint32_t* o = out + 8 * (size_t)id;
    for (int a = 0; a < 3; a++) { o[a] = __float_as_uint(mn[a]); o[3 + a] = __float_as_uint(mx[a]); }
    o[6] = (uint32_t)(e - s <= 1 ? -((s << 3) | 0) - 2 : 0);      // leaf of one box (backend :393 encoding)
    o[7] = (uint32_t)(id + size < total ? id + size : -1);
}

// One wave per node: its box from its range of sorted boxes, in the range's
// order. Merging in any grouping gives the bits of the tree's own merges: of
// equal operands both keep the last, and no operand is NaN (a leaf has taken
// 1e30 / -1e30 in its place). Lanes hold consecutive pieces of the range; a
// lane without one holds the neutral 1e30 / -1e30.

__global__ __launch_bounds__(kT) void k_wave_boxes(const float2* __restrict__ sorted, int n, int total,
                                                   uint32_t* __restrict__ out) {
    const int id = __builtin_amdgcn_readfirstlane(blockIdx.x * (kT / 64) + (threadIdx.x >> 6)), lane = threadIdx.x & 63;
    if (id >= total) return;
    int s, e, l;
    node_range(n, id, s, e, l);
    const int per = (e - s + 63) >> 6;
    float mn[3] = {1e30f, 1e30f, 1e30f}, mx[3] = {-1e30f, -1e30f, -1e30f};
    const int hi = min(e, s + (lane + 1) * per);
#pragma unroll 8
    for (int k = s + lane * per; k < hi; k++) {
        const float2 p = sorted[3 * k], q = sorted[3 * k + 1], r = sorted[3 * k + 2];
        const float b[6] = {p.x, p.y, q.x, q.y, r.x, r.y};
        for (int a = 0; a < 3; a++) {
            mn[a] = host_fminf(mn[a], host_fminf(1e30f, b[a]));
            mx[a] = host_fmaxf(mx[a], host_fmaxf(-1e30f, b[3 + a]));
        }
    }
    for (int o = 1; o < 64; o <<= 1)
        for (int a = 0; a < 3; a++) {
            mn[a] = host_fminf(mn[a], __shfl_down(mn[a], o, 64));
            mx[a] = host_fmaxf(mx[a], __shfl_down(mx[a], o, 64));
        }
    if (lane == 0) put_node(out, id, s, e, total, mn, mx);
}

// Boxes of the nodes at tree level L (children done by the previous launch):
// a leaf takes its box, an inner node merges its children's as the host does
// (fminf(left, right), fmaxf(left, right)). Writes the node's DFS record.
__global__ __launch_bounds__(kT) void k_level_boxes(const float* __restrict__ aabbs, const int* ordered, int n,
                                                    int total, const int* level, int L, uint32_t* out) {
    const int id = blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= total || level[id] != L) return;
    int s, e, l;
    node_range(n, id, s, e, l);
    float mn[3], mx[3];
    if (e - s <= 1) {
        const float* b = aabbs + 6 * (size_t)ordered[s];
        for (int a = 0; a < 3; a++) { mn[a] = host_fminf(1e30f, b[a]); mx[a] = host_fmaxf(-1e30f, b[3 + a]); }
    } else {
        const int m = s + (e - s) / 2;
        const float* L_ = reinterpret_cast<const float*>(out + 8 * (size_t)(id + 1));
        const float* R_ = reinterpret_cast<const float*>(out + 8 * (size_t)(id + 2 * (m - s)));
        for (int a = 0; a < 3; a++) { mn[a] = host_fminf(L_[a], R_[a]); mx[a] = host_fmaxf(L_[3 + a], R_[3 + a]); }
    }
    put_node(out, id, s, e, total, mn, mx);
}

}  // namespace rtl

namespace rtk {

size_t lbvh_scratch_bytes(int n) {
    const size_t N = (size_t)n;
    return N * 12 + N * 4 + (2 * N) * 4 + 64 + radix_pairs_bytes(n) + 256;
}

int lbvh_build(const float* d_aabbs, int n, uint32_t* d_nodes, int* d_ordered, void* ws, hipStream_t s) {
    if (n <= 0) { rt::set_error("lbvh: no boxes"); return -1; }
    const size_t N = (size_t)n;
    const int total = 2 * n - 1;
    const int T = rtl::kT;
    char* p = (char*)ws;
    float* cen = (float*)p; p += N * 12;
    uint32_t* keys = (uint32_t*)p; p += N * 4;
    int* level = (int*)p; p += (2 * N) * 4;
    int* small = (int*)p; p += 64;                   // bounds (6 ints)
    void* sortWs = p;
    if (n <= rtl::kSmallBoxes) {
        hipLaunchKernelGGL(rtl::k_rank_sort, dim3((n + 63) / 64), dim3(rtl::kRankT), 0, s, d_aabbs, n, d_ordered,
                           (float2*)ws);
        hipLaunchKernelGGL(rtl::k_wave_boxes, dim3((total + T / 64 - 1) / (T / 64)), dim3(T), 0, s, (const float2*)ws, n,
                           total, d_nodes);
    } else {
        const int g = (int)std::min<size_t>((N + T - 1) / T, 1024);
        hipLaunchKernelGGL(rtl::k_init_bounds, dim3(1), dim3(64), 0, s, small);
        hipLaunchKernelGGL(rtl::k_centroids, dim3(g), dim3(T), 0, s, d_aabbs, n, cen, small);
        hipLaunchKernelGGL(rtl::k_keys, dim3((n + T - 1) / T), dim3(T), 0, s, cen, n, small, keys, d_ordered);
        if (radix_sort_pairs(keys, d_ordered, n, 30, sortWs, s) != 0) return -1;
        // bottom-up, one tree level per launch; the deepest is ceil(log2 n)
        const dim3 gt((unsigned)((total + T - 1) / T));
        hipLaunchKernelGGL(rtl::k_levels, gt, dim3(T), 0, s, n, total, level);
        int deepest = 0;
        while ((1ll << deepest) < n) deepest++;
        for (int L = deepest; L >= 0; L--)
            hipLaunchKernelGGL(rtl::k_level_boxes, gt, dim3(T), 0, s, d_aabbs, d_ordered, n, total, level, L, d_nodes);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) { rt::set_error("lbvh launch failed: %s", hipGetErrorString(e)); return -1; }
    return 0;
}

}  // namespace rtk
