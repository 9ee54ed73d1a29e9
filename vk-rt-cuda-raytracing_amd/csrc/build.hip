// build.hip — binned-SAH BVH2 -> BVH4 build on the GPU.
//
// The algorithm is the reference's host builder (layer/cuda_bvh_backend.cu
// :201-251: 16 centroid bins per axis, bin = floor((c-cmin)/(cmax-cmin)*15),
// cost = nL*SA(L)/SA(P) + nR*SA(R)/SA(P) + 1, leaves of <= maxLeaf
// triangles) with two rules made exact: the partition is taken on the
// evaluated bin boundary and is stable, and a node whose centroids coincide on
// every axis splits at the middle of its range. Under those rules the tree is
// a pure function of the input, and this build yields bit for bit the tree of
// a recursive host build:
//
//  * top phase, one level at a time, for nodes of more than kSmall
//    primitives: bins in LDS per 4096-primitive chunk of a node, merged with
//    atomics (box min/max as order-preserving integers, so the order does not
//    matter); one workgroup per node evaluates the 45 SAH candidates in the
//    host order and, from the chunks' bin counts, where each chunk's left
//    primitives go; a stable scatter moves the chunk and reduces the
//    children's box and centroid bounds;
//  * bottom phase, one launch: a workgroup takes a node of at most kSmall
//    primitives with its boxes in LDS and builds the whole subtree, one wave
//    per node and level, then the subtree's collapse costs;
//  * a node's depth-first pre-order number needs no renumbering passes: it is
//    twice the number of leaves before its first primitive (one scan of the
//    leaf-start flags) plus the left turns on its path (less one per earlier
//    tree of a forest);
//  * the BVH2 is collapsed into the reference's 64-byte BVH4 nodes (backend
//    :31-34, :391-418), FP16 bounds rounded outward. Which BVH2 nodes become
//    BVH4 nodes is a surface-area choice (dynamic programming over the BVH2,
//    bottom-up costs then top-down slot counts): the least total area of BVH4
//    nodes, i.e. the fewest expected node visits, with up to four slots per
//    node. The reference opens both children of every other level, which
//    leaves 45 % of the nodes 2-wide on the 3.4 M-triangle terrain.
//
// What bounds it: LDS atomics and dependent LDS steps of the bottom phase, the
// memory passes (two per level) and launches (four per level) of the top one.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <vector>

#include "rt_internal.h"
#include "rt_scan.h"

namespace rtb {

constexpr int kBins = 16;
constexpr int kBinInts = 7;                 // box min xyz, max xyz (ordered ints), count
constexpr int kCells = 3 * kBins;           // bins of the three axes
constexpr int kSlotInts = kBinInts * kCells;   // a node's bins: [7][3][16]
constexpr int kThreads = 256;

// Nodes of at most kSmall primitives are built to their leaves by one
// workgroup (k_subtree); larger ones are split level by level in chunks of
// kChunk primitives.
constexpr int kSmall = 2048;
constexpr int kTopThreads = 512;
constexpr int kPerThread = 8;
constexpr int kChunk = kTopThreads * kPerThread;

__device__ __forceinline__ int f2o(float f) {
    const int i = __float_as_int(f);
    return i >= 0 ? i : i ^ 0x7fffffff;
}
__device__ __forceinline__ float o2f(int i) { return __int_as_float(i >= 0 ? i : i ^ 0x7fffffff); }
constexpr int kOrdPosInf = 0x7f800000;      // f2o(+inf)
constexpr int kOrdNegInf = (int)0x807fffff; // f2o(-inf)

__device__ __forceinline__ float area(float x0, float y0, float z0, float x1, float y1, float z1) {
    const float dx = x1 - x0, dy = y1 - y0, dz = z1 - z0;
    return 2.f * (dx * dy + dy * dz + dz * dx);
}

__device__ __forceinline__ int bin_of(float c, float cmin, float cmax) {
    int b = (int)((c - cmin) / (cmax - cmin) * (float)(kBins - 1));
    return b < 0 ? 0 : (b >= kBins ? kBins - 1 : b);
}

// --- cross-lane primitives (DPP) ---
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp(int old, int v) {
    return __builtin_amdgcn_update_dpp(old, v, CTRL, ROWS, 0xf, false);
}
// min / max over the 64 lanes (every lane active), wave-uniform result
__device__ __forceinline__ int wave_min(int v) {
    v = min(v, dpp<0x111, 0xf>(v, v)); v = min(v, dpp<0x112, 0xf>(v, v));
    v = min(v, dpp<0x114, 0xf>(v, v)); v = min(v, dpp<0x118, 0xf>(v, v));
    v = min(v, dpp<0x142, 0xa>(v, v)); v = min(v, dpp<0x143, 0xc>(v, v));
    return __builtin_amdgcn_readlane(v, 63);
}
__device__ __forceinline__ int wave_max(int v) {
    v = max(v, dpp<0x111, 0xf>(v, v)); v = max(v, dpp<0x112, 0xf>(v, v));
    v = max(v, dpp<0x114, 0xf>(v, v)); v = max(v, dpp<0x118, 0xf>(v, v));
    v = max(v, dpp<0x142, 0xa>(v, v)); v = max(v, dpp<0x143, 0xc>(v, v));
    return __builtin_amdgcn_readlane(v, 63);
}
__device__ __forceinline__ float wave_minf(float x) { return o2f(wave_min(f2o(x))); }
// lane l's value as seen from D lanes to the left (row_shr) / right (row_shl)
// within its 16-lane row; `none` beyond the row
template <int D> __device__ __forceinline__ int from_left(int none, int v) { return dpp<0x110 + D, 0xf>(none, v); }
template <int D> __device__ __forceinline__ int from_right(int none, int v) { return dpp<0x100 + D, 0xf>(none, v); }
template <int D> __device__ __forceinline__ float from_left(float none, float v) {
    return __int_as_float(from_left<D>(__float_as_int(none), __float_as_int(v)));
}
template <int D> __device__ __forceinline__ float from_right(float none, float v) {
    return __int_as_float(from_right<D>(__float_as_int(none), __float_as_int(v)));
}
__device__ __forceinline__ float lane_of(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// ------------------------------- data ----------------------------------------
// A tree node while it is being built covers the primitives at positions
// [s, s + c). lt: left turns on its path from the root; tree: its scene.
struct Seg { int s, c, lt, tree; };

// An internal node of the top phase. left / right: >= 0 a top node, < 0 the
// subtree -1 - ref.
struct Top { int s, m, lt, tree, left, right; float box[6]; };   // m: first primitive of the right child

// A subtree of at most kSmall primitives. buf: which of the two index buffers
// holds its primitives; bounds: box and centroid bounds (ordered ints).
// level: BVH2 level of its root; levels: its own (set by k_subtree).
struct Small { Seg g; int buf, level, levels, pad; int bounds[12]; };

// A node of a subtree: box, first primitive and left turns (both counted from
// the subtree's), and either the left child's record (the right one follows)
// with the split position m, or kLeaf and the primitive count in m.
struct Rec { float4 a; float2 b; unsigned short s, lt, child, m; };
constexpr unsigned short kLeaf = 0xffff;

struct Build {
    int n, maxLeaf, numScenes, maxBig;
    int maxNodes;            // top nodes, and subtrees, that there is room for
    float4* pbox;            // [n][2] primitive boxes, original index
    int* idx[2];             // [n] primitive at position (ping-pong of the top phase)
    int* ordered;            // [n] final order
    int* leafFlag;           // [n] 1 where a leaf starts
    const int* off;          // [numScenes + 1] scene offsets
    const int* primBase;     // [numScenes + 1] chunks of kChunk primitives before each scene
    int* rootAcc;            // [numScenes][12] root bounds (ordered ints)
    int* rootRef;            // [numScenes] top node or -1 - subtree
    unsigned long long* bnd; // [numScenes][6] scene bounds as (ordered value, first position) keys
    // active nodes of a level (ping-pong)
    Seg* act[2];             // [maxBig]
    int* actAcc[2];          // [maxBig][12]
    int* chunkBase[2];       // [maxBig + 1] chunks before each active node
    int* bins[2];            // [2 maxBig][3][16][7]
    int* childAcc;           // [2 maxBig][12]
    int* sAxis;              // [maxBig] split axis (-1: middle split)
    int* sBin;               // last left bin
    int* sNl;                // left count
    int* chunkHist;          // [chunks][48] primitives per axis and bin
    int* chunkLeft;          // [chunks] left primitives of the node before the chunk
    int* count;              // [8]: 0 active nodes, 1 their chunks, 2 subtrees, 3 set when maxNodes is exceeded, 4 / 5 leaf and head totals, 6 / 7 BVH4 / BVH2 levels
    int* topLevel;           // [maxNodes + 2] first top node of each level
    Top* top;                // top nodes, level by level
    float4* topCost;
    int2* topAsg;            // (slots presented as, BVH4 level)
    Small* small;
    float4* smallCost;
    int2* smallAsg;
    Rec* rec;                // subtree records: from 2 * first position
    float4* cost;            // collapse costs, as rec
    unsigned short* lvl;     // first record of each level of a subtree, from 2 * first position
    int* leafRank;           // [n] leaves before a position
};

__device__ __forceinline__ int pre_of(const Build& b, int s, int lt, int tree) { return 2 * b.leafRank[s] + lt - tree; }

// Scene of primitive i: the last s with off[s] <= i (off: numScenes+1 ascending offsets).
__device__ __forceinline__ int scene_of(const int* off, int numScenes, int i) {
    int lo = 0, hi = numScenes - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (off[mid] <= i) lo = mid; else hi = mid - 1;
    }
    return lo;
}

// Segment of chunk c: the last j < m with base[j] <= c (a 64-ary search, the
// same in every wave).
__device__ __forceinline__ int find_seg(const int* base, int m, int c) {
    const int lane = threadIdx.x & 63;
    int lo = 0, len = m;
    while (len > 1) {
        const int step = (len + 63) >> 6;
        const int k = lo + lane * step;
        const bool le = lane * step < len && base[k] <= c;
        const int hits = __popcll(__ballot(le));
        lo += (hits - 1) * step;
        len = min(step, m - lo);
    }
    return lo;
}

__device__ __forceinline__ void load_box(const float4* pbox, int p, float (&v)[6]) {
    const float4 a = pbox[2 * (size_t)p];
    const float2 b = *(const float2*)&pbox[2 * (size_t)p + 1];
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y;
}
// Centroid of a primitive box (one float expression everywhere).
__device__ __forceinline__ float centroid(const float (&v)[6], int a) { return (v[a] + v[3 + a]) * .5f; }

// Bounds of up to kPerThread primitives per thread (box and centroid, ordered
// ints), reduced over the workgroup into dst with 12 atomics.
template <int NT>
struct BoundsAcc {
    int v[12];
    __device__ __forceinline__ void init() {
#pragma unroll
        for (int k = 0; k < 12; k++) v[k] = (k % 6) < 3 ? kOrdPosInf : kOrdNegInf;
    }
    __device__ __forceinline__ void add(const float (&bx)[6]) {
#pragma unroll
        for (int a = 0; a < 3; a++) {
            v[a] = min(v[a], f2o(bx[a])); v[3 + a] = max(v[3 + a], f2o(bx[3 + a]));
            const int c = f2o(centroid(bx, a));
            v[6 + a] = min(v[6 + a], c); v[9 + a] = max(v[9 + a], c);
        }
    }
    // lds: NT / 64 * 12 ints; every thread of the workgroup calls it
    __device__ __forceinline__ void flush(int* lds, int* dst) {
        const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
        for (int k = 0; k < 12; k++) {
            const int r = (k % 6) < 3 ? wave_min(v[k]) : wave_max(v[k]);
            if (lane == 0) lds[w * 12 + k] = r;
        }
        __syncthreads();
        if (threadIdx.x < 12) {
            const int k = threadIdx.x;
            int r = lds[k];
            for (int j = 1; j < NT / 64; j++) r = (k % 6) < 3 ? min(r, lds[j * 12 + k]) : max(r, lds[j * 12 + k]);
            if ((k % 6) < 3) atomicMin(&dst[k], r); else atomicMax(&dst[k], r);
        }
        __syncthreads();
    }
};

// Empty value of word i of (consecutive) bins.
__device__ __forceinline__ int empty_bin(int i) {
    const int f = i % kSlotInts / kCells;
    return f < 3 ? kOrdPosInf : (f < 6 ? kOrdNegInf : 0);
}

__global__ void k_build_init(Build b, int slots) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < b.numScenes * 12) b.rootAcc[i] = (i % 6) < 3 ? kOrdPosInf : kOrdNegInf;
    if (i < b.numScenes * 6) b.bnd[i] = ~0ull;
    if (i < 8) b.count[i] = 0;
    if (i == 0) b.topLevel[0] = 0;
    if (i < slots * kSlotInts) {
        b.bins[0][i] = empty_bin(i);
    }
}

// ------------------------------- top phase -----------------------------------
// Primitive boxes and identity order, the scenes' root bounds and their exact
// bounds. The latter keep, as a sequential std::min / std::max pass over the
// scene's triangles would, the first of equal values (the sign of a zero) and
// skip NaN: each axis reduces a 64-bit key of the ordered value and the
// position of the coordinate.
__global__ __launch_bounds__(kTopThreads) void k_prims(Build b, const float* __restrict__ tris) {
    __shared__ int lds[kTopThreads / 64 * 12];
    __shared__ unsigned long long lk[kTopThreads / 64][6];
    const int j = find_seg(b.primBase, b.numScenes, blockIdx.x);
    const int s = b.off[j], c = b.off[j + 1] - s;
    const int p0 = (blockIdx.x - b.primBase[j]) * kChunk;
    BoundsAcc<kTopThreads> acc;
    acc.init();
    unsigned long long key[6];
#pragma unroll
    for (int k = 0; k < 6; k++) key[k] = ~0ull;
    for (int k = 0; k < kPerThread; k++) {
        const int q = p0 + k * kTopThreads + threadIdx.x;
        if (q >= c) break;
        const int i = s + q;
        const float* t = tris + 9 * (size_t)i;
        float x[9], v[6];
#pragma unroll
        for (int e = 0; e < 9; e++) x[e] = t[e];
#pragma unroll
        for (int a = 0; a < 3; a++) {
            v[a] = fminf(fminf(x[a], x[3 + a]), x[6 + a]) + 0.0f;   // + 0: -0 -> +0
            v[3 + a] = fmaxf(fmaxf(x[a], x[3 + a]), x[6 + a]) + 0.0f;
        }
        b.pbox[2 * (size_t)i] = make_float4(v[0], v[1], v[2], v[3]);
        b.pbox[2 * (size_t)i + 1] = make_float4(v[4], v[5], 0.f, 0.f);
        b.idx[0][i] = i;
        acc.add(v);
#pragma unroll
        for (int e = 0; e < 9; e++) {
            if (x[e] == x[e]) {
                const int a = e % 3;
                const unsigned int o = (unsigned int)f2o(x[e] + 0.0f) ^ 0x80000000u;
                const unsigned int pos = 3u * (unsigned int)i + (unsigned int)(e / 3);
                const unsigned long long lo = (unsigned long long)o << 32 | pos;
                const unsigned long long hi = (unsigned long long)~o << 32 | pos;
                if (lo < key[a]) key[a] = lo;
                if (hi < key[3 + a]) key[3 + a] = hi;
            }
        }
    }
    acc.flush(lds, b.rootAcc + 12 * (size_t)j);
#pragma unroll
    for (int k = 0; k < 6; k++) {
        unsigned long long v = key[k];
        for (int d = 32; d > 0; d >>= 1) {
            const unsigned long long o = __shfl_xor(v, d, 64);
            if (o < v) v = o;
        }
        if ((threadIdx.x & 63) == 0) lk[threadIdx.x >> 6][k] = v;
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        unsigned long long v = lk[0][threadIdx.x];
        for (int w = 1; w < kTopThreads / 64; w++) v = min(v, lk[w][threadIdx.x]);
        atomicMin(&b.bnd[6 * (size_t)j + threadIdx.x], v);
    }
}

// Keys -> the coordinates they name (n of them, six per scene); an axis without
// a value below 1e30 (above -1e30) keeps that bound, as the sequential pass does.
__global__ void k_scene_bounds(const float* tris, const unsigned long long* bnd, int n, float* out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, k = i % 6;
    if (i >= n) return;
    float r = k < 3 ? 1e30f : -1e30f;
    if (bnd[i] != ~0ull) {
        const unsigned int pos = (unsigned int)bnd[i];
        const float x = tris[9 * (size_t)(pos / 3) + 3 * (pos % 3) + k % 3];
        if (k < 3 ? x < r : r < x) r = x;
    }
    out[i] = r;
}

// Next level's active nodes: the children (2 m of them, or with `init` the
// numScenes roots) of more than kSmall primitives in order, with their chunk
// numbering; the others become subtrees. One workgroup. `out` is the parity
// of the arrays written (and of the index buffer that holds the children's
// primitives).
__global__ __launch_bounds__(1024) void k_top_next(Build b, int out, int init, int level) {
    __shared__ int lds[1024 / 64 + 1];
    const int in = out ^ 1;
    const int m = init ? 0 : b.count[0], kids = init ? b.numScenes : 2 * m;
    const int topBase = init ? 0 : b.topLevel[level];
    const int smallBase = b.count[2];
    __syncthreads();                       // every thread has read count before it changes
    int nbig = 0, nsmall = 0, nchunks = 0;
    for (int k0 = 0; k0 < kids; k0 += 1024) {
        const int k = k0 + threadIdx.x;
        const bool valid = k < kids;
        Seg g{0, 0, 0, 0};
        const int* acc = nullptr;
        if (valid && init) {
            g = Seg{b.off[k], b.off[k + 1] - b.off[k], 0, k};
            acc = b.rootAcc + 12 * (size_t)k;
        } else if (valid) {
            const Seg p = b.act[in][k >> 1];
            const int nl = b.sNl[k >> 1];
            g = (k & 1) ? Seg{p.s + nl, p.c - nl, p.lt, p.tree} : Seg{p.s, nl, p.lt + 1, p.tree};
            acc = b.childAcc + 12 * (size_t)k;
        }
        const bool big = valid && g.c > kSmall;
        const int chunks = big ? (g.c + kChunk - 1) / kChunk : 0;
        int tb, ts, tc;
        const int rb = nbig + rts::block_exclusive_scan<1024>(big ? 1 : 0, lds, &tb);
        const int rs = nsmall + rts::block_exclusive_scan<1024>(valid && !big ? 1 : 0, lds, &ts);
        const int rc = nchunks + rts::block_exclusive_scan<1024>(chunks, lds, &tc);
        if (valid) {
            int ref;
            if (big) {
                b.act[out][rb] = g;
                b.chunkBase[out][rb] = rc;
                for (int q = 0; q < 12; q++) b.actAcc[out][12 * (size_t)rb + q] = acc[q];
                ref = topBase + m + rb;            // top nodes are numbered level by level
            } else if (smallBase + rs >= b.maxNodes) {
                ref = -1;                          // no room (flagged below): the build starts over
            } else {
                Small& sm = b.small[smallBase + rs];
                sm.g = g;
                sm.buf = out;
                sm.level = init ? 0 : level + 1;
                for (int q = 0; q < 12; q++) sm.bounds[q] = acc[q];
                ref = -1 - (smallBase + rs);
            }
            if (init) b.rootRef[k] = ref;
            else if (k & 1) b.top[topBase + (k >> 1)].right = ref;
            else b.top[topBase + (k >> 1)].left = ref;
        }
        nbig += tb; nsmall += ts; nchunks += tc;
    }
    if (threadIdx.x == 0) {
        const bool full = smallBase + nsmall > b.maxNodes || topBase + m + nbig > b.maxNodes;
        b.chunkBase[out][nbig] = nchunks;
        b.count[0] = full ? 0 : nbig;
        b.count[1] = full ? 0 : nchunks;
        if (full) b.count[3] = 1;
        b.count[2] = smallBase + nsmall;
        b.topLevel[init ? 0 : level + 1] = topBase + m;
    }
}

// Bins of one chunk of an active node: LDS copies (a coherent mesh puts a
// wave's primitives in one bin, and one copy would serialise its atomics),
// merged into the node's bins; the chunk's counts per bin stay for the
// partition.
constexpr int kBinCopies = 8;
constexpr int kCopyStride = kSlotInts + 9;        // copies start on different banks
__global__ __launch_bounds__(kTopThreads) void k_top_bin(Build b, int cur) {
    __shared__ int lb[kBinCopies * kCopyStride];
    if ((int)blockIdx.x >= b.count[1]) return;
    const int j = find_seg(b.chunkBase[cur], b.count[0], blockIdx.x);
    const Seg g = b.act[cur][j];
    const int p0 = ((int)blockIdx.x - b.chunkBase[cur][j]) * kChunk;
    const int* nc = b.actAcc[cur] + 12 * (size_t)j + 6;
    float cmin[3], cmax[3];
    bool use[3];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        cmin[a] = o2f(nc[a]); cmax[a] = o2f(nc[3 + a]);
        use[a] = !(cmax[a] - cmin[a] < 1e-8f);
    }
    for (int i = threadIdx.x; i < kBinCopies * kCopyStride; i += kTopThreads) lb[i] = empty_bin(i % kCopyStride);
    __syncthreads();
    int* mine = lb + (threadIdx.x % kBinCopies) * kCopyStride;
    const int* idx = b.idx[cur] + g.s;
#pragma unroll 2
    for (int k = 0; k < kPerThread; k++) {
        const int i = p0 + k * kTopThreads + threadIdx.x;
        if (i >= g.c) break;
        float v[6];
        load_box(b.pbox, idx[i], v);
#pragma unroll
        for (int a = 0; a < 3; a++) {
            if (!use[a]) continue;
            int* d = mine + a * kBins + bin_of(centroid(v, a), cmin[a], cmax[a]);
#pragma unroll
            for (int e = 0; e < 3; e++) {
                atomicMin(&d[e * kCells], f2o(v[e]));
                atomicMax(&d[(3 + e) * kCells], f2o(v[3 + e]));
            }
            atomicAdd(&d[6 * kCells], 1);
        }
    }
    __syncthreads();
    int* out = b.bins[cur] + (size_t)j * kSlotInts;
    for (int i = threadIdx.x; i < kSlotInts; i += kTopThreads) {
        const int f = i / kCells;
        int v = lb[i];
        for (int k = 1; k < kBinCopies; k++) {
            const int o = lb[k * kCopyStride + i];
            v = f < 3 ? min(v, o) : (f < 6 ? max(v, o) : v + o);
        }
        if (f == 6) {
            b.chunkHist[(size_t)blockIdx.x * kCells + i - 6 * kCells] = v;
            if (v) atomicAdd(&out[i], v);
        } else if (f < 3) {
            if (v != kOrdPosInf) atomicMin(&out[i], v);
        } else if (v != kOrdNegInf) {
            atomicMax(&out[i], v);
        }
    }
}

// SAH candidates of one axis, a 16-lane row per node: the lane of bin q holds
// the candidate that splits after it. In: its bin (ordered ints, count); out:
// left and right box and counts (row scans). Integers order and combine as
// the floats do; with a NaN in some box (`nan`, wave-uniform) the scans run on
// floats, whose min / max skip it.
struct Cand { float L[6], R[6]; int nl, nr; };
__device__ __forceinline__ void sah_scan(const int (&B)[6], int n, bool nan, Cand& c) {
    int ln = n, rn = n;
    if (!nan) {
        int L[6], S[6];
#pragma unroll
        for (int k = 0; k < 6; k++) L[k] = S[k] = B[k];
#define RTB_SCAN(D)                                                                                     \
    {                                                                                                   \
        _Pragma("unroll") for (int k = 0; k < 3; k++) {                                                 \
            L[k] = min(L[k], from_left<D>(kOrdPosInf, L[k]));                                           \
            L[3 + k] = max(L[3 + k], from_left<D>(kOrdNegInf, L[3 + k]));                               \
            S[k] = min(S[k], from_right<D>(kOrdPosInf, S[k]));                                          \
            S[3 + k] = max(S[3 + k], from_right<D>(kOrdNegInf, S[3 + k]));                              \
        }                                                                                               \
        ln += from_left<D>(0, ln);                                                                      \
        rn += from_right<D>(0, rn);                                                                     \
    }
        RTB_SCAN(1) RTB_SCAN(2) RTB_SCAN(4) RTB_SCAN(8)
#undef RTB_SCAN
#pragma unroll
        for (int k = 0; k < 6; k++) {
            c.L[k] = o2f(L[k]);
            c.R[k] = o2f(from_right<1>(k < 3 ? kOrdPosInf : kOrdNegInf, S[k]));
        }
    } else {
        float L[6], S[6];
#pragma unroll
        for (int k = 0; k < 6; k++) L[k] = S[k] = o2f(B[k]);
#define RTB_SCAN(D)                                                                                     \
    {                                                                                                   \
        _Pragma("unroll") for (int k = 0; k < 3; k++) {                                                 \
            L[k] = fminf(L[k], from_left<D>(INFINITY, L[k]));                                           \
            L[3 + k] = fmaxf(L[3 + k], from_left<D>(-INFINITY, L[3 + k]));                              \
            S[k] = fminf(S[k], from_right<D>(INFINITY, S[k]));                                          \
            S[3 + k] = fmaxf(S[3 + k], from_right<D>(-INFINITY, S[3 + k]));                             \
        }                                                                                               \
        ln += from_left<D>(0, ln);                                                                      \
        rn += from_right<D>(0, rn);                                                                     \
    }
        RTB_SCAN(1) RTB_SCAN(2) RTB_SCAN(4) RTB_SCAN(8)
#undef RTB_SCAN
#pragma unroll
        for (int k = 0; k < 6; k++) {
            c.L[k] = L[k];
            c.R[k] = from_right<1>(k < 3 ? INFINITY : -INFINITY, S[k]);
        }
    }
    c.nl = ln;
    c.nr = from_right<1>(0, rn);
}
// An ordered integer outside [-inf, +inf] is a NaN.
__device__ __forceinline__ bool ord_nan(int o) { return o > kOrdPosInf || o < kOrdNegInf; }
__device__ __forceinline__ float sah_cost(const Cand& c, float pA) {
    return (float)c.nl * area(c.L[0], c.L[1], c.L[2], c.L[3], c.L[4], c.L[5]) / pA +
           (float)c.nr * area(c.R[0], c.R[1], c.R[2], c.R[3], c.R[4], c.R[5]) / pA + 1.f;
}

// SAH over 3 axes x 15 boundaries in one wave: lane 16 a + q holds bin q of
// axis a; the first candidate of least cost in the host order (axis-major,
// strict <) wins.
struct Sah {
    int axis, bin, nl;         // split (axis -1: middle split), last left bin, left count; wave-uniform
    int src;                   // the winning lane
    Cand c;                    // this lane's candidate
    bool nan;                  // some bin's box holds a NaN (wave-uniform)
};
__device__ __forceinline__ void sah_wave(const int* bins, float pA, bool use0, bool use1, bool use2, int cnt, Sah& r) {
    const int lane = threadIdx.x & 63;
    const int ax = lane >> 4, q = lane & 15;
    int B[6] = {kOrdPosInf, kOrdPosInf, kOrdPosInf, kOrdNegInf, kOrdNegInf, kOrdNegInf};
    int n = 0;
    if (lane < kCells) {
#pragma unroll
        for (int k = 0; k < 6; k++) B[k] = bins[k * kCells + lane];
        n = bins[6 * kCells + lane];
    }
    r.nan = __any(ord_nan(B[0]) || ord_nan(B[1]) || ord_nan(B[2]) || ord_nan(B[3]) || ord_nan(B[4]) || ord_nan(B[5]));
    sah_scan(B, n, r.nan, r.c);
    const bool use = ax == 0 ? use0 : (ax == 1 ? use1 : (ax == 2 && use2));
    const float cost = sah_cost(r.c, pA);
    const bool ok = use && q < kBins - 1 && r.c.nl != 0 && r.c.nr != 0 && cost < 1e30f;
    const float least = wave_minf(ok ? cost : INFINITY);
    const uint64_t best = __ballot(ok && cost == least);
    if (best == 0) {                               // coincident centroids: middle split
        r.axis = -1; r.bin = -1; r.nl = cnt / 2; r.src = 0;
    } else {
        r.src = __ffsll((unsigned long long)best) - 1;
        r.axis = r.src >> 4;
        r.bin = r.src & 15;
        r.nl = __builtin_amdgcn_readlane(r.c.nl, r.src);
    }
}

// One workgroup per active node: the SAH choice (first wave), the top node,
// the children's empty bounds, cleared bins for two nodes of the next level,
// and the left primitives before each of the node's chunks.
__global__ __launch_bounds__(kThreads) void k_top_split(Build b, int cur, int level) {
    __shared__ int choice[3];
    __shared__ int lds[kThreads / 64 + 1];
    const int j = blockIdx.x;
    if (j >= b.count[0]) return;
    const Seg g = b.act[cur][j];
    const int* nb = b.actAcc[cur] + 12 * (size_t)j;
    if (threadIdx.x < 64) {
        float bx[6], cb[6];
#pragma unroll
        for (int k = 0; k < 6; k++) { bx[k] = o2f(nb[k]); cb[k] = o2f(nb[6 + k]); }
        Sah r;
        sah_wave(b.bins[cur] + (size_t)j * kSlotInts, area(bx[0], bx[1], bx[2], bx[3], bx[4], bx[5]),
                 !(cb[3] - cb[0] < 1e-8f), !(cb[4] - cb[1] < 1e-8f), !(cb[5] - cb[2] < 1e-8f), g.c, r);
        if (threadIdx.x == 0) {
            choice[0] = r.axis; choice[1] = r.bin; choice[2] = r.nl;
            b.sAxis[j] = r.axis; b.sBin[j] = r.bin; b.sNl[j] = r.nl;
            Top& t = b.top[b.topLevel[level] + j];
            t.s = g.s; t.m = g.s + r.nl; t.lt = g.lt; t.tree = g.tree;
#pragma unroll
            for (int k = 0; k < 6; k++) t.box[k] = bx[k];
        }
    }
    if (threadIdx.x < 24) b.childAcc[24 * (size_t)j + threadIdx.x] = (threadIdx.x % 6) < 3 ? kOrdPosInf : kOrdNegInf;
    int* clr = b.bins[cur ^ 1] + 2 * (size_t)j * kSlotInts;
    for (int i = threadIdx.x; i < 2 * kSlotInts; i += kThreads) clr[i] = empty_bin(i);
    __syncthreads();
    const int ax = choice[0], bin = choice[1], nl = choice[2];
    const int c0 = b.chunkBase[cur][j], nch = b.chunkBase[cur][j + 1] - c0;
    int carry = 0;
    for (int q0 = 0; q0 < nch; q0 += kThreads) {
        const int q = q0 + threadIdx.x;
        int left = 0;
        if (q < nch) {
            if (ax < 0) {
                left = max(0, min(nl - q * kChunk, kChunk));
            } else {
                const int* h = b.chunkHist + (size_t)(c0 + q) * kCells + ax * kBins;
                for (int k = 0; k <= bin; k++) left += h[k];
            }
        }
        int tot;
        const int ex = rts::block_exclusive_scan<kThreads>(left, lds, &tot);
        if (q < nch) b.chunkLeft[c0 + q] = carry + ex;
        carry += tot;
    }
}

// Stable partition of one chunk into the other index buffer, and the
// children's box and centroid bounds. A thread takes kPerThread consecutive
// primitives, so one scan of the per-thread left counts ranks the chunk.
__global__ __launch_bounds__(kTopThreads) void k_top_scatter(Build b, int cur) {
    __shared__ int lds[kTopThreads / 64 * 12 + 1];
    if ((int)blockIdx.x >= b.count[1]) return;
    const int j = find_seg(b.chunkBase[cur], b.count[0], blockIdx.x);
    const Seg g = b.act[cur][j];
    const int p0 = ((int)blockIdx.x - b.chunkBase[cur][j]) * kChunk;
    const int ax = b.sAxis[j], bin = b.sBin[j], nl = b.sNl[j];
    const int* nc = b.actAcc[cur] + 12 * (size_t)j + 6;
    const float cmin = ax >= 0 ? o2f(nc[ax]) : 0.f, cmax = ax >= 0 ? o2f(nc[3 + ax]) : 0.f;
    const int* idx = b.idx[cur] + g.s;
    const int i0 = p0 + (int)threadIdx.x * kPerThread;
    int p[kPerThread];
    unsigned int lm = 0;
    BoundsAcc<kTopThreads> accL, accR;
    accL.init();
    accR.init();
#pragma unroll
    for (int k = 0; k < kPerThread; k++) p[k] = i0 + k < g.c ? idx[i0 + k] : -1;
#pragma unroll
    for (int k = 0; k < kPerThread; k++) {
        if (p[k] < 0) continue;
        float v[6];
        load_box(b.pbox, p[k], v);
        bool left;
        if (ax < 0) {
            left = i0 + k < nl;
        } else {
            const float c = ax == 0 ? centroid(v, 0) : (ax == 1 ? centroid(v, 1) : centroid(v, 2));
            left = bin_of(c, cmin, cmax) <= bin;
        }
        if (left) { lm |= 1u << k; accL.add(v); }
        else accR.add(v);
    }
    int tot;
    int before = b.chunkLeft[blockIdx.x] + rts::block_exclusive_scan<kTopThreads>(__popc(lm), lds, &tot);
    int* o = b.idx[cur ^ 1] + g.s;
#pragma unroll
    for (int k = 0; k < kPerThread; k++) {
        if (p[k] < 0) continue;
        if (lm >> k & 1) { o[before] = p[k]; before++; }
        else o[nl + (i0 + k - before)] = p[k];
    }
    accL.flush(lds, b.childAcc + 24 * (size_t)j);
    accR.flush(lds, b.childAcc + 24 * (size_t)j + 12);
}

// ------------------------------- collapse ------------------------------------
// --- BVH2 -> BVH4 collapse (same rule and float operation order as the
// oracle's collapse_costs / collapse_split / collapse_gather) ---
// cost = (c1, c2, c3, c4): least total area of the BVH4 nodes needed to
// present a subtree as k slots; a leaf is one free slot; for an internal node,
// g_k = min over a of c_a(left) + c_{k-a}(right), c1 = area + min g_k.
constexpr float kCostInf = 3.0e38f;

__device__ __forceinline__ float4 leaf_cost() { return make_float4(0.0f, kCostInf, kCostInf, kCostInf); }
__device__ __forceinline__ float4 node_cost(float ar, const float4& L, const float4& R) {
    const float l[4] = {L.x, L.y, L.z, L.w}, r[4] = {R.x, R.y, R.z, R.w};
    float g[5] = {kCostInf, kCostInf, kCostInf, kCostInf, kCostInf};
#pragma unroll
    for (int k = 2; k <= 4; k++)
#pragma unroll
        for (int a = 1; a < k; a++) {
            const float x = l[a - 1] + r[k - a - 1];
            if (x < g[k]) g[k] = x;
        }
    float best = g[2];
    if (g[3] < best) best = g[3];
    if (g[4] < best) best = g[4];
    return make_float4(ar + best, g[2], g[3], g[4]);
}

// Top-down step at an internal node presented as m slots at BVH4 level lev
// (m 0: not reached): a node presented as one slot heads a BVH4 node of its
// cheapest width (ties: the narrower); one presented as m >= 2 slots is
// dissolved into its parent's node. Returns the children's (slots, level) and
// whether the node is a head. lev: BVH4 level of a head / of the node whose
// slots a dissolved node fills.
__device__ __forceinline__ bool assign_slots(const float4& c, const float4& L, const float4& R, int m, int lev, int2& al,
                                             int2& ar) {
    al = ar = make_int2(0, 0);
    if (m == 0) return false;
    int k = m, cl = lev;
    if (m == 1) {
        k = 2;
        if (c.z < c.y) k = 3;
        if (c.w < (k == 3 ? c.z : c.y)) k = 4;
        cl = lev + 1;
    }
    // left slots of k (ties: the smaller)
    const float l[4] = {L.x, L.y, L.z, L.w}, r[4] = {R.x, R.y, R.z, R.w};
    int ba = 1;
    float bx = kCostInf;
#pragma unroll
    for (int a = 1; a < 4; a++) {
        if (a >= k) break;
        const int o = k - a - 1;
        const float x = l[a - 1] + (o == 0 ? r[0] : (o == 1 ? r[1] : r[2]));
        if (x < bx) { bx = x; ba = a; }
    }
    al = make_int2(ba, cl);
    ar = make_int2(k - ba, cl);
    return m == 1;
}

// ------------------------------- subtrees ------------------------------------
// A whole subtree per workgroup: primitive boxes in LDS, level by level. A
// wave takes one node (up to 64 primitives stay in registers, one per lane),
// or four nodes of at most kTiny primitives, a 16-lane row each: most inner
// nodes are that small, and the SAH of one costs nearly as many instructions
// as of four. Leaves write their part of the final order at once.
// MAXQ: most active nodes of a level (kSmall / (maxLeaf + 1)).
constexpr int kSubThreads = 512, kSubWaves = kSubThreads / 64;
constexpr int kTiny = 16;

template <int MAXQ>
struct SubLds {
    float box[6][kSmall];
    unsigned short perm[2][kSmall];
    // active nodes: larger ones from the front, tiny ones from the back
    unsigned int seg[2][MAXQ];                 // start | count << 12
    unsigned short rec[2][MAXQ];
    unsigned short lt[2][MAXQ];                // left turns below the subtree's root
    float pA[2][MAXQ];                         // area of the node's box
    int bins[kSubWaves][kBinInts * 64];
    int nbig[2], ntiny[2], next, recs;
};

// Where a subtree's nodes go.
struct SubOut { Rec* rec; int maxLeaf; };

// The two children of node `rid`: records, and queue entries of those that
// are not leaves. Called by lane 0 of a wave or by one lane per node.
template <int MAXQ>
__device__ __forceinline__ void sub_children(SubLds<MAXQ>& S, const SubOut& o, int nxt, int rid, int lt, int start, int cnt,
                                             int nl, const float (&L)[6], const float (&R)[6]) {
    const int base = atomicAdd(&S.recs, 2);
    o.rec[rid].child = (unsigned short)base;
    o.rec[rid].m = (unsigned short)(start + nl);
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const int cs = k ? start + nl : start, cc = k ? cnt - nl : nl, cl = k ? lt : lt + 1;
        const float x[6] = {k ? R[0] : L[0], k ? R[1] : L[1], k ? R[2] : L[2], k ? R[3] : L[3], k ? R[4] : L[4],
                            k ? R[5] : L[5]};
        Rec& c = o.rec[base + k];
        c.a = make_float4(x[0], x[1], x[2], x[3]);
        c.b = make_float2(x[4], x[5]);
        c.s = (unsigned short)cs;
        c.lt = (unsigned short)cl;
        if (cc <= o.maxLeaf) {
            c.child = kLeaf;
            c.m = (unsigned short)cc;
        } else {
            const int q = cc > kTiny ? atomicAdd(&S.nbig[nxt], 1) : MAXQ - 1 - atomicAdd(&S.ntiny[nxt], 1);
            S.seg[nxt][q] = (unsigned int)cs | (unsigned int)cc << 12;
            S.rec[nxt][q] = (unsigned short)(base + k);
            S.lt[nxt][q] = (unsigned short)cl;
            S.pA[nxt][q] = area(x[0], x[1], x[2], x[3], x[4], x[5]);
        }
    }
}

// One node by one wave.
template <int MAXQ>
__device__ __forceinline__ void sub_node(SubLds<MAXQ>& S, const SubOut& o, int cur, int j, int* lb, const int* idxIn,
                                         int* ordered, int* leafFlag) {
    const int lane = threadIdx.x & 63;
    const unsigned int sg = S.seg[cur][j];
    const int start = __builtin_amdgcn_readfirstlane((int)(sg & 0xfffu));
    const int cnt = __builtin_amdgcn_readfirstlane((int)(sg >> 12));
    const float pA = S.pA[cur][j];
    const unsigned short* perm = S.perm[cur];
    unsigned short* perm2 = S.perm[cur ^ 1];
    const bool one = cnt <= 64;                // the node's primitives fit the wave's lanes
    int myp = 0;
    float v[6] = {0, 0, 0, 0, 0, 0};
    // centroid bounds
    int cb[6] = {kOrdPosInf, kOrdPosInf, kOrdPosInf, kOrdNegInf, kOrdNegInf, kOrdNegInf};
    for (int i = lane; i < cnt; i += 64) {
        myp = perm[start + i];
#pragma unroll
        for (int k = 0; k < 6; k++) v[k] = S.box[k][myp];
#pragma unroll
        for (int a = 0; a < 3; a++) {
            const int c = f2o(centroid(v, a));
            cb[a] = min(cb[a], c); cb[3 + a] = max(cb[3 + a], c);
        }
    }
    float cmin[3], cmax[3];
    bool use[3];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        cmin[a] = o2f(wave_min(cb[a])); cmax[a] = o2f(wave_max(cb[3 + a]));
        use[a] = !(cmax[a] - cmin[a] < 1e-8f);
    }
    // bins
    if (lane < kCells) {
#pragma unroll
        for (int f = 0; f < kBinInts; f++) lb[f * kCells + lane] = f < 3 ? kOrdPosInf : (f < 6 ? kOrdNegInf : 0);
    }
    wave_lds_fence();
    int mb[3] = {0, 0, 0};
    for (int i = lane; i < cnt; i += 64) {
        if (!one) {
            myp = perm[start + i];
#pragma unroll
            for (int k = 0; k < 6; k++) v[k] = S.box[k][myp];
        }
#pragma unroll
        for (int a = 0; a < 3; a++) {
            if (!use[a]) continue;
            mb[a] = bin_of(centroid(v, a), cmin[a], cmax[a]);
            int* d = lb + a * kBins + mb[a];
#pragma unroll
            for (int e = 0; e < 3; e++) {
                atomicMin(&d[e * kCells], f2o(v[e]));
                atomicMax(&d[(3 + e) * kCells], f2o(v[3 + e]));
            }
            atomicAdd(&d[6 * kCells], 1);
        }
    }
    wave_lds_fence();
    Sah r;
    sah_wave(lb, pA, use[0], use[1], use[2], cnt, r);
    const int ax = r.axis, bin = r.bin, nl = r.nl;
    const bool leafL = nl <= o.maxLeaf, leafR = cnt - nl <= o.maxLeaf;
    // Stable partition. The children's boxes are the winning candidate's; a
    // middle split has none, and with a NaN box the scans (which skip NaN)
    // could differ from a reduction over ordered integers, so those reduce.
    const bool exact = ax < 0 || r.nan;
    const float smin = ax == 1 ? cmin[1] : (ax == 2 ? cmin[2] : cmin[0]);
    const float smax = ax == 1 ? cmax[1] : (ax == 2 ? cmax[2] : cmax[0]);
    int xb[12];
#pragma unroll
    for (int k = 0; k < 12; k++) xb[k] = (k % 6) < 3 ? kOrdPosInf : kOrdNegInf;
    int leftBefore = 0;
    for (int base = 0; base < cnt; base += 64) {
        const int i = base + lane;
        const bool valid = i < cnt;
        bool left = false;
        if (valid) {
            if (!one) {
                myp = perm[start + i];
                if (ax >= 0) mb[0] = bin_of((S.box[ax][myp] + S.box[3 + ax][myp]) * .5f, smin, smax);
            } else {
                mb[0] = ax == 1 ? mb[1] : (ax == 2 ? mb[2] : mb[0]);
            }
            left = ax < 0 ? i < nl : mb[0] <= bin;
            if (exact) {
#pragma unroll
                for (int e = 0; e < 3; e++) {
                    const int lo = f2o(S.box[e][myp]), hi = f2o(S.box[3 + e][myp]);
                    if (left) { xb[e] = min(xb[e], lo); xb[3 + e] = max(xb[3 + e], hi); }
                    else { xb[6 + e] = min(xb[6 + e], lo); xb[9 + e] = max(xb[9 + e], hi); }
                }
            }
        }
        const uint64_t lm = __ballot(valid && left);
        const int lr = leftBefore + __popcll(lm & ((1ull << lane) - 1ull));
        if (valid) {
            const int pos = start + (left ? lr : nl + (i - lr));
            if (left ? leafL : leafR) {
                ordered[pos] = idxIn[myp];
                leafFlag[pos] = pos == start + (left ? 0 : nl);
            } else {
                perm2[pos] = (unsigned short)myp;
            }
        }
        leftBefore += __popcll(lm);
    }
    float L[6], R[6];
    if (exact) {
#pragma unroll
        for (int k = 0; k < 6; k++) {
            L[k] = o2f(k < 3 ? wave_min(xb[k]) : wave_max(xb[k]));
            R[k] = o2f(k < 3 ? wave_min(xb[6 + k]) : wave_max(xb[6 + k]));
        }
    } else {
#pragma unroll
        for (int k = 0; k < 6; k++) { L[k] = lane_of(r.c.L[k], r.src); R[k] = lane_of(r.c.R[k], r.src); }
    }
    if (lane == 0) sub_children(S, o, cur ^ 1, S.rec[cur][j], S.lt[cur][j], start, cnt, nl, L, R);
}

// min / max over a 16-lane row, in every lane of it
__device__ __forceinline__ int row_min(int v) {
    v = min(v, dpp<0x128, 0xf>(v, v)); v = min(v, dpp<0x124, 0xf>(v, v));   // rotations by 8, 4, 2, 1
    v = min(v, dpp<0x122, 0xf>(v, v)); return min(v, dpp<0x121, 0xf>(v, v));
}
__device__ __forceinline__ int row_max(int v) {
    v = max(v, dpp<0x128, 0xf>(v, v)); v = max(v, dpp<0x124, 0xf>(v, v));
    v = max(v, dpp<0x122, 0xf>(v, v)); return max(v, dpp<0x121, 0xf>(v, v));
}

// Four tiny nodes by one wave: queue entries [t0, min(t0 + 4, count)) counted
// from the back, one per 16-lane row, one axis at a time. Each lane keeps its
// cheapest candidate of the three axes (the first of equals); the row's least
// (cost, axis, bin) wins and that lane writes the children. Rows that need
// the general path (no candidate, a NaN box) are left to sub_node.
template <int MAXQ>
__device__ __forceinline__ void sub_tiny(SubLds<MAXQ>& S, const SubOut& o, int cur, int t0, int count, int* lb,
                                         const int* idxIn, int* ordered, int* leafFlag) {
    const int lane = threadIdx.x & 63, row = lane >> 4, q = lane & 15;
    const bool node = t0 + row < count;
    const int j = node ? MAXQ - 1 - (t0 + row) : MAXQ - 1;
    const unsigned int sg = S.seg[cur][j];
    const int start = (int)(sg & 0xfffu), cnt = node ? (int)(sg >> 12) : 0;
    const float pA = S.pA[cur][j];
    const bool valid = q < cnt;
    int myp = 0;
    float v[6] = {0, 0, 0, 0, 0, 0};
    int ob[6] = {kOrdPosInf, kOrdPosInf, kOrdPosInf, kOrdNegInf, kOrdNegInf, kOrdNegInf};
    float cen[3], cmin[3], cmax[3];
    bool use[3];
    if (valid) {
        myp = S.perm[cur][start + q];
#pragma unroll
        for (int k = 0; k < 6; k++) { v[k] = S.box[k][myp]; ob[k] = f2o(v[k]); }
    }
#pragma unroll
    for (int a = 0; a < 3; a++) {
        cen[a] = centroid(v, a);
        const int c = f2o(cen[a]);
        cmin[a] = o2f(row_min(valid ? c : kOrdPosInf));
        cmax[a] = o2f(row_max(valid ? c : kOrdNegInf));
        use[a] = !(cmax[a] - cmin[a] < 1e-8f);
    }
    const bool nan = __any(ord_nan(ob[0]) || ord_nan(ob[1]) || ord_nan(ob[2]) || ord_nan(ob[3]) || ord_nan(ob[4]) ||
                           ord_nan(ob[5]));
    int best = -1;                                 // axis * 16 + bin of this lane's cheapest candidate
    float bestCost = INFINITY;
    int nl = 0, mybin[3] = {0, 0, 0};
    float L[6], R[6];
#pragma unroll
    for (int k = 0; k < 6; k++) L[k] = R[k] = 0.f;
    if (!nan) {
#pragma unroll
        for (int a = 0; a < 3; a++) {
            // one axis' bins of the four nodes: [7][64], a lane's bin in its column
#pragma unroll
            for (int f = 0; f < kBinInts; f++) lb[f * 64 + lane] = f < 3 ? kOrdPosInf : (f < 6 ? kOrdNegInf : 0);
            wave_lds_fence();
            if (valid && use[a]) {
                mybin[a] = bin_of(cen[a], cmin[a], cmax[a]);
                int* d = lb + row * 16 + mybin[a];
#pragma unroll
                for (int e = 0; e < 3; e++) {
                    atomicMin(&d[e * 64], ob[e]);
                    atomicMax(&d[(3 + e) * 64], ob[3 + e]);
                }
                atomicAdd(&d[6 * 64], 1);
            }
            wave_lds_fence();
            int B[6];
#pragma unroll
            for (int k = 0; k < 6; k++) B[k] = lb[k * 64 + lane];
            const int n = lb[6 * 64 + lane];
            wave_lds_fence();
            Cand c;
            sah_scan(B, n, false, c);
            const float cost = sah_cost(c, pA);
            if (use[a] && q < kBins - 1 && c.nl != 0 && c.nr != 0 && cost < 1e30f && cost < bestCost) {
                bestCost = cost;
                best = a * 16 + q;
                nl = c.nl;
#pragma unroll
                for (int k = 0; k < 6; k++) { L[k] = c.L[k]; R[k] = c.R[k]; }
            }
        }
    }
    constexpr int kNone = 1 << 20;
    const int least = row_min(f2o(bestCost));
    const int key = best >= 0 && f2o(bestCost) == least ? best : kNone;
    const int wk = row_min(key);
    const bool won = node && wk != kNone;          // the row has a split
    const int rnl = row_max(key == wk ? nl : -1);
    const int ax = wk >> 4;
    const bool left = valid && (ax == 0 ? mybin[0] : (ax == 1 ? mybin[1] : mybin[2])) <= (wk & 15);
    const unsigned int lm = (unsigned int)(__ballot(left) >> (row * 16)) & 0xffffu;
    if (won && valid) {
        const int lr = __popc(lm & ((1u << q) - 1u));
        const int pos = start + (left ? lr : rnl + (q - lr));
        if ((left ? rnl : cnt - rnl) <= o.maxLeaf) {
            ordered[pos] = idxIn[myp];
            leafFlag[pos] = pos == start + (left ? 0 : rnl);
        } else {
            S.perm[cur ^ 1][pos] = (unsigned short)myp;
        }
    }
    if (won && key == wk) sub_children(S, o, cur ^ 1, S.rec[cur][j], S.lt[cur][j], start, cnt, nl, L, R);
    uint64_t rest = __ballot(node && !won && q == 0);
    while (rest) {
        const int r = (__ffsll((unsigned long long)rest) - 1) >> 4;
        rest &= rest - 1;
        wave_lds_fence();
        sub_node(S, o, cur, MAXQ - 1 - (t0 + r), lb, idxIn, ordered, leafFlag);
    }
}

template <int MAXQ>
__global__ __launch_bounds__(kSubThreads) void k_subtree(Build b) {
    __shared__ __attribute__((aligned(16))) SubLds<MAXQ> S;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const Small& sm = b.small[blockIdx.x];
    const Seg g = sm.g;
    const int* idxIn = b.idx[sm.buf] + g.s;
    int* ordered = b.ordered + g.s;
    int* leafFlag = b.leafFlag + g.s;
    Rec* rec = b.rec + 2 * (size_t)g.s;
    unsigned short* lvl = b.lvl + 2 * (size_t)g.s;
    const SubOut o{rec, b.maxLeaf};
    float rb[6];
#pragma unroll
    for (int k = 0; k < 6; k++) rb[k] = o2f(sm.bounds[k]);
    const bool rootLeaf = g.c <= b.maxLeaf;
    for (int i = tid; i < g.c; i += kSubThreads) {
        const int p = idxIn[i];
        float v[6];
        load_box(b.pbox, p, v);
#pragma unroll
        for (int k = 0; k < 6; k++) S.box[k][i] = v[k];
        S.perm[0][i] = (unsigned short)i;
        if (rootLeaf) { ordered[i] = p; leafFlag[i] = i == 0; }
    }
    if (tid == 0) {
        rec[0].a = make_float4(rb[0], rb[1], rb[2], rb[3]);
        rec[0].b = make_float2(rb[4], rb[5]);
        rec[0].s = rec[0].lt = 0;
        if (rootLeaf) { rec[0].child = kLeaf; rec[0].m = (unsigned short)g.c; }
        S.recs = 1;
        S.next = 0;
        const bool tiny = g.c <= kTiny;
        S.nbig[0] = !rootLeaf && !tiny; S.ntiny[0] = !rootLeaf && tiny;
        S.nbig[1] = S.ntiny[1] = 0;
        const int q = tiny ? MAXQ - 1 : 0;
        S.seg[0][q] = (unsigned int)g.c << 12;
        S.rec[0][q] = 0;
        S.lt[0][q] = 0;
        S.pA[0][q] = area(rb[0], rb[1], rb[2], rb[3], rb[4], rb[5]);
        lvl[0] = 0;
        lvl[1] = 1;
    }
    __syncthreads();
    int level = 0;
    int* const lb = S.bins[w];
    for (int cur = 0;; cur ^= 1, level++) {
        const int nbig = S.nbig[cur], ntiny = S.ntiny[cur], items = nbig + (ntiny + 3) / 4;
        if (items == 0) break;
        for (;;) {
            int it = 0;
            if (lane == 0) it = atomicAdd(&S.next, 1);
            it = __builtin_amdgcn_readfirstlane(it);
            if (it >= items) break;
            if (it < nbig) sub_node(S, o, cur, it, lb, idxIn, ordered, leafFlag);
            else sub_tiny(S, o, cur, 4 * (it - nbig), ntiny, lb, idxIn, ordered, leafFlag);
            wave_lds_fence();
        }
        __syncthreads();
        if (tid == 0) { S.nbig[cur] = S.ntiny[cur] = 0; S.next = 0; lvl[level + 2] = (unsigned short)S.recs; }
        __syncthreads();
    }
    // collapse costs, bottom-up; levels [0, level] hold records
    const int total = S.recs;
    __syncthreads();
    float4* cst = (float4*)&S;
    static_assert(sizeof(SubLds<MAXQ>) >= (2 * kSmall - 1) * sizeof(float4), "collapse costs fit the LDS");
    float4* gc = b.cost + 2 * (size_t)g.s;
    for (int L = level; L >= 0; L--) {
        const int r0 = lvl[L], r1 = L == level ? total : lvl[L + 1];
        for (int k = r0 + tid; k < r1; k += kSubThreads) {
            const Rec& rc = rec[k];
            float4 c = leaf_cost();
            if (rc.child != kLeaf)
                c = node_cost(area(rc.a.x, rc.a.y, rc.a.z, rc.a.w, rc.b.x, rc.b.y), cst[rc.child], cst[rc.child + 1]);
            cst[k] = c;
            gc[k] = c;
        }
        __syncthreads();
    }
    if (tid == 0) {
        lvl[level + 1] = (unsigned short)total;
        b.smallCost[blockIdx.x] = cst[0];
        b.small[blockIdx.x].levels = level + 1;
    }
}

// ------------------------------- numbering and emission -----------------------
// depth: BVH4 levels, BVH2 levels
struct Emit { rt::Node2* n2; int* head; unsigned char* assign; int* depth; };

__device__ __forceinline__ void emit_node(const Emit& e, int p, const float (&bx)[6], int left, int right, int triStart,
                                          int triCount, bool head, int m) {
    rt::Node2 nd;
#pragma unroll
    for (int k = 0; k < 3; k++) { nd.box.mn[k] = bx[k]; nd.box.mx[k] = bx[3 + k]; }
    nd.left = left; nd.right = right; nd.triStart = triStart; nd.triCount = triCount;
    e.n2[p] = nd;
    e.head[p] = head ? 1 : 0;
    e.assign[p] = (unsigned char)m;
}

// The top nodes: costs bottom-up, then slots top-down and their BVH2 nodes
// (one workgroup; a few thousand nodes at most in a balanced tree).
__global__ __launch_bounds__(1024) void k_top_collapse(Build b, Emit e, int levels) {
    __shared__ int dmax;
    auto cost_of = [&](int ref) { return ref >= 0 ? b.topCost[ref] : b.smallCost[-1 - ref]; };
    if (threadIdx.x == 0) dmax = 0;
    for (int L = levels - 1; L >= 0; L--) {
        const int t0 = b.topLevel[L], t1 = b.topLevel[L + 1];
        for (int k = t0 + (int)threadIdx.x; k < t1; k += 1024) {
            const Top& t = b.top[k];
            b.topCost[k] = node_cost(area(t.box[0], t.box[1], t.box[2], t.box[3], t.box[4], t.box[5]), cost_of(t.left),
                                     cost_of(t.right));
        }
        __syncthreads();
    }
    auto set = [&](int ref, int2 a) { if (ref >= 0) b.topAsg[ref] = a; else b.smallAsg[-1 - ref] = a; };
    for (int k = threadIdx.x; k < b.numScenes; k += 1024) set(b.rootRef[k], make_int2(1, 0));
    __syncthreads();
    int depth = 0;
    for (int L = 0; L < levels; L++) {
        const int t0 = b.topLevel[L], t1 = b.topLevel[L + 1];
        for (int k = t0 + (int)threadIdx.x; k < t1; k += 1024) {
            const Top& t = b.top[k];
            const int2 a = b.topAsg[k];
            int2 al, ar;
            const bool head = assign_slots(b.topCost[k], cost_of(t.left), cost_of(t.right), a.x, a.y, al, ar);
            set(t.left, al);
            set(t.right, ar);
            const int p = pre_of(b, t.s, t.lt, t.tree);
            emit_node(e, p, t.box, p + 1, pre_of(b, t.m, t.lt, t.tree), 0, 0, head, a.x);
            if (head) depth = max(depth, a.y + 1);
        }
        __syncthreads();
    }
    atomicMax(&dmax, depth);
    __syncthreads();
    if (threadIdx.x == 0 && dmax) atomicMax(e.depth, dmax);
}

// A subtree's slots top-down and its BVH2 nodes.
__global__ __launch_bounds__(kThreads) void k_sub_emit(Build b, Emit e) {
    __shared__ unsigned int asg[2 * kSmall];      // slots | BVH4 level << 4
    __shared__ int dmax;
    const Small& sm = b.small[blockIdx.x];
    const Seg g = sm.g;
    const Rec* rec = b.rec + 2 * (size_t)g.s;
    const float4* cost = b.cost + 2 * (size_t)g.s;
    const unsigned short* lvl = b.lvl + 2 * (size_t)g.s;
    const int levels = sm.levels;
    if (threadIdx.x == 0) {
        const int2 a = b.smallAsg[blockIdx.x];
        asg[0] = (unsigned int)a.x | (unsigned int)a.y << 4;
        dmax = 0;
    }
    __syncthreads();
    int depth = 0;
    for (int L = 0; L < levels; L++) {
        const int r0 = lvl[L], r1 = lvl[L + 1];
        for (int k = r0 + (int)threadIdx.x; k < r1; k += kThreads) {
            const Rec rc = rec[k];
            const float bx[6] = {rc.a.x, rc.a.y, rc.a.z, rc.a.w, rc.b.x, rc.b.y};
            const int lt = g.lt + rc.lt, p = pre_of(b, g.s + rc.s, lt, g.tree);
            const int m = (int)(asg[k] & 15u), lev = (int)(asg[k] >> 4);
            if (rc.child == kLeaf) {
                emit_node(e, p, bx, 0, 0, g.s + rc.s, rc.m, false, m);
            } else {
                int2 al, ar;
                const bool head = assign_slots(cost[k], cost[rc.child], cost[rc.child + 1], m, lev, al, ar);
                asg[rc.child] = (unsigned int)al.x | (unsigned int)al.y << 4;
                asg[rc.child + 1] = (unsigned int)ar.x | (unsigned int)ar.y << 4;
                emit_node(e, p, bx, p + 1, pre_of(b, g.s + rc.m, lt, g.tree), 0, 0, head, m);
                if (head) depth = max(depth, lev + 1);
            }
        }
        __syncthreads();
    }
    if (depth) atomicMax(&dmax, depth);
    __syncthreads();
    if (threadIdx.x == 0) {
        atomicMax(&e.depth[0], dmax);
        atomicMax(&e.depth[1], sm.level + levels);
    }
}

// BVH4 root of each tree (a root is the head at its pre-order position).
__global__ void k_root4(Build b, const int* b4id, int* root4) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < b.numScenes) root4[s] = b4id[pre_of(b, b.off[s], 0, s)];
}

__device__ __forceinline__ uint16_t h_bits(_Float16 h) { return __builtin_bit_cast(uint16_t, h); }
__device__ __forceinline__ float h_val(uint16_t u) { return (float)__builtin_bit_cast(_Float16, u); }

// Largest half <= x / smallest half >= x: round to nearest even, then step
// once when the rounding went the wrong way (the host rule of the oracle).
__device__ __forceinline__ uint16_t f2h_down(float x) {
    uint16_t h = h_bits((_Float16)x);
    if (h_val(h) > x) {
        if ((h & 0x7fffu) == 0) h = 0x8001u;
        else if (h & 0x8000u) { if (h != 0xfc00u) h++; }
        else h--;
    }
    return h;
}
__device__ __forceinline__ uint16_t f2h_up(float x) {
    uint16_t h = h_bits((_Float16)x);
    if (h_val(h) < x) {
        if ((h & 0x7fffu) == 0) h = 0x0001u;
        else if (h & 0x8000u) h--;
        else if (h != 0x7c00u) h++;
    }
    return h;
}

__device__ __forceinline__ int32_t leaf_code(int first, int count) { return -((first << 3) | (count - 1)) - 2; }

// One BVH4 node per head (pre-order position p with head[p]); b4id[p] is the
// exclusive count of heads before p, i.e. the node's pre-order BVH4 index.
// Its slots are the nodes of assign 1 below it, reached through dissolved
// nodes (assign >= 2), left to right, so they stay in BVH2 pre-order.
__global__ void k_emit_bvh4(const rt::Node2* n2, const int* head, const int* b4id, const unsigned char* assign, int count,
                            uint4* out) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= count || !head[p]) return;
    const rt::Node2& nd = n2[p];
    int gather[4], ng = 0;
    int stk[4], sp = 0;
    stk[sp++] = nd.right;
    stk[sp++] = nd.left;
    while (sp > 0 && ng < 4) {
        const int q = stk[--sp];
        const rt::Node2& qn = n2[q];
        if (qn.triCount > 0 || assign[q] <= 1) { gather[ng++] = q; continue; }
        if (sp + 2 > 4) break;                  // unreachable: at most four slots
        stk[sp++] = qn.right;
        stk[sp++] = qn.left;
    }
    uint16_t hx[8], hy[8], hz[8];
    int32_t child[4];
    for (int i = 0; i < 4; i++) {
        if (i < ng) {
            const rt::Node2& g = n2[gather[i]];
            hx[i] = f2h_down(g.box.mn[0]); hx[4 + i] = f2h_up(g.box.mx[0]);
            hy[i] = f2h_down(g.box.mn[1]); hy[4 + i] = f2h_up(g.box.mx[1]);
            hz[i] = f2h_down(g.box.mn[2]); hz[4 + i] = f2h_up(g.box.mx[2]);
            child[i] = g.triCount > 0 ? leaf_code(g.triStart, g.triCount) : b4id[gather[i]];
        } else {
            hx[i] = hy[i] = hz[i] = 0x7c00u;
            hx[4 + i] = hy[4 + i] = hz[4 + i] = 0xfc00u;
            child[i] = -1;
        }
    }
    uint4* o = out + 4 * (size_t)b4id[p];
    o[0] = make_uint4(hx[0] | (uint32_t)hx[1] << 16, hx[2] | (uint32_t)hx[3] << 16, hx[4] | (uint32_t)hx[5] << 16,
                      hx[6] | (uint32_t)hx[7] << 16);
    o[1] = make_uint4(hy[0] | (uint32_t)hy[1] << 16, hy[2] | (uint32_t)hy[3] << 16, hy[4] | (uint32_t)hy[5] << 16,
                      hy[6] | (uint32_t)hy[7] << 16);
    o[2] = make_uint4(hz[0] | (uint32_t)hz[1] << 16, hz[2] | (uint32_t)hz[3] << 16, hz[4] | (uint32_t)hz[5] << 16,
                      hz[6] | (uint32_t)hz[7] << 16);
    o[3] = make_uint4((uint32_t)child[0], (uint32_t)child[1], (uint32_t)child[2], (uint32_t)child[3]);
}

// A tree whose root is a leaf (n <= maxLeaf): one BVH4 node with one slot.
__global__ void k_emit_leaf_root(const rt::Node2* n2, uint4* out) {
    const rt::Node2& r = n2[0];
    uint16_t h[3][8];
    for (int a = 0; a < 3; a++) {
        for (int i = 0; i < 4; i++) { h[a][i] = 0x7c00u; h[a][4 + i] = 0xfc00u; }
        h[a][0] = f2h_down(r.box.mn[a]);
        h[a][4] = f2h_up(r.box.mx[a]);
    }
    for (int a = 0; a < 3; a++)
        out[a] = make_uint4(h[a][0] | (uint32_t)h[a][1] << 16, h[a][2] | (uint32_t)h[a][3] << 16,
                            h[a][4] | (uint32_t)h[a][5] << 16, h[a][6] | (uint32_t)h[a][7] << 16);
    out[3] = make_uint4((uint32_t)leaf_code(r.triStart, r.triCount), 0xffffffffu, 0xffffffffu, 0xffffffffu);
}

// Leaf-order triangles {v0.xyz, bits(id)}, {v1.xyz, 0}, {v2.xyz, 0} and the
// inverse permutation.
// In a forest the id is the index within the triangle's scene.
__global__ void k_leaf_tris(const float* __restrict__ tris, const int* idx, int n, float4* out, int* leafOf,
                            const int* off, int numScenes) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int p = idx[i];
    const float* s = tris + 9 * (size_t)p;
    const int id = numScenes == 1 ? p : p - off[scene_of(off, numScenes, p)];
    out[3 * (size_t)i] = make_float4(s[0], s[1], s[2], __int_as_float(id));
    out[3 * (size_t)i + 1] = make_float4(s[3], s[4], s[5], 0.f);
    out[3 * (size_t)i + 2] = make_float4(s[6], s[7], s[8], 0.f);
    leafOf[p] = i;
}

// ------------------------------- scan ---------------------------------------
constexpr int kScanItems = 8;
constexpr int kScanTile = kThreads * kScanItems;

__global__ __launch_bounds__(kThreads) void k_tile_sums(const int* in, int n, int* tiles) {
    __shared__ int lds[kThreads / 64 + 1];
    const int base = blockIdx.x * kScanTile + threadIdx.x * kScanItems;
    int s = 0;
    for (int k = 0; k < kScanItems; k++) s += (base + k < n) ? in[base + k] : 0;
    int total;
    rts::block_exclusive_scan<kThreads>(s, lds, &total);
    if (threadIdx.x == 0) tiles[blockIdx.x] = total;
}

__global__ __launch_bounds__(1024) void k_scan_tile_sums(int* tiles, int nb, int* total) {
    __shared__ int lds[1024 / 64 + 1];
    int carry = 0;
    for (int base = 0; base < nb; base += 1024) {
        const int i = base + threadIdx.x;
        const int v = i < nb ? tiles[i] : 0;
        int tot;
        const int ex = rts::block_exclusive_scan<1024>(v, lds, &tot);
        if (i < nb) tiles[i] = carry + ex;
        carry += tot;
    }
    if (threadIdx.x == 0) *total = carry;
}

__global__ __launch_bounds__(kThreads) void k_tile_scan(const int* in, int n, const int* tiles, int* out) {
    __shared__ int lds[kThreads / 64 + 1];
    const int base = blockIdx.x * kScanTile + threadIdx.x * kScanItems;
    int v[kScanItems], s = 0;
    for (int k = 0; k < kScanItems; k++) { v[k] = (base + k < n) ? in[base + k] : 0; s += v[k]; }
    int total;
    int run = tiles[blockIdx.x] + rts::block_exclusive_scan<kThreads>(s, lds, &total);
    for (int k = 0; k < kScanItems; k++) {
        if (base + k < n) out[base + k] = run;
        run += v[k];
    }
}

// Triangle gather from device vertex / index buffers (one thread per
// triangle): corner k of triangle t is vertex idx[3t + k] (or 3t + k without
// an index buffer), three floats at byte offset index * stride. An index at or
// beyond numVertices sets *bad and writes zeros instead of reading.
__global__ void k_gather_tris(const uint8_t* verts, int numVertices, int stride, const void* idx, int indexBytes,
                              int numTris, float* out, int* bad) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= numTris) return;
    for (int k = 0; k < 3; k++) {
        const size_t c = 3 * (size_t)t + k;
        unsigned int v;
        if (indexBytes == 4) v = ((const uint32_t*)idx)[c];
        else if (indexBytes == 2) v = ((const uint16_t*)idx)[c];
        else v = (unsigned int)c;
        float x = 0.f, y = 0.f, z = 0.f;
        if (v < (unsigned int)numVertices) {
            const float* p = (const float*)(verts + (size_t)v * stride);
            x = p[0]; y = p[1]; z = p[2];
        } else {
            atomicOr(bad, 1);
        }
        out[9 * (size_t)t + 3 * k] = x;
        out[9 * (size_t)t + 3 * k + 1] = y;
        out[9 * (size_t)t + 3 * k + 2] = z;
    }
}

// One tree of a forest as a BVH of its own: BVH4 nodes [first, first+count)
// with inner children rebased by -first and leaf triangle starts by -triShift
// (trees and their leaf triangles lie one after another in a forest).
__global__ void k_slice_nodes4(const uint4* __restrict__ src, int first, int count, int triShift, uint4* dst) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    const uint4* a = src + 4 * (size_t)(first + i);
    uint4* o = dst + 4 * (size_t)i;
    o[0] = a[0]; o[1] = a[1]; o[2] = a[2];
    const uint4 c = a[3];
    uint32_t w[4] = {c.x, c.y, c.z, c.w};
    for (int k = 0; k < 4; k++) {
        const int v = (int)w[k];
        if (v >= 0) {
            w[k] = (uint32_t)(v - first);
        } else if (v < -1) {
            const int enc = -(v + 2);
            w[k] = (uint32_t)leaf_code((enc >> 3) - triShift, (enc & 7) + 1);
        }
    }
    o[3] = make_uint4(w[0], w[1], w[2], w[3]);
}

// dst[i] = src[i] - sub, i < n
__global__ void k_slice_sub(const int* __restrict__ src, int n, int sub, int* dst) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[i] - sub;
}

}  // namespace rtb

namespace rtk {
int launch_slice_forest(const void* nodes4, int first4, int count4, const void* tris, const int* leafOf, int t0,
                        int ntris, void* dNodes4, void* dTris, int* dLeafOf, hipStream_t s) {
    const int T = 256;
    hipLaunchKernelGGL(rtb::k_slice_nodes4, dim3((count4 + T - 1) / T), dim3(T), 0, s, (const uint4*)nodes4, first4,
                       count4, t0, (uint4*)dNodes4);
    hipLaunchKernelGGL(rtb::k_slice_sub, dim3((ntris + T - 1) / T), dim3(T), 0, s, leafOf + t0, ntris, t0, dLeafOf);
    hipMemcpyAsync(dTris, (const char*)tris + (size_t)t0 * 48, (size_t)ntris * 48, hipMemcpyDeviceToDevice, s);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) { rt::set_error("forest slice launch failed: %s", hipGetErrorString(e)); return -1; }
    return 0;
}

hipError_t launch_gather_tris(const void* verts, int numVertices, int stride, const void* idx, int indexBytes,
                              int numTris, float* out, int* bad, hipStream_t s) {
    hipLaunchKernelGGL(rtb::k_gather_tris, dim3((numTris + 255) / 256), dim3(256), 0, s, (const uint8_t*)verts,
                       numVertices, stride, idx, indexBytes, numTris, out, bad);
    return hipGetLastError();
}
}  // namespace rtk

namespace rt {

// Device-wide exclusive scan of n ints (out may not alias in); *total (device)
// receives the sum. tiles needs ceil(n / 2048) ints.
void scan_exclusive(const int* in, int* out, int n, int* total, int* tiles, hipStream_t s) {
    const int nb = (n + rtb::kScanTile - 1) / rtb::kScanTile;
    if (nb > 0) hipLaunchKernelGGL(rtb::k_tile_sums, dim3(nb), dim3(rtb::kThreads), 0, s, in, n, tiles);
    hipLaunchKernelGGL(rtb::k_scan_tile_sums, dim3(1), dim3(1024), 0, s, tiles, nb, total);
    if (nb > 0) hipLaunchKernelGGL(rtb::k_tile_scan, dim3(nb), dim3(rtb::kThreads), 0, s, in, n, tiles, out);
}

int scan_tiles_needed(int n) { return (n + rtb::kScanTile - 1) / rtb::kScanTile + 1; }

static double now_ms() {
    return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now().time_since_epoch()).count();
}

// One device allocation cut into pieces (the build needs some thirty arrays).
struct Slab {
    struct Piece { void** p; size_t bytes; };
    std::vector<Piece> want;
    void* base = nullptr;
    template <class T> void add(T** p, size_t count) {
        want.push_back({(void**)p, (std::max<size_t>(count, 1) * sizeof(T) + 255) & ~size_t(255)});
    }
    bool alloc() {
        size_t total = 0;
        for (const Piece& w : want) total += w.bytes;
        base = dev_alloc(total);
        if (!base) return false;
        char* c = (char*)base;
        for (const Piece& w : want) { *w.p = c; c += w.bytes; }
        return true;
    }
    bool idle = false;               // the build has waited for its last kernel
    ~Slab() { if (idle) dev_free(base); else dev_release(base); }
};

#define BUILD_CHECK(cond, msg)              \
    do {                                    \
        if (!(cond)) { set_error("%s", msg); return -1; } \
    } while (0)

// Builds the BVH on the device from d_tris (n x 9 floats, original order).
// Outputs (device, allocated here): nodes4 (numNodes4 x 64 B), leaf-order
// triangles (n x 48 B), leafOf (n ints), ordered (n ints, leaf order ->
// original index), nodes2 (pre-order rt::Node2). Returns 0 on success.
// With room for maxNodes top nodes and subtrees; full is set (and -1 returned)
// when they do not suffice.
static int build_with_room(const float* d_tris, int n, int maxLeaf, hipStream_t s, GpuBVH& out, const int* sceneOff,
                           int numScenes, std::vector<int>* roots4, size_t maxNodes, bool& full) {
    using namespace rtb;
    const double tBegin = verbose() ? now_ms() : 0.0;
    struct Report {
        double t0;
        ~Report() { if (verbose()) fprintf(stderr, "[CudaBVH] gpu_build: %.2f ms incl. workspace free\n", now_ms() - t0); }
    } report{tBegin};
    const int R = numScenes;
    // host tables: scene offsets, then chunks of kChunk primitives before each scene
    std::vector<int> tab(2 * (size_t)(R + 1));
    int* hOff = tab.data();
    int* hBase = tab.data() + R + 1;
    int largest = 0, big0 = 0;
    for (int k = 0; k <= R; k++) hOff[k] = sceneOff ? sceneOff[k] : k * n;
    hBase[0] = 0;
    for (int k = 0; k < R; k++) {
        const int c = hOff[k + 1] - hOff[k];
        if (c <= 0 || (R > 1 && c <= maxLeaf)) {
            set_error("gpu build: scene %d has %d primitives (a batch needs more than %d per scene)", k, c, maxLeaf);
            return -1;
        }
        largest = std::max(largest, c);
        big0 += c > kSmall;
        hBase[k + 1] = hBase[k] + (c + kChunk - 1) / kChunk;
    }
    const size_t N = (size_t)n;
    Build b{};
    b.n = n; b.maxLeaf = maxLeaf; b.numScenes = R;
    b.maxBig = n / (kSmall + 1) + 1;              // active nodes of one level
    const size_t maxChunks = N / kChunk + b.maxBig + 1;
    const size_t M = maxNodes;
    b.maxNodes = (int)M;
    Slab slab;
    int *dTab = nullptr, *tiles = nullptr, *head = nullptr, *b4id = nullptr, *dRoot4 = nullptr;
    unsigned char* assign = nullptr;
    float* dBounds = nullptr;
    slab.add(&dTab, 2 * (size_t)(R + 1));
    slab.add(&b.pbox, 2 * N);
    slab.add(&b.idx[0], N); slab.add(&b.idx[1], N);
    slab.add(&b.leafFlag, N); slab.add(&b.leafRank, N);
    slab.add(&b.rootAcc, 12 * (size_t)R); slab.add(&b.rootRef, R); slab.add(&b.bnd, 6 * (size_t)R);
    for (int k = 0; k < 2; k++) {
        slab.add(&b.act[k], b.maxBig); slab.add(&b.actAcc[k], 12 * (size_t)b.maxBig);
        slab.add(&b.chunkBase[k], b.maxBig + 1); slab.add(&b.bins[k], 2 * (size_t)b.maxBig * kSlotInts);
    }
    slab.add(&b.childAcc, 24 * (size_t)b.maxBig);
    slab.add(&b.sAxis, b.maxBig); slab.add(&b.sBin, b.maxBig); slab.add(&b.sNl, b.maxBig);
    slab.add(&b.chunkHist, maxChunks * kCells); slab.add(&b.chunkLeft, maxChunks);
    slab.add(&b.count, 8);
    slab.add(&b.topLevel, M + 2);                 // a level splits at least one node
    slab.add(&b.top, M); slab.add(&b.topCost, M); slab.add(&b.topAsg, M);
    slab.add(&b.small, M); slab.add(&b.smallCost, M); slab.add(&b.smallAsg, M);
    slab.add(&b.rec, 2 * N); slab.add(&b.cost, 2 * N); slab.add(&b.lvl, 2 * N + 2);
    slab.add(&head, 2 * N); slab.add(&assign, 2 * N); slab.add(&b4id, 2 * N);
    slab.add(&tiles, scan_tiles_needed((int)std::min<size_t>(2 * N, 0x7fffffff)) + 8);
    slab.add(&dRoot4, R);
    slab.add(&dBounds, 6 * (size_t)R);
    BUILD_CHECK(slab.alloc(), "gpu build: out of device memory");
    out.ordered = (int*)dev_alloc(N * 4);
    out.tris = dev_alloc(N * 48);
    out.leafOf = (int*)dev_alloc(N * 4);
    if (!out.ordered || !out.tris || !out.leafOf) {
        set_error("gpu build: out of device memory");
        return -1;
    }
    b.ordered = out.ordered;
    b.off = dTab; b.primBase = dTab + R + 1;
    if (hipMemcpyAsync(dTab, tab.data(), tab.size() * sizeof(int), hipMemcpyHostToDevice, s) != hipSuccess) {
        set_error("gpu build: upload failed");
        return -1;
    }
    const int T = kThreads;
    auto grid = [](long long items) { return dim3((unsigned)((items + kThreads - 1) / kThreads)); };
    const int slots0 = std::max(big0, 1);
    hipLaunchKernelGGL(k_build_init, grid(std::max(R * 12, slots0 * kSlotInts)), dim3(T), 0, s, b, slots0);
    hipLaunchKernelGGL(k_prims, dim3(hBase[R]), dim3(kTopThreads), 0, s, b, d_tris);
    hipLaunchKernelGGL(k_scene_bounds, grid(6 * (long long)R), dim3(T), 0, s, d_tris, b.bnd, 6 * R, dBounds);
    hipLaunchKernelGGL(k_top_next, dim3(1), dim3(1024), 0, s, b, 0, 1, 0);
    // Levels until no node of more than kSmall primitives is left. The
    // largest scene needs at least log2(c / kSmall) levels, so the first
    // read-back of the node count (a wait for the device) comes after those.
    int levels = 0, cur = 0;
    if (big0 > 0) {
        int need = 0;
        while (((long long)kSmall << need) < largest) need++;
        long long nodes = big0;
        for (;;) {
            const int gn = (int)std::min<long long>(nodes, b.maxBig);
            const int gc = (int)std::min<long long>((long long)(N / kChunk) + gn + 1, (long long)maxChunks);
            hipLaunchKernelGGL(k_top_bin, dim3(gc), dim3(kTopThreads), 0, s, b, cur);
            hipLaunchKernelGGL(k_top_split, dim3(gn), dim3(T), 0, s, b, cur, levels);
            hipLaunchKernelGGL(k_top_scatter, dim3(gc), dim3(kTopThreads), 0, s, b, cur);
            hipLaunchKernelGGL(k_top_next, dim3(1), dim3(1024), 0, s, b, cur ^ 1, 0, levels);
            cur ^= 1;
            levels++;
            nodes = std::min<long long>(2 * nodes, b.maxBig);
            if (levels < need) continue;
            int m = 0;
            if (hipMemcpyAsync(&m, b.count, 4, hipMemcpyDeviceToHost, s) != hipSuccess ||
                hipStreamSynchronize(s) != hipSuccess) {
                set_error("gpu build: level %d failed", levels - 1);
                return -1;
            }
            if (m == 0) break;
            nodes = m;
        }
    }
    int hc[8] = {0};
    if (hipMemcpyAsync(hc, b.count, sizeof hc, hipMemcpyDeviceToHost, s) != hipSuccess || hipStreamSynchronize(s) != hipSuccess) {
        set_error("gpu build: top levels failed");
        return -1;
    }
    if (hc[3]) {
        full = true;
        return -1;
    }
    const int numSmall = hc[2];
    // subtrees: narrow queues (more workgroups per CU) where the leaves hold four
    if (maxLeaf >= 4)
        hipLaunchKernelGGL((k_subtree<kSmall / 5 + 1>), dim3(numSmall), dim3(kSubThreads), 0, s, b);
    else
        hipLaunchKernelGGL((k_subtree<kSmall / 2 + 1>), dim3(numSmall), dim3(kSubThreads), 0, s, b);
    scan_exclusive(b.leafFlag, b.leafRank, n, b.count + 4, tiles, s);
    int leaves = 0;
    if (hipMemcpyAsync(&leaves, b.count + 4, 4, hipMemcpyDeviceToHost, s) != hipSuccess || hipStreamSynchronize(s) != hipSuccess) {
        set_error("gpu build: subtrees failed");
        return -1;
    }
    const int nodeCount = 2 * leaves - R;
    out.numNodes2 = nodeCount;
    if (leaves <= 0 || !(out.nodes2 = (Node2*)dev_alloc((size_t)nodeCount * sizeof(Node2)))) {
        set_error("gpu build: out of device memory");
        return -1;
    }
    const Emit em{out.nodes2, head, assign, b.count + 6};
    hipLaunchKernelGGL(k_top_collapse, dim3(1), dim3(1024), 0, s, b, em, levels);
    hipLaunchKernelGGL(k_sub_emit, dim3(numSmall), dim3(T), 0, s, b, em);
    scan_exclusive(head, b4id, nodeCount, b.count + 5, tiles, s);
    hipLaunchKernelGGL(k_leaf_tris, grid(n), dim3(T), 0, s, d_tris, b.ordered, n, (float4*)out.tris, out.leafOf, b.off, R);
    out.sceneBounds.resize(6 * (size_t)R);
    int fin[3] = {0, 0, 0};                       // heads, BVH4 and BVH2 levels
    if (hipMemcpyAsync(fin, b.count + 5, sizeof fin, hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipMemcpyAsync(out.sceneBounds.data(), dBounds, 24 * (size_t)R, hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess) {
        set_error("gpu build: numbering failed");
        return -1;
    }
    for (int a = 0; a < 3; a++) { out.bmin[a] = 1e30f; out.bmax[a] = -1e30f; }
    for (int k = 0; k < R; k++)
        for (int a = 0; a < 3; a++) {
            out.bmin[a] = std::min(out.bmin[a], out.sceneBounds[6 * (size_t)k + a]);
            out.bmax[a] = std::max(out.bmax[a], out.sceneBounds[6 * (size_t)k + 3 + a]);
        }
    const int heads = fin[0];
    out.numNodes4 = std::max(heads, 1);
    out.depth4 = std::max(fin[1], 1);             // a leaf root is one node
    if (!(out.nodes4 = dev_alloc((size_t)out.numNodes4 * 64))) {
        set_error("gpu build: out of device memory");
        return -1;
    }
    if (heads > 0)
        hipLaunchKernelGGL(k_emit_bvh4, grid(nodeCount), dim3(T), 0, s, out.nodes2, head, b4id, assign, nodeCount,
                           (uint4*)out.nodes4);
    else
        hipLaunchKernelGGL(k_emit_leaf_root, dim3(1), dim3(1), 0, s, out.nodes2, (uint4*)out.nodes4);
    if (roots4) {
        hipLaunchKernelGGL(k_root4, grid(R), dim3(T), 0, s, b, b4id, dRoot4);
        roots4->assign(R, 0);
        if (hipMemcpyAsync(roots4->data(), dRoot4, R * sizeof(int), hipMemcpyDeviceToHost, s) != hipSuccess) {
            set_error("gpu build: root download failed");
            return -1;
        }
    }
    hipError_t e = hipStreamSynchronize(s);
    if (e == hipSuccess) e = hipGetLastError();
    if (e != hipSuccess) { set_error("gpu build failed: %s", hipGetErrorString(e)); return -1; }
    out.levels = fin[2];
    slab.idle = true;
    return 0;
}

// The subtrees of a tree hold hundreds to 2048 primitives each; room for one
// per 128 is enough for all but trees that split off a few primitives at a
// time, level after level, and those start over with room for the worst case.
int gpu_build(const float* d_tris, int n, int maxLeaf, hipStream_t s, GpuBVH& out, const int* sceneOff,
              int numScenes, std::vector<int>* roots4) {
    const size_t N = (size_t)std::max(n, 1), room = std::min(N, N / 128 + 1024 + (size_t)numScenes);
    bool full = false;
    int rc = build_with_room(d_tris, n, maxLeaf, s, out, sceneOff, numScenes, roots4, room, full);
    if (rc != 0 && full) {
        for (void* p : {(void*)out.ordered, out.tris, (void*)out.leafOf}) dev_release(p);
        out = GpuBVH();
        full = false;
        rc = build_with_room(d_tris, n, maxLeaf, s, out, sceneOff, numScenes, roots4, N, full);
    }
    return rc;
}

}  // namespace rt
