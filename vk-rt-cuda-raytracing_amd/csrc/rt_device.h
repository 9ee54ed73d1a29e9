// rt_device.h — device-side ray/box/triangle arithmetic for gfx950.
//
// Every FP32 expression here is written in the exact operation order of the
// CPU oracle and compiled with -ffp-contract=off, IEEE division and square
// root and no denormal flushing, so hit IDs, t, u, v and visit counters are
// bit-identical to the oracle's on the same BVH and rays.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <float.h>

namespace rtd {

// 1 + 2*gamma(3) rounded to float: far-distance inflation of the robust slab
// test (T. Ize, "Robust BVH Ray Traversal", JCGT 2013).
#define RT_ROBUST_TFAR (1.0f + 3.0f * 0x1p-23f)
#define RT_MISS_T 1e30f

struct Ray {
    float ox, oy, oz, dx, dy, dz, tmin, tmax;
    float ix, iy, iz;          // 1/d, IEEE (infinite for a zero or tiny component)
    float Sx, Sy, Sz;          // watertight shear constants
    int kx, ky, kz;            // watertight axis permutation
};

// A ray with an infinite reciprocal component can meet (b - o) * inv =
// 0 * inf = NaN when its origin lies exactly on a box plane.
__device__ __forceinline__ bool ray_flat(const Ray& r) {
    return __builtin_isinf(r.ix) || __builtin_isinf(r.iy) || __builtin_isinf(r.iz);
}

__device__ __forceinline__ float sel3(int k, float a, float b, float c) {
    return k == 0 ? a : (k == 1 ? b : c);
}

// Per-ray set-up: reciprocal direction for the slab test, and the dominant
// axis / shear of the watertight test (Woop, Benthin, Wald, JCGT 2013).
__device__ __forceinline__ void ray_setup(Ray& r) {
    r.ix = 1.0f / r.dx;
    r.iy = 1.0f / r.dy;
    r.iz = 1.0f / r.dz;
    float ax = fabsf(r.dx), ay = fabsf(r.dy), az = fabsf(r.dz);
    int kz = 0;
    if (ay > ax) kz = 1;
    if (az > (kz == 0 ? ax : ay)) kz = 2;
    int kx = kz + 1; if (kx == 3) kx = 0;
    int ky = kx + 1; if (ky == 3) ky = 0;
    float dkz = sel3(kz, r.dx, r.dy, r.dz);
    if (dkz < 0.0f) { int t = kx; kx = ky; ky = t; }
    r.kx = kx; r.ky = ky; r.kz = kz;
    r.Sx = sel3(kx, r.dx, r.dy, r.dz) / dkz;
    r.Sy = sel3(ky, r.dx, r.dy, r.dz) / dkz;
    r.Sz = 1.0f / dkz;
}

// Component k of (a, b, c); K >= 0 fixes k at compile time.
template <int K>
__device__ __forceinline__ float pick(int k, float a, float b, float c) {
    if constexpr (K == 0) return a;
    else if constexpr (K == 1) return b;
    else if constexpr (K == 2) return c;
    else return sel3(k, a, b, c);
}

// Watertight ray-triangle test. Returns true with t, u (weight of v1) and v
// (weight of v2) when the ray's line crosses the triangle with a non-zero
// determinant; the caller applies (tmin, tmax) and the closest-hit rule.
// KX, KY, KZ >= 0 name the ray's axis permutation at compile time (the same
// arithmetic without the per-lane component selects); -1 reads it from r.
template <int KX = -1, int KY = -1, int KZ = -1>
__device__ __forceinline__ bool isect_watertight(const Ray& r, float4 p0, float4 p1, float4 p2,
                                                 float& t, float& u, float& v) {
    float A0 = p0.x - r.ox, A1 = p0.y - r.oy, A2 = p0.z - r.oz;
    float B0 = p1.x - r.ox, B1 = p1.y - r.oy, B2 = p1.z - r.oz;
    float C0 = p2.x - r.ox, C1 = p2.y - r.oy, C2 = p2.z - r.oz;
    float Akz = pick<KZ>(r.kz, A0, A1, A2), Bkz = pick<KZ>(r.kz, B0, B1, B2), Ckz = pick<KZ>(r.kz, C0, C1, C2);
    float Ax = pick<KX>(r.kx, A0, A1, A2) - r.Sx * Akz, Ay = pick<KY>(r.ky, A0, A1, A2) - r.Sy * Akz;
    float Bx = pick<KX>(r.kx, B0, B1, B2) - r.Sx * Bkz, By = pick<KY>(r.ky, B0, B1, B2) - r.Sy * Bkz;
    float Cx = pick<KX>(r.kx, C0, C1, C2) - r.Sx * Ckz, Cy = pick<KY>(r.ky, C0, C1, C2) - r.Sy * Ckz;
    float U = Cx * By - Cy * Bx;
    float V = Ax * Cy - Ay * Cx;
    float W = Bx * Ay - By * Ax;
    if (U == 0.0f || V == 0.0f || W == 0.0f) {   // FP64 fallback on an edge (paper, sec. 3.2)
        U = (float)((double)Cx * (double)By - (double)Cy * (double)Bx);
        V = (float)((double)Ax * (double)Cy - (double)Ay * (double)Cx);
        W = (float)((double)Bx * (double)Ay - (double)By * (double)Ax);
    }
    if ((U < 0.0f || V < 0.0f || W < 0.0f) && (U > 0.0f || V > 0.0f || W > 0.0f)) return false;
    float det = U + V + W;
    if (det == 0.0f) return false;
    float Az = r.Sz * Akz, Bz = r.Sz * Bkz, Cz = r.Sz * Ckz;
    float T = U * Az + V * Bz + W * Cz;
    float rcp = 1.0f / det;
    t = T * rcp; u = V * rcp; v = W * rcp;
    return true;
}

// Axis permutation of the watertight test as one code 0-5: 2 * kz, plus 1
// when kx and ky are exchanged (negative direction along kz).
__device__ __forceinline__ int perm_code(const Ray& r) {
    return 2 * r.kz + (r.kx == (r.kz == 2 ? 0 : r.kz + 1) ? 0 : 1);
}

// Wave-uniform permutation code of a wave's live lanes (-1 when they
// differ). Every lane of the wave must call it; dead lanes do not vote.
__device__ __forceinline__ int wave_perm(const Ray& r, bool live) {
    const int mine = live ? perm_code(r) : -1;
    const uint64_t lm = __ballot(live);
    const int lead = lm ? (int)__builtin_ctzll(lm) : 0;
    const int p = __builtin_amdgcn_readlane(mine, lead);
    return __all(!live || mine == p) ? p : -1;
}

// Watertight test with the permutation fixed when the wave shares one
// (pc >= 0, wave-uniform), so that the branch is taken by the whole wave.
__device__ __forceinline__ bool isect_watertight_wave(const Ray& r, int pc, float4 p0, float4 p1, float4 p2,
                                                      float& t, float& u, float& v) {
    switch (pc) {
    case 0: return isect_watertight<1, 2, 0>(r, p0, p1, p2, t, u, v);
    case 1: return isect_watertight<2, 1, 0>(r, p0, p1, p2, t, u, v);
    case 2: return isect_watertight<2, 0, 1>(r, p0, p1, p2, t, u, v);
    case 3: return isect_watertight<0, 2, 1>(r, p0, p1, p2, t, u, v);
    case 4: return isect_watertight<0, 1, 2>(r, p0, p1, p2, t, u, v);
    case 5: return isect_watertight<1, 0, 2>(r, p0, p1, p2, t, u, v);
    default: return isect_watertight(r, p0, p1, p2, t, u, v);
    }
}

// Moller-Trumbore with the reference's thresholds (layer/cuda_bvh_backend.cu
// :145-156), IEEE division in place of the fast-math reciprocal.
__device__ __forceinline__ bool isect_mt(const Ray& r, float4 p0, float4 p1, float4 p2,
                                         float& t, float& u, float& v) {
    float e1x = p1.x - p0.x, e1y = p1.y - p0.y, e1z = p1.z - p0.z;
    float e2x = p2.x - p0.x, e2y = p2.y - p0.y, e2z = p2.z - p0.z;
    float ppx = r.dy * e2z - r.dz * e2y, ppy = r.dz * e2x - r.dx * e2z, ppz = r.dx * e2y - r.dy * e2x;
    float det = e1x * ppx + e1y * ppy + e1z * ppz;
    if (fabsf(det) < 1e-12f) return false;
    float inv = 1.f / det;
    float tx = r.ox - p0.x, ty = r.oy - p0.y, tz = r.oz - p0.z;
    float uu = inv * (tx * ppx + ty * ppy + tz * ppz);
    if (uu < 0.f || uu > 1.f) return false;
    float qx = ty * e1z - tz * e1y, qy = tz * e1x - tx * e1z, qz = tx * e1y - ty * e1x;
    float vv = inv * (r.dx * qx + r.dy * qy + r.dz * qz);
    if (vv < 0.f || uu + vv > 1.f) return false;
    t = inv * (e2x * qx + e2y * qy + e2z * qz); u = uu; v = vv;
    return true;
}

template <bool MT>
__device__ __forceinline__ bool isect(const Ray& r, float4 p0, float4 p1, float4 p2, float& t, float& u, float& v) {
    if constexpr (MT) return isect_mt(r, p0, p1, p2, t, u, v);
    else return isect_watertight(r, p0, p1, p2, t, u, v);
}

__device__ __forceinline__ float h_lo(uint32_t w) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)(w & 0xffffu));
}
__device__ __forceinline__ float h_hi(uint32_t w) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)(w >> 16));
}

// RN(h - o) for the FP16 value h in the low (HI = false) or high half of w,
// in one v_fma_mix_f32: h * 1.0 - o with h widened exactly and one rounding,
// which is the value of (float)h - o. Saves the separate conversion.
template <bool HI>
__device__ __forceinline__ float h_sub(uint32_t w, float o) {
    float r;
    if constexpr (HI) asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(w), "v"(o));
    else asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(w), "v"(o));
    return r;
}

// Bounds words of a 64-byte BVH4 node (x, y, z halves; per axis the mins of
// slots 0-3, then the maxes) as one traversal variant reads them. FLAT
// (chosen per wave when any lane's ray is flat) keeps the stored order and
// takes per-axis min / max of the two plane distances. The other variant
// exchanges the min and max words of every axis whose direction is negative,
// so that the first half holds the entry planes and the second the exit
// planes: with lo <= hi (outward rounding) and a finite non-zero reciprocal,
// (lo - o) * i <= (hi - o) * i when i > 0 and >= when i < 0, so the entry and
// exit distances are the per-axis min and max without computing them.
template <bool FLAT>
struct NodeBox { uint4 x, y, z; };

// The exchange is a bitwise select (one v_bfi_b32 per word) under an
// all-ones / all-zeros mask taken from the reciprocal's sign bit: written as
// a conditional, the compiler turns it into loads from selected addresses or
// into branches.
__device__ __forceinline__ uint4 orient(const uint4& q, float inv) {
    const uint32_t m = (uint32_t)(__float_as_int(inv) >> 31);
    return make_uint4((q.z & m) | (q.x & ~m), (q.w & m) | (q.y & ~m), (q.x & m) | (q.z & ~m), (q.y & m) | (q.w & ~m));
}

template <bool FLAT>
__device__ __forceinline__ NodeBox<FLAT> node_box(const Ray& r, const uint4& qx, const uint4& qy, const uint4& qz) {
    if constexpr (FLAT) return NodeBox<FLAT>{qx, qy, qz};
    else return NodeBox<FLAT>{orient(qx, r.ix), orient(qy, r.iy), orient(qz, r.iz)};
}

// Slab test of child slot C. Robust far distance. FLAT resolves the 0*inf
// NaN so that a parallel axis whose plane holds the origin does not constrain
// the interval; for other rays both variants give the same entry distance and
// the same answer. True when the box may hold a hit in [tmin, limit].
template <int C, bool FLAT>
__device__ __forceinline__ bool slab_child(const Ray& r, const NodeBox<FLAT>& b, float limit, float& tnear) {
    const uint32_t wxl = (C < 2) ? b.x.x : b.x.y, wxh = (C < 2) ? b.x.z : b.x.w;
    const uint32_t wyl = (C < 2) ? b.y.x : b.y.y, wyh = (C < 2) ? b.y.z : b.y.w;
    const uint32_t wzl = (C < 2) ? b.z.x : b.z.y, wzh = (C < 2) ? b.z.z : b.z.w;
    constexpr bool HI = (C & 1) != 0;
    float t1x = h_sub<HI>(wxl, r.ox) * r.ix, t2x = h_sub<HI>(wxh, r.ox) * r.ix;
    float t1y = h_sub<HI>(wyl, r.oy) * r.iy, t2y = h_sub<HI>(wyh, r.oy) * r.iy;
    float t1z = h_sub<HI>(wzl, r.oz) * r.iz, t2z = h_sub<HI>(wzh, r.oz) * r.iz;
    float tN, tF;
    if constexpr (FLAT) {
        t1x = t1x != t1x ? -r.ix : t1x; t2x = t2x != t2x ? r.ix : t2x;
        t1y = t1y != t1y ? -r.iy : t1y; t2y = t2y != t2y ? r.iy : t2y;
        t1z = t1z != t1z ? -r.iz : t1z; t2z = t2z != t2z ? r.iz : t2z;
        tN = fmaxf(fmaxf(fminf(t1x, t2x), fminf(t1y, t2y)), fminf(t1z, t2z));
        tF = fminf(fminf(fmaxf(t1x, t2x), fmaxf(t1y, t2y)), fmaxf(t1z, t2z)) * RT_ROBUST_TFAR;
    } else {
        tN = fmaxf(fmaxf(t1x, t1y), t1z);
        tF = fminf(fminf(t2x, t2y), t2z) * RT_ROBUST_TFAR;
    }
    tnear = tN;
    return (tN <= tF) && (tF >= r.tmin) && (tN <= limit);
}

// Slot C of a node: true, with the entry distance, when the slot holds a
// child (ref != -1) whose box passes the slab test. The slab test runs for
// empty slots too, so the four slots of a node are tested without branches.
// An empty slot stores the box (+inf, -inf): the FLAT variant's min / max
// turn it into the whole line, so its result is discarded by ref; in the
// other variant it reads entry +inf and exit -inf and misses by itself.
template <int C, bool FLAT>
__device__ __forceinline__ bool child_hit(const Ray& r, const NodeBox<FLAT>& b, int ref, float limit, float& tnear) {
    const bool h = slab_child<C, FLAT>(r, b, limit, tnear);
    if constexpr (FLAT) return h & (ref != -1);
    else return h;
}

// Pinhole ray for pixel (px, py) of a W x H image; the same sequence as the
// oracle's generator: sx = ((px+0.5)/W)*2-1, d = f + (sx*sX)*r + (sy*sY)*u,
// d *= 1/sqrt(d.d).
struct Cam { float o[3], f[3], r[3], u[3], sx, sy; };

__device__ __forceinline__ void pinhole_ray(const Cam& c, int px, int py, int W, int H, Ray& r) {
    float sx = ((float)px + 0.5f) / (float)W * 2.0f - 1.0f;
    float sy = ((float)py + 0.5f) / (float)H * 2.0f - 1.0f;
    float a = sx * c.sx, b = sy * c.sy;
    float dx = (c.f[0] + a * c.r[0]) + b * c.u[0];
    float dy = (c.f[1] + a * c.r[1]) + b * c.u[1];
    float dz = (c.f[2] + a * c.r[2]) + b * c.u[2];
    float inv = 1.0f / sqrtf((dx * dx + dy * dy) + dz * dz);
    r.ox = c.o[0]; r.oy = c.o[1]; r.oz = c.o[2];
    r.dx = dx * inv; r.dy = dy * inv; r.dz = dz * inv;
    r.tmin = 0.0f; r.tmax = RT_MISS_T;
}

// Pixel of slot i when a W x H image is walked tile by tile: the complete
// 8x8 pixel tiles first, 64 consecutive slots per tile (row-major inside),
// tiles in vertical strips 8 tiles (64 pixels) wide and row-major inside a
// strip, strips left to right; then the pixels of the right and bottom
// margins that no complete tile covers, row-major. A bijection on [0, W*H).
// Work taken in slot order then stays in compact image blocks, which keeps
// neighbouring rays on one XCD's L2.
__device__ __forceinline__ int tile_strip_pixel(int i, int W, int H) {
    const int tx8 = W >> 3, ty8 = H >> 3, inTiles = tx8 * ty8 * 64;
    if (i < inTiles) {
        const int tile = i >> 6, k = i & 63;
        const int full = tx8 / 8, per = 8 * ty8;
        int strip = tile / per, r = tile - strip * per, w = 8;
        if (strip >= full) { strip = full; r = tile - full * per; w = tx8 - full * 8; }
        const int ty = r / w, tx = strip * 8 + (r - ty * w);
        return (ty * 8 + (k >> 3)) * W + tx * 8 + (k & 7);
    }
    int j = i - inTiles;
    const int rw = W - tx8 * 8, H8 = ty8 * 8;
    if (j < H8 * rw) {
        const int y = j / rw;
        return y * W + tx8 * 8 + (j - y * rw);
    }
    j -= H8 * rw;
    return (H8 + j / W) * W + j % W;
}

// 16-byte loads through the global address space. A pointer chosen at run
// time between arrays the compiler cannot trace to global memory (the TLAS
// or an instance's BLAS, read from a descriptor) otherwise turns its loads
// into generic flat loads, whose waits also cover every pending LDS access.
typedef unsigned rt_v4u __attribute__((ext_vector_type(4)));
typedef float rt_v4f __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint4 ldg_u4(const uint4* p) {
    const rt_v4u v = *(const __attribute__((address_space(1))) rt_v4u*)p;
    return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ float4 ldg_f4(const float4* p) {
    const rt_v4f v = *(const __attribute__((address_space(1))) rt_v4f*)p;
    return make_float4(v.x, v.y, v.z, v.w);
}

// Node visit of the uncounted traversals, in the counted ones' order: the
// nearest hit child (closest hit) or the last one (any hit, slot order) is
// taken next (ref, tn), the others go on the stack, nearest on top. Returns
// false when no child is hit. The stack is LDS slots [0, LDSD) of this
// thread's column, beyond them push(ref, tn).
//
// The stack entries are written without branches: three slots whatever the
// number of hit children; what lies above the new top is garbage that the next
// push overwrites. (A branch per push was a fifth of the visit's instructions:
// 23 M incoherent rays 5.05 to 4.97 ms, cost-ordered 1080p primaries 373 to
// 362 us.) Any-hit entries have no distance.
template <bool ANY, bool FLAT, int LDSD, int BLOCK, class Push>
__device__ __forceinline__ bool visit_free(const Ray& r, uint4 nx, uint4 ny, uint4 nz, uint4 qc, float limit, int& ref,
                                           float& tn, int* s_ref, float* s_tn, int tid, int& sp, Push&& push) {
    const NodeBox<FLAT> b = node_box<FLAT>(r, nx, ny, nz);
    float d[4];
    int c[4] = {(int)qc.x, (int)qc.y, (int)qc.z, (int)qc.w};
    // a hit's distance stays below the missed children's, so that these sort last
    if (!ANY) limit = fminf(limit, 3.402823466e38f);
    const bool h0 = child_hit<0, FLAT>(r, b, c[0], limit, d[0]);
    const bool h1 = child_hit<1, FLAT>(r, b, c[1], limit, d[1]);
    const bool h2 = child_hit<2, FLAT>(r, b, c[2], limit, d[2]);
    const bool h3 = child_hit<3, FLAT>(r, b, c[3], limit, d[3]);
    const int n = (int)h0 + (int)h1 + (int)h2 + (int)h3;
    if (n == 0) return false;
    if constexpr (ANY) {
        if (sp + 3 <= LDSD) {
            int p = sp * BLOCK + tid;
            s_ref[p] = c[0]; p += h0 ? BLOCK : 0;
            s_ref[p] = c[1]; p += h1 ? BLOCK : 0;
            s_ref[p] = c[2];
            sp += n - 1;
            ref = h3 ? c[3] : h2 ? c[2] : h1 ? c[1] : c[0];
        } else {
            int nxt = -1;
            if (h0) nxt = c[0];
            if (h1) { if (nxt != -1) push(nxt, 0.f); nxt = c[1]; }
            if (h2) { if (nxt != -1) push(nxt, 0.f); nxt = c[2]; }
            if (h3) { if (nxt != -1) push(nxt, 0.f); nxt = c[3]; }
            ref = nxt;
        }
        tn = 0.f;
    } else {
        d[0] = h0 ? d[0] : INFINITY;
        d[1] = h1 ? d[1] : INFINITY;
        d[2] = h2 ? d[2] : INFINITY;
        d[3] = h3 ? d[3] : INFINITY;
#define RTD_CSWAP(i, j)                                                                 \
    {                                                                                   \
        const bool s = d[i] > d[j];                                                     \
        const float di = d[i], dj = d[j];                                               \
        const int ci = c[i], cj = c[j];                                                 \
        d[i] = s ? dj : di; d[j] = s ? di : dj; c[i] = s ? cj : ci; c[j] = s ? ci : cj; \
    }
        RTD_CSWAP(0, 1) RTD_CSWAP(2, 3) RTD_CSWAP(0, 2) RTD_CSWAP(1, 3) RTD_CSWAP(1, 2)
#undef RTD_CSWAP
        if (sp + 3 <= LDSD) {
            // farthest first: c[n - 1] .. c[1]
            const int p = sp * BLOCK + tid;
            s_ref[p] = n == 4 ? c[3] : n == 3 ? c[2] : c[1];
            s_tn[p] = n == 4 ? d[3] : n == 3 ? d[2] : d[1];
            s_ref[p + BLOCK] = n == 4 ? c[2] : c[1];
            s_tn[p + BLOCK] = n == 4 ? d[2] : d[1];
            s_ref[p + 2 * BLOCK] = c[1];
            s_tn[p + 2 * BLOCK] = d[1];
            sp += n - 1;
        } else {
            if (n > 3) push(c[3], d[3]);
            if (n > 2) push(c[2], d[2]);
            if (n > 1) push(c[1], d[1]);
        }
        ref = c[0];
        tn = d[0];
    }
    return true;
}

// Work distribution of the persistent traversal kernels. Work items [0, n)
// (rays, or 64 per 8x8 pinhole tile) are taken in 64-item chunks, and the
// chunks are split into kBands contiguous bands, one per XCD: the dispatcher
// places workgroups on the eight XCDs round robin, so blockIdx.x % 8 names
// the XCD a wave runs on, and each wave starts on its own XCD's band. Nearby
// pixels (or rays queued together) then share one XCD's L2 instead of being
// spread over all eight. A wave whose band is used up moves on to the next
// band, so no XCD idles while another still has work. ctr holds kBands
// counters of chunks taken, kBandStride words apart, zeroed before the
// launch; band is the wave's current band (wave-uniform). Returns the first
// item of the chunk, or n when every band is used up.
//
// Each counter has a 128-byte cache line of its own: eight counters packed
// into one line made every trace about twice as slow as a single counter,
// while one line per counter makes the banded order 12-20 % faster than the
// single counter's row-major order on the 1080p terrain frame.
constexpr int kBands = 8;
constexpr int kBandStride = 32;

// Maximum of v over the 64 lanes of a wave (every lane active).
__device__ __forceinline__ int wave_max(int v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
    return v;
}

__device__ __forceinline__ int take_chunk(uint32_t* ctr, int n, int& band) {
    const int nc = (n + 63) >> 6;
    for (int k = 0; k < kBands; ++k) {
        const int b = (band + k) & (kBands - 1);
        const int lo = (int)(((long long)nc * b) / kBands);
        const int hi = (int)(((long long)nc * (b + 1)) / kBands);
        if (lo >= hi) continue;
        uint32_t t = 0;
        if ((threadIdx.x & 63) == 0) t = atomicAdd(&ctr[b * kBandStride], 1u);
        t = (uint32_t)__builtin_amdgcn_readfirstlane((int)t);
        if ((long long)lo + t < hi) {
            band = b;
            return (lo + (int)t) << 6;
        }
    }
    return n;
}

}  // namespace rtd
