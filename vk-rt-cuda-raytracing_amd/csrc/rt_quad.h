// rt_quad.h — BVH4 traversal with four lanes per ray.
//
// A lane that traces a ray alone spends some 120 instructions on a node visit
// (four slab tests and the ordering of their results) and twice 75 on a pair
// of triangles; where a launch has few rays left per wave, or few rays at all,
// the chain of those steps is its time. Here the four lanes of a quad take one
// child slot each of a node, or one triangle each of a leaf, so a step is
// about half as long and a leaf of four triangles one step, at the price of
// four lanes per ray. Each lane reads only its own slot: the entry and exit
// bound of its child per axis (2-byte loads whose address holds the ray's
// direction signs) and its child word, or the vertex components of its
// triangle already in the order of the ray's watertight axis permutation.
//
// In the one-level traversal node and triangle addresses are 32-bit offsets
// from the arrays' (uniform) bases, which keeps a lane's addresses in single
// registers: its callers use quads only where both arrays fit (fits()).
//
// Every value is computed by the expressions of rt_device.h, children are
// visited in the same order, and a ray's hit is the lexicographic minimum of
// (t, ID) over the triangles whose boxes pass, so results equal those of the
// one-lane traversal bit for bit. (The order matters for triangles at equal t
// whose boxes' entry rounds above it: the first one visited hides the others.)
#pragma once

#include <hip/hip_runtime.h>

#include "rt_device.h"

namespace rtq {

// Global memory: loads through a pointer that was itself loaded would
// otherwise be flat ones.
typedef const __attribute__((address_space(1))) char* gptr;
template <class T>
__device__ __forceinline__ T gload(gptr p) { return *(const __attribute__((address_space(1))) T*)p; }

inline bool fits(long long nodes, long long tris) { return nodes * 64 <= 0xffffffffll && tris * 48 <= 0xffffffffll; }

template <int CTRL>
__device__ __forceinline__ int quad_perm(int v) { return __builtin_amdgcn_update_dpp(v, v, CTRL, 0xf, 0xf, false); }
template <int CTRL>
__device__ __forceinline__ float quad_perm(float v) { return __int_as_float(quad_perm<CTRL>(__float_as_int(v))); }
constexpr int kXor1 = 0xb1, kXor2 = 0x4e, kMid = 0xd8;   // quad_perm [1,0,3,2], [2,3,0,1], [0,2,1,3]

// A ray held by the four lanes of a quad, in the axis order (x, y, z here) of
// its watertight test throughout: the slab test is the same in any order. t,
// u, v, id: this lane's closest candidate, at first the hit so far or (tmax,
// -1) in every lane; best: the quad's closest distance. tmax: any hit only.
struct Ray4 {
    float ox, oy, oz, ix, iy, iz, Sx, Sy, Sz, tmin, tmax;
    uint32_t kx, ky, kz;                              // the axes
    float t, u, v, best;
    int id;
    int ref, sp, col;                                 // node to visit next, stack entries, stack column
    float tn;
    bool found;
};

// Fills the ray part from a set-up ray (rtd::ray_setup).
__device__ __forceinline__ void set_ray(Ray4& q, const rtd::Ray& r) {
    q.ox = rtd::sel3(r.kx, r.ox, r.oy, r.oz);
    q.oy = rtd::sel3(r.ky, r.ox, r.oy, r.oz);
    q.oz = rtd::sel3(r.kz, r.ox, r.oy, r.oz);
    q.ix = rtd::sel3(r.kx, r.ix, r.iy, r.iz);
    q.iy = rtd::sel3(r.ky, r.ix, r.iy, r.iz);
    q.iz = rtd::sel3(r.kz, r.ix, r.iy, r.iz);
    q.Sx = r.Sx; q.Sy = r.Sy; q.Sz = r.Sz;
    q.tmin = r.tmin; q.tmax = r.tmax;
    q.kx = r.kx; q.ky = r.ky; q.kz = r.kz;
}

// Watertight test of the triangle (3 x float4) at tb + o, components addressed
// in the ray's axis order; the arithmetic of rtd::isect_watertight.
__device__ __forceinline__ bool isect(const Ray4& q, gptr tb, uint32_t o, float& t, float& u, float& v, int& id) {
    const uint32_t ox = o + 4u * q.kx, oy = o + 4u * q.ky, oz = o + 4u * q.kz;
    auto ld = [&](uint32_t off, int vertex) { return gload<float>(tb + off + 16 * vertex); };
    const float ax = ld(ox, 0), bx = ld(ox, 1), cx = ld(ox, 2);
    const float ay = ld(oy, 0), by = ld(oy, 1), cy = ld(oy, 2);
    const float az = ld(oz, 0), bz = ld(oz, 1), cz = ld(oz, 2);
    id = gload<int>(tb + o + 12);
    const float Akz = az - q.oz, Bkz = bz - q.oz, Ckz = cz - q.oz;
    const float Ax = (ax - q.ox) - q.Sx * Akz, Ay = (ay - q.oy) - q.Sy * Akz;
    const float Bx = (bx - q.ox) - q.Sx * Bkz, By = (by - q.oy) - q.Sy * Bkz;
    const float Cx = (cx - q.ox) - q.Sx * Ckz, Cy = (cy - q.oy) - q.Sy * Ckz;
    float U = Cx * By - Cy * Bx;
    float V = Ax * Cy - Ay * Cx;
    float W = Bx * Ay - By * Ax;
    if (U == 0.0f || V == 0.0f || W == 0.0f) {
        // one after the other, and fused (a product of two floats is exact in
        // 64 bits, so the bits are those of product and difference): fewer
        // registers at once
        U = (float)__builtin_fma(-(double)Cy, (double)Bx, (double)Cx * (double)By);
        __builtin_amdgcn_sched_barrier(0);
        V = (float)__builtin_fma(-(double)Ay, (double)Cx, (double)Ax * (double)Cy);
        __builtin_amdgcn_sched_barrier(0);
        W = (float)__builtin_fma(-(double)By, (double)Ax, (double)Bx * (double)Ay);
    }
    if ((U < 0.0f || V < 0.0f || W < 0.0f) && (U > 0.0f || V > 0.0f || W > 0.0f)) return false;
    const float det = U + V + W;
    if (det == 0.0f) return false;
    const float T = U * (q.Sz * Akz) + V * (q.Sz * Bkz) + W * (q.Sz * Ckz);
    const float rcp = 1.0f / det;
    t = T * rcp; u = V * rcp; v = W * rcp;
    return true;
}

// This lane's child of a node: the entry and exit bound per axis, in the ray's
// axis order, and the child word.
struct Slot { uint32_t hx, hy, hz, gx, gy, gz; int child; };

// Offsets in a node of a lane's bounds of entry (exit: bit 3 turned) and of
// its child word.
struct Offsets { uint32_t x, y, z, child; };

__device__ __forceinline__ Offsets offsets(const Ray4& q, int c) {
    auto entry = [&](float inv, uint32_t axis) { return 16u * axis + 2u * c + (__float_as_uint(inv) >> 31) * 8u; };
    return {entry(q.ix, q.kx), entry(q.iy, q.ky), entry(q.iz, q.kz), 48u + 4u * c};
}

// The slot of the node at nb + o (nb uniform): one 32-bit offset per load.
__device__ __forceinline__ Slot slot_at(gptr nb, uint32_t o, const Offsets& e) {
    auto half = [&](uint32_t off) { return (uint32_t)gload<uint16_t>(nb + off); };
    const uint32_t x = o + e.x, y = o + e.y, z = o + e.z;
    return {half(x), half(y), half(z), half(x ^ 8u), half(y ^ 8u), half(z ^ 8u), gload<int>(nb + (o + e.child))};
}

// The slot of the node at nb (different per quad): one 64-bit address per axis
// for both bounds, exchanged by the direction's sign.
__device__ __forceinline__ Slot slot_of(const Ray4& q, gptr nb, int c) {
    auto half = [&](gptr p) { return (uint32_t)gload<uint16_t>(p); };
    const gptr x = nb + (16u * q.kx + 2u * c), y = nb + (16u * q.ky + 2u * c), z = nb + (16u * q.kz + 2u * c);
    const uint32_t lx = half(x), ux = half(x + 8), ly = half(y), uy = half(y + 8), lz = half(z), uz = half(z + 8);
    const bool sx = __float_as_int(q.ix) < 0, sy = __float_as_int(q.iy) < 0, sz = __float_as_int(q.iz) < 0;
    return {sx ? ux : lx, sy ? uy : ly, sz ? uz : lz, sx ? lx : ux, sy ? ly : uy, sz ? lz : uz,
            gload<int>(nb + (48u + 4u * c))};
}

// One compare-exchange of the children's order: this lane keeps the smaller
// distance of its own and lane P's (low -INFINITY) or the larger one
// (INFINITY), and the child with it; equal ones stay.
template <int P>
__device__ __forceinline__ void exchange(float low, float& d, int& child) {
    const float m = __builtin_amdgcn_fmed3f(d, quad_perm<P>(d), low);
    const int other = quad_perm<P>(child);
    child = m != d ? other : child;
    d = m;
}

// Visits a node: this lane's child, then the quad's order of the hit ones. The
// nearest becomes q.ref, the others are pushed. False when no child is hit.
//
// The order is that of the one-lane visits' network (compare-exchanges 01, 23,
// 02, 13, 12 on the entry distances, misses at infinity), taken literally: it
// is not stable, and the order of boxes at equal distances decides between
// triangles at equal t (see above). Any hit may use any order.
//
// Of a flat ray (an infinite reciprocal) the distance to a plane through its
// origin is 0 * inf = NaN: such an axis bounds nothing, and the NaN-ignoring
// max / min leave it out, which is what rt_device.h's FLAT variant computes
// with its -inf / +inf. Where all three are NaN no box is hit: such a ray has
// no finite reciprocal, so its triangle tests give no finite t either.
template <bool ANY, class Push>
__device__ __forceinline__ bool visit(Ray4& q, int c, int sh, const Slot& s, int maxStack, int* status, Push&& push) {
    const float t1x = rtd::h_sub<false>(s.hx, q.ox) * q.ix, t2x = rtd::h_sub<false>(s.gx, q.ox) * q.ix;
    const float t1y = rtd::h_sub<false>(s.hy, q.oy) * q.iy, t2y = rtd::h_sub<false>(s.gy, q.oy) * q.iy;
    const float t1z = rtd::h_sub<false>(s.hz, q.oz) * q.iz, t2z = rtd::h_sub<false>(s.gz, q.oz) * q.iz;
    const float tN = fmaxf(fmaxf(t1x, t1y), t1z);
    const float tF = fminf(fminf(t2x, t2y), t2z) * RT_ROBUST_TFAR;
    const float limit = ANY ? q.tmax : q.best;
    const bool hit = (tN <= tF) && (tF >= q.tmin) && (tN <= limit) && s.child != -1;
    const uint32_t hm = (uint32_t)(__ballot(hit) >> sh) & 15u;
    if (!hm) return false;
    // Missed children sort last. (Opaque copies of c and the infinity: held
    // through the traversal, what is made of them would cost registers.)
    int lo = c, hi = c >> 1, inf = 0x7f800000;
    asm volatile("" : "+v"(lo), "+v"(hi), "+v"(inf));
    float d = __int_as_float(hit ? min(__float_as_int(tN), 0x7f7fffff) : inf);
    int child = s.child;
    const float low1 = __int_as_float((lo << 31) ^ (int)0xff800000), low2 = __int_as_float((hi << 31) ^ (int)0xff800000);
    exchange<kXor1>(low1, d, child);
    exchange<kXor2>(low2, d, child);
    exchange<kMid>(low2, d, child);
    // lane c holds the c-th of them
    const int n = __popc(hm);
    const int at = q.sp + n - 1 - c;
    if (c > 0 && c < n && at < maxStack) push(q, at, child, d);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // the quad's lanes read each other's entries
    q.sp += n - 1;
    if (q.sp > maxStack) { q.sp = maxStack; atomicOr(status, 1); }
    q.ref = quad_perm<0x00>(child);
    q.tn = quad_perm<0x00>(d);
    return true;
}

// Tests the cnt triangles from tb + o on, one per lane. closer(t, id): whether
// a hit replaces this lane's candidate. True when an any-hit ray is done.
template <bool ANY, class Closer>
__device__ __forceinline__ bool leaf(Ray4& q, int c, int sh, gptr tb, uint32_t o, int cnt, Closer&& closer) {
    bool hit = false;
    for (int b = 0; b < cnt; b += 4) {
        if (b + c < cnt) {
            float t, u, v;
            int id;
            if (isect(q, tb, o + 48u * (b + c), t, u, v, id) && t > q.tmin) {
                if (ANY) hit |= t < q.tmax;
                else if (closer(t, id)) { q.t = t; q.id = id; q.u = u; q.v = v; }
            }
        }
    }
    if (ANY) return ((__ballot(hit) >> sh) & 15u) != 0;
    const float m = fminf(q.t, quad_perm<kXor1>(q.t));
    q.best = fminf(m, quad_perm<kXor2>(m));
    return false;
}

// Traverses from q.ref (a node or a leaf code) until the ray is done. ANY:
// stops at the first hit (q.found). push(q, pos, ref, tn) and pop(q, pos,
// ref, tn) access entry pos < maxStack of the quad's stack; more entries (none
// in a tree of the depth that maxStack was made for) are dropped and flagged
// in *status. Control flow is the same in the four lanes of a quad. Returns
// the steps taken.
template <bool ANY, class Push, class Pop>
__device__ __forceinline__ int traverse(Ray4& q, int lane, const void* nodes, const void* tris, int maxStack, int* status,
                                        Push&& push, Pop&& pop) {
    const int c = lane & 3, sh = lane & 60;
    const Offsets e = offsets(q, c);
    int steps = 0;
    for (;;) {
        steps++;
        if (q.ref < 0) {
            if (ANY || q.tn <= q.best) {
                const int enc = -(q.ref + 2);
                if (leaf<ANY>(q, c, sh, (gptr)tris, (uint32_t)(enc >> 3) * 48u, (enc & 7) + 1, [&](float t, int id) {
                        return t < q.t || (t == q.t && id < q.id);
                    })) {
                    q.found = true;
                    break;
                }
            }
        } else if (ANY || q.tn <= q.best) {
            if (visit<ANY>(q, c, sh, slot_at((gptr)nodes, (uint32_t)q.ref << 6, e), maxStack, status, push)) continue;
        }
        if (q.sp == 0) break;
        q.sp--;
        pop(q, q.sp, q.ref, q.tn);
    }
    return steps;
}

// The quad's closest hit into every lane (ties: the lowest ID; no hit: id -1).
__device__ __forceinline__ void reduce(Ray4& q) {
#define RTQ_STEP(P)                                                                                                  \
    {                                                                                                                \
        const float t = quad_perm<P>(q.t), u = quad_perm<P>(q.u), v = quad_perm<P>(q.v);                             \
        const int id = quad_perm<P>(q.id);                                                                           \
        if (t < q.t || (t == q.t && (uint32_t)id < (uint32_t)q.id)) { q.t = t; q.u = u; q.v = v; q.id = id; }        \
    }
    RTQ_STEP(kXor1) RTQ_STEP(kXor2)
#undef RTQ_STEP
}

// Lane of the wave whose state quad k takes over: the k-th set bit of mask
// (at most 16 bits set; every lane calls it). -1 for quads beyond the last.
__device__ __forceinline__ int source_lane(uint64_t mask, int lane) {
    const int k = __popcll(mask & ((1ull << lane) - 1ull));
    const bool mine = (mask >> lane) & 1ull;
    // quad k's lane 0 receives the k-th live lane; the others send to lane 1
    const int got = __builtin_amdgcn_ds_permute(4 * (mine ? 4 * k : 1), lane);
    const int src = quad_perm<0x00>(got);
    return (lane >> 2) < __popcll(mask) ? src : -1;
}
__device__ __forceinline__ int take(int src, int v) { return __builtin_amdgcn_ds_bpermute(4 * src, v); }
__device__ __forceinline__ float take(int src, float v) { return __int_as_float(take(src, __float_as_int(v))); }

}  // namespace rtq
