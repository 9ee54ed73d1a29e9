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
// Node and triangle addresses are 32-bit offsets from the arrays' (uniform)
// bases, which keeps a lane's addresses in single registers: the caller uses
// quads only where both arrays fit (fits()).
//
// Every value is computed by the expressions of rt_device.h, and a ray's hit
// is the lexicographic minimum of (t, ID) over the triangles whose boxes pass,
// in any visiting order, so results equal those of the one-lane traversal bit
// for bit.
#pragma once

#include <hip/hip_runtime.h>

#include "rt_device.h"

namespace rtq {

inline bool fits(long long nodes, long long tris) { return nodes * 64 <= 0xffffffffll && tris * 48 <= 0xffffffffll; }

template <int CTRL>
__device__ __forceinline__ int quad_perm(int v) { return __builtin_amdgcn_update_dpp(v, v, CTRL, 0xf, 0xf, false); }
template <int CTRL>
__device__ __forceinline__ float quad_perm(float v) { return __int_as_float(quad_perm<CTRL>(__float_as_int(v))); }
constexpr int kXor1 = 0xb1, kXor2 = 0x4e;             // quad_perm [1,0,3,2], [2,3,0,1]
constexpr int kRot1 = 0x39, kRot2 = 0x4e, kRot3 = 0x93;   // lane c reads lane (c + k) & 3

// A ray held by the four lanes of a quad. t, u, v, id: this lane's own closest
// candidate; best: the quad's closest distance.
struct Ray4 {
    float ox, oy, oz, ix, iy, iz;
    float okx, oky, okz, Sx, Sy, Sz, tmin, tmax;      // permuted origin, shear
    uint32_t kxo, kyo, kzo;                           // byte offsets of the permuted components
    float t, u, v, best;
    int id;
    int ref, sp, col;                                 // node to visit next, stack entries, stack column
    float tn;
    bool found;
};

// Fills the ray part from a set-up ray (rtd::ray_setup).
__device__ __forceinline__ void set_ray(Ray4& q, const rtd::Ray& r) {
    q.ox = r.ox; q.oy = r.oy; q.oz = r.oz;
    q.ix = r.ix; q.iy = r.iy; q.iz = r.iz;
    q.Sx = r.Sx; q.Sy = r.Sy; q.Sz = r.Sz;
    q.tmin = r.tmin; q.tmax = r.tmax;
    q.okx = rtd::sel3(r.kx, r.ox, r.oy, r.oz);
    q.oky = rtd::sel3(r.ky, r.ox, r.oy, r.oz);
    q.okz = rtd::sel3(r.kz, r.ox, r.oy, r.oz);
    q.kxo = 4u * r.kx; q.kyo = 4u * r.ky; q.kzo = 4u * r.kz;
}

// Watertight test of triangle ti (3 x float4), components addressed in the
// ray's axis order; the arithmetic of rtd::isect_watertight.
__device__ __forceinline__ bool isect(const Ray4& q, const void* tris, int ti, float& t, float& u, float& v, int& id) {
    const char* tb = (const char*)tris;
    const uint32_t o = (uint32_t)ti * 48u, ox = o + q.kxo, oy = o + q.kyo, oz = o + q.kzo;
    auto ld = [&](uint32_t off, int vertex) { return *(const float*)(tb + off + 16 * vertex); };
    const float ax = ld(ox, 0), bx = ld(ox, 1), cx = ld(ox, 2);
    const float ay = ld(oy, 0), by = ld(oy, 1), cy = ld(oy, 2);
    const float az = ld(oz, 0), bz = ld(oz, 1), cz = ld(oz, 2);
    id = *(const int*)(tb + o + 12);
    const float Akz = az - q.okz, Bkz = bz - q.okz, Ckz = cz - q.okz;
    const float Ax = (ax - q.okx) - q.Sx * Akz, Ay = (ay - q.oky) - q.Sy * Akz;
    const float Bx = (bx - q.okx) - q.Sx * Bkz, By = (by - q.oky) - q.Sy * Bkz;
    const float Cx = (cx - q.okx) - q.Sx * Ckz, Cy = (cy - q.oky) - q.Sy * Ckz;
    float U = Cx * By - Cy * Bx;
    float V = Ax * Cy - Ay * Cx;
    float W = Bx * Ay - By * Ax;
    if (U == 0.0f || V == 0.0f || W == 0.0f) {         // one after the other: fewer registers at once
        U = (float)((double)Cx * (double)By - (double)Cy * (double)Bx);
        __builtin_amdgcn_sched_barrier(0);
        V = (float)((double)Ax * (double)Cy - (double)Ay * (double)Cx);
        __builtin_amdgcn_sched_barrier(0);
        W = (float)((double)Bx * (double)Ay - (double)By * (double)Ax);
    }
    if ((U < 0.0f || V < 0.0f || W < 0.0f) && (U > 0.0f || V > 0.0f || W > 0.0f)) return false;
    const float det = U + V + W;
    if (det == 0.0f) return false;
    const float T = U * (q.Sz * Akz) + V * (q.Sz * Bkz) + W * (q.Sz * Ckz);
    const float rcp = 1.0f / det;
    t = T * rcp; u = V * rcp; v = W * rcp;
    return true;
}

// Traverses from q.ref (a node or a leaf code) until the ray is done. ANY:
// stops at the first hit (q.found). FLAT: the slab variant for rays with an
// infinite reciprocal (chosen per wave). push(q, pos, ref, tn) and pop(q, pos,
// ref, tn) access entry pos < maxStack of the quad's stack; more entries (none
// in a tree of the depth that maxStack was made for) are dropped and flagged
// in *status. Control flow is the same in the four lanes of a quad. Returns
// the steps taken.
template <bool ANY, bool FLAT, class Push, class Pop>
__device__ __forceinline__ int traverse(Ray4& q, int lane, const void* nodes, const void* tris, int maxStack, int* status,
                                        Push&& push, Pop&& pop) {
    const int c = lane & 3, sh = lane & 60;
    const char* nb = (const char*)nodes;
    // offsets in a node of this lane's entry and exit bound per axis
    auto entry = [&](float inv, int axis) {
        return 16u * axis + 2u * c + (FLAT ? 0u : (__float_as_uint(inv) >> 31) * 8u);
    };
    const uint32_t eX = entry(q.ix, 0), eY = entry(q.iy, 1), eZ = entry(q.iz, 2), eC = 48u + 4u * c;
    auto half = [&](uint32_t off) { return (uint32_t)*(const uint16_t*)(nb + off); };
    int steps = 0;
    for (;;) {
        steps++;
        if (q.ref < 0) {
            if (ANY || q.tn <= q.best) {
                const int enc = -(q.ref + 2), ts = enc >> 3, cnt = (enc & 7) + 1;
                bool hit = false;
                for (int b = 0; b < cnt; b += 4) {
                    if (b + c < cnt) {
                        float t, u, v;
                        int id;
                        if (isect(q, tris, ts + b + c, t, u, v, id) && t > q.tmin && t < q.tmax) {
                            if (ANY) hit = true;
                            else if (t < q.t || (t == q.t && id < q.id)) { q.t = t; q.id = id; q.u = u; q.v = v; }
                        }
                    }
                }
                if (ANY) {
                    if ((__ballot(hit) >> sh) & 15u) { q.found = true; break; }
                } else {
                    float m = fminf(q.t, quad_perm<kXor1>(q.t));
                    q.best = fminf(m, quad_perm<kXor2>(m));
                }
            }
        } else if (ANY || q.tn <= q.best) {
            const uint32_t o = (uint32_t)q.ref << 6, oX = o + eX, oY = o + eY, oZ = o + eZ;
            const uint32_t hx = half(oX), hy = half(oY), hz = half(oZ);
            const uint32_t gx = half(oX ^ 8u), gy = half(oY ^ 8u), gz = half(oZ ^ 8u);
            const int child = *(const int*)(nb + (o + eC));
            float t1x = rtd::h_sub<false>(hx, q.ox) * q.ix, t2x = rtd::h_sub<false>(gx, q.ox) * q.ix;
            float t1y = rtd::h_sub<false>(hy, q.oy) * q.iy, t2y = rtd::h_sub<false>(gy, q.oy) * q.iy;
            float t1z = rtd::h_sub<false>(hz, q.oz) * q.iz, t2z = rtd::h_sub<false>(gz, q.oz) * q.iz;
            float tN, tF;
            if (FLAT) {
                t1x = t1x != t1x ? -q.ix : t1x; t2x = t2x != t2x ? q.ix : t2x;
                t1y = t1y != t1y ? -q.iy : t1y; t2y = t2y != t2y ? q.iy : t2y;
                t1z = t1z != t1z ? -q.iz : t1z; t2z = t2z != t2z ? q.iz : t2z;
                tN = fmaxf(fmaxf(fminf(t1x, t2x), fminf(t1y, t2y)), fminf(t1z, t2z));
                tF = fminf(fminf(fmaxf(t1x, t2x), fmaxf(t1y, t2y)), fmaxf(t1z, t2z)) * RT_ROBUST_TFAR;
            } else {
                tN = fmaxf(fmaxf(t1x, t1y), t1z);
                tF = fminf(fminf(t2x, t2y), t2z) * RT_ROBUST_TFAR;
            }
            const float limit = ANY ? q.tmax : q.best;
            const bool hit = (tN <= tF) && (tF >= q.tmin) && (tN <= limit) && child != -1;
            const uint32_t hm = (uint32_t)(__ballot(hit) >> sh) & 15u;
            if (hm) {
                // rank of this lane's child among the quad's hits, nearest
                // first: keys of the entry distance (from 0 up) with the lane
                // in the two low bits, so that no two are equal
                const int key = hit ? (__float_as_int(fmaxf(tN, 0.0f)) & ~3) | c : 0x7ffffffc | c;
                const int k1 = quad_perm<kRot1>(key), k2 = quad_perm<kRot2>(key), k3 = quad_perm<kRot3>(key);
                const int rank = -(((k1 - key) >> 31) + ((k2 - key) >> 31) + ((k3 - key) >> 31));
                const int n = __popc(hm);
                const int at = q.sp + n - 1 - rank;
                if (hit && rank > 0 && at < maxStack) push(q, at, child, tN);
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // the quad's lanes read each other's entries
                q.sp += n - 1;
                if (q.sp > maxStack) { q.sp = maxStack; atomicOr(status, 1); }
                const bool first = hit && rank == 0;
                int rf = first ? child : 0, tb = first ? __float_as_int(tN) : 0;
                rf |= quad_perm<kXor1>(rf); tb |= quad_perm<kXor1>(tb);
                q.ref = rf | quad_perm<kXor2>(rf);
                q.tn = __int_as_float(tb | quad_perm<kXor2>(tb));
                continue;
            }
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
