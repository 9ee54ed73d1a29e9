// scene_dev.h — device pieces of the two-level traversal shared by the
// traversal kernels (scene.hip) and the path tracer's tail kernel (pt.hip): the
// instance transform, the node visit, and a traversal with four lanes per ray.
#pragma once

#include <hip/hip_runtime.h>

#include <climits>

#include "rt_device.h"
#include "rt_quad.h"
#include "scene.h"

namespace rtk {

using rtd::Ray;

constexpr int kReturnMark = INT_MIN;   // return marker: leave the instance

// World-space unit geometric normal of leaf-order triangle li of instance I's
// BLAS B: the object-space e1 x e2 (the mesh's winding, not turned toward any
// ray) mapped with the transpose of the world-to-object 3x3 (the inverse
// transpose of the object-to-world map), then normalised.
__device__ __forceinline__ void world_normal(const InstanceDev& I, const BlasDev& B, int li, float& nx, float& ny,
                                             float& nz) {
    const float4 p0 = rtd::ldg_f4(B.tris + 3 * li), p1 = rtd::ldg_f4(B.tris + 3 * li + 1),
                 p2 = rtd::ldg_f4(B.tris + 3 * li + 2);
    const float e1x = p1.x - p0.x, e1y = p1.y - p0.y, e1z = p1.z - p0.z;
    const float e2x = p2.x - p0.x, e2y = p2.y - p0.y, e2z = p2.z - p0.z;
    const float mx = e1y * e2z - e1z * e2y, my = e1z * e2x - e1x * e2z, mz = e1x * e2y - e1y * e2x;
    const float* W = I.w2o;
    nx = (W[0] * mx + W[4] * my) + W[8] * mz;
    ny = (W[1] * mx + W[5] * my) + W[9] * mz;
    nz = (W[2] * mx + W[6] * my) + W[10] * mz;
    const float nl = 1.0f / sqrtf((nx * nx + ny * ny) + nz * nz);
    nx = nx * nl; ny = ny * nl; nz = nz * nl;
}

__device__ __forceinline__ void xform(const float* M, const Ray& w, Ray& o) {
    o.ox = ((M[0] * w.ox + M[1] * w.oy) + M[2] * w.oz) + M[3];
    o.oy = ((M[4] * w.ox + M[5] * w.oy) + M[6] * w.oz) + M[7];
    o.oz = ((M[8] * w.ox + M[9] * w.oy) + M[10] * w.oz) + M[11];
    o.dx = (M[0] * w.dx + M[1] * w.dy) + M[2] * w.dz;
    o.dy = (M[4] * w.dx + M[5] * w.dy) + M[6] * w.dz;
    o.dz = (M[8] * w.dx + M[9] * w.dy) + M[10] * w.dz;
    o.tmin = w.tmin;
    o.tmax = w.tmax;
    rtd::ray_setup(o);
}

template <bool ANY, bool FLAT, class Push>
__device__ __forceinline__ void visit2(const uint4* __restrict__ nodes, const Ray& r, float limit, int& ref, float& tn,
                                       Push&& push) {
    const uint4* np = nodes + 4 * (size_t)ref;
    const uint4 qc = rtd::ldg_u4(np + 3);
    const rtd::NodeBox<FLAT> b = rtd::node_box<FLAT>(r, rtd::ldg_u4(np), rtd::ldg_u4(np + 1), rtd::ldg_u4(np + 2));
    if constexpr (ANY) {
        float d0, d1, d2, d3;
        const bool h0 = rtd::child_hit<0, FLAT>(r, b, (int)qc.x, limit, d0);
        const bool h1 = rtd::child_hit<1, FLAT>(r, b, (int)qc.y, limit, d1);
        const bool h2 = rtd::child_hit<2, FLAT>(r, b, (int)qc.z, limit, d2);
        const bool h3 = rtd::child_hit<3, FLAT>(r, b, (int)qc.w, limit, d3);
        int nxt = -1;
        if (h0) { nxt = (int)qc.x; }
        if (h1) { if (nxt != -1) push(nxt, 0.f); nxt = (int)qc.y; }
        if (h2) { if (nxt != -1) push(nxt, 0.f); nxt = (int)qc.z; }
        if (h3) { if (nxt != -1) push(nxt, 0.f); nxt = (int)qc.w; }
        ref = nxt;
        tn = 0.f;
    } else {
        float d[4];
        int c[4];
        float tt;
        if (rtd::child_hit<0, FLAT>(r, b, (int)qc.x, limit, tt)) { d[0] = tt; c[0] = (int)qc.x; } else { d[0] = INFINITY; c[0] = -1; }
        if (rtd::child_hit<1, FLAT>(r, b, (int)qc.y, limit, tt)) { d[1] = tt; c[1] = (int)qc.y; } else { d[1] = INFINITY; c[1] = -1; }
        if (rtd::child_hit<2, FLAT>(r, b, (int)qc.z, limit, tt)) { d[2] = tt; c[2] = (int)qc.z; } else { d[2] = INFINITY; c[2] = -1; }
        if (rtd::child_hit<3, FLAT>(r, b, (int)qc.w, limit, tt)) { d[3] = tt; c[3] = (int)qc.w; } else { d[3] = INFINITY; c[3] = -1; }
#define RT_CSWAP(i, j)                                                                  \
    {                                                                                   \
        const bool s = d[i] > d[j];                                                     \
        const float di = d[i], dj = d[j];                                               \
        const int ci = c[i], cj = c[j];                                                 \
        d[i] = s ? dj : di; d[j] = s ? di : dj; c[i] = s ? cj : ci; c[j] = s ? ci : cj; \
    }
        RT_CSWAP(0, 1) RT_CSWAP(2, 3) RT_CSWAP(0, 2) RT_CSWAP(1, 3) RT_CSWAP(1, 2)
#undef RT_CSWAP
        int nxt = -1;
        float nt = 0.f;
        if (c[3] != -1) { nxt = c[3]; nt = d[3]; }
        if (c[2] != -1) { if (nxt != -1) push(nxt, nt); nxt = c[2]; nt = d[2]; }
        if (c[1] != -1) { if (nxt != -1) push(nxt, nt); nxt = c[1]; nt = d[1]; }
        if (c[0] != -1) { if (nxt != -1) push(nxt, nt); nxt = c[0]; nt = d[0]; }
        ref = nxt;
        tn = nt;
    }
}

// Node visit with the slab variant picked per wave: the one that resolves
// 0*inf when any active lane's current ray (world or object space) is flat,
// the plain one otherwise; both agree on every ray that is not flat.
template <bool ANY, class Push>
__device__ __forceinline__ void visit2w(const uint4* __restrict__ nodes, const Ray& r, bool flat, float limit, int& ref,
                                        float& tn, Push&& push) {
    if (__any(flat)) visit2<ANY, true>(nodes, r, limit, ref, tn, push);
    else visit2<ANY, false>(nodes, r, limit, ref, tn, push);
}


// A two-level traversal held by the four lanes of a quad (rt_quad.h): the
// current ray, in world or object space. The world ray stays in LDS (at w:
// three components of the origin, then of the direction, `stride` apart).
struct Quad2 : rtq::Ray4 {
    int inst, hinst;                    // current instance (-1: world), instance of this lane's candidate
    rtq::gptr nodes, tris;
};

// Lane C's value in every lane of a quad.
template <int C>
__device__ __forceinline__ float quad_bcast(float v) { return rtq::quad_perm<C * 0x55>(v); }

// Makes the world ray current (TLAS nodes; no triangles are tested in it, so
// the shear is not set up). Each lane divides for its own axis.
__device__ __forceinline__ void quad_world(Quad2& q, int c, const float* w, int stride, const void* tlasNodes) {
    const float inv = 1.0f / w[(3 + min(c, 2)) * stride];
    q.ox = w[0]; q.oy = w[stride]; q.oz = w[2 * stride];
    q.ix = quad_bcast<0>(inv); q.iy = quad_bcast<1>(inv); q.iz = quad_bcast<2>(inv);
    q.kx = 0; q.ky = 1; q.kz = 2;
    q.inst = -1;
    q.nodes = (rtq::gptr)tlasNodes;
}

// Makes instance k's object-space ray current: xform and rtd::ray_setup with
// the same operations, each lane transforming and dividing for its own axis.
__device__ __forceinline__ void quad_enter(Quad2& q, int c, const float* w, int stride, int k, const InstanceDev* insts,
                                           const BlasDev* blas) {
    const InstanceDev& I = insts[k];
    const float4 M = ((const float4*)I.w2o)[min(c, 2)];
    const BlasDev& B = blas[I.blas];
    const float o = ((M.x * w[0] + M.y * w[stride]) + M.z * w[2 * stride]) + M.w;
    const float d = (M.x * w[3 * stride] + M.y * w[4 * stride]) + M.z * w[5 * stride];
    const float inv = 1.0f / d;
    const float dx = quad_bcast<0>(d), dy = quad_bcast<1>(d), dz = quad_bcast<2>(d);
    const float ix = quad_bcast<0>(inv), iy = quad_bcast<1>(inv), iz = quad_bcast<2>(inv);
    const float ax = fabsf(dx), ay = fabsf(dy), az = fabsf(dz);
    int kz = 0;
    if (ay > ax) kz = 1;
    if (az > (kz == 0 ? ax : ay)) kz = 2;
    int kx = kz + 1; if (kx == 3) kx = 0;
    int ky = kx + 1; if (ky == 3) ky = 0;
    const float dkz = rtd::sel3(kz, dx, dy, dz);
    if (dkz < 0.0f) { const int t = kx; kx = ky; ky = t; }
    const float S = (c == 0 ? rtd::sel3(kx, dx, dy, dz) : c == 1 ? rtd::sel3(ky, dx, dy, dz) : 1.0f) / dkz;
    q.Sx = quad_bcast<0>(S); q.Sy = quad_bcast<1>(S); q.Sz = quad_bcast<2>(S);
    const float ox = quad_bcast<0>(o), oy = quad_bcast<1>(o), oz = quad_bcast<2>(o);
    q.ox = rtd::sel3(kx, ox, oy, oz); q.oy = rtd::sel3(ky, ox, oy, oz); q.oz = rtd::sel3(kz, ox, oy, oz);
    q.ix = rtd::sel3(kx, ix, iy, iz); q.iy = rtd::sel3(ky, ix, iy, iz); q.iz = rtd::sel3(kz, ix, iy, iz);
    q.kx = kx; q.ky = ky; q.kz = kz;
    q.inst = k;
    q.nodes = (rtq::gptr)B.nodes;
    q.tris = (rtq::gptr)B.tris;
}

// Two-level traversal of the rays of quads with `has`, from q.ref (a node or
// leaf code, a return marker, or -1: what the stack holds next) until they are
// done; the current ray is set up. Culling and tie rule of k_trace2l; the
// stack as in rtq::traverse. Returns the steps taken; q.found: an any-hit
// ray's result. A closest-hit ray with `first` also ends at its first hit (one
// below q.tmax). The loop has one way through and ends for all quads at once:
// with quads leaving it, or continuing it, from within, each of the some 30
// registers of state had a second one and was copied in every step.
template <bool ANY, class Push, class Pop>
__device__ __forceinline__ int quad_trace2(Quad2& q, bool has, int c, int sh, const float* w, int stride,
                                           const void* tlasNodes, const float4* tlasTris, const InstanceDev* insts,
                                           const BlasDev* blas, int maxStack, int* status, Push&& push, Pop&& pop,
                                           bool first = false) {
    int steps = 0;
    while (__any(has)) {
        steps++;
        bool next = false;
        if (has) {
            if (q.ref >= 0) {
                if (ANY || q.tn <= q.best)
                    next = rtq::visit<ANY>(q, c, sh, rtq::slot_of(q, q.nodes + ((size_t)(uint32_t)q.ref << 6), c), maxStack,
                                           status, push);
            } else if (q.ref == kReturnMark) {
                quad_world(q, c, w, stride, tlasNodes);
            } else if (q.ref != -1 && (ANY || q.tn <= q.best)) {
                const int enc = -(q.ref + 2);
                if (q.inst < 0) {
                    // TLAS leaf: enter its instance
                    const int k = __float_as_int(tlasTris[3 * (enc >> 3)].w);
                    if (q.sp < maxStack) {
                        if (c == 0) push(q, q.sp, kReturnMark, -INFINITY);
                        q.sp++;
                    } else {
                        atomicOr(status, 1);   // unreachable: maxStack bounds a DFS of the two levels
                    }
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    quad_enter(q, c, w, stride, k, insts, blas);
                    q.ref = 0;
                    q.tn = -INFINITY;
                    next = true;
                } else {
                    q.found = rtq::leaf<ANY>(q, c, sh, q.tris + (size_t)(enc >> 3) * 48, 0, (enc & 7) + 1, [&](float t, int id) {
                        const bool closer =
                            t < q.t || (t == q.t && (q.inst < q.hinst || (q.inst == q.hinst && id < q.id)));
                        if (closer) q.hinst = q.inst;
                        return closer;
                    });
                }
            }
            if (!next) {
                has = q.sp > 0 && !(ANY ? q.found : first && q.best < q.tmax);
                if (has) {
                    q.sp--;
                    pop(q, q.sp, q.ref, q.tn);
                }
            }
        }
    }
    return steps;
}

// The quad's closest hit into every lane (ties: the lowest instance, then ID).
__device__ __forceinline__ void quad_reduce2(Quad2& q) {
#define RT_QSTEP(P)                                                                                          \
    {                                                                                                        \
        const float t = rtq::quad_perm<P>(q.t), u = rtq::quad_perm<P>(q.u), v = rtq::quad_perm<P>(q.v);      \
        const int id = rtq::quad_perm<P>(q.id), in = rtq::quad_perm<P>(q.hinst);                             \
        if (t < q.t || (t == q.t && (in < q.hinst || (in == q.hinst && id < q.id)))) {                       \
            q.t = t; q.u = u; q.v = v; q.id = id; q.hinst = in;                                              \
        }                                                                                                    \
    }
    RT_QSTEP(rtq::kXor1) RT_QSTEP(rtq::kXor2)
#undef RT_QSTEP
}

}  // namespace rtk
