// scene.hip — two-level scenes: a TLAS (BVH4 over instance boxes, one
// instance per leaf) above per-mesh BLAS handles, and its closest-hit /
// any-hit traversal.
//
// One depth-first traversal per ray: reaching a TLAS leaf pushes a return
// marker, transforms the ray into the instance's object space with the
// world-to-object affine map (unnormalised, so t stays the world distance
// parameter) and continues into the BLAS; popping the marker restores the
// world ray. The closest hit is the lexicographic minimum of (t, instance,
// primitive). The schedule is the while-while one of trace.hip (node and leaf
// phases, idle lanes refilled from a wave-local pool of 64-ray batches).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>

#include "rt_device.h"
#include "rt_internal.h"
#include "scene.h"
#include "scene_dev.h"
#include "trace_launch.h"

namespace rtk {

using rtd::Ray;

template <bool ANY, int LDSD, int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_trace2l(Trace2LArgs a) {
    __shared__ int s_ref[LDSD * BLOCK];
    __shared__ float s_tn[LDSD * BLOCK];
    const int tid = threadIdx.x, lane = tid & 63;
    const int gtid = blockIdx.x * BLOCK + tid;
    if (a.gate && *a.gate <= a.gateMax) return;
    const int n = a.nDev ? min(*a.nDev, a.n) : a.n;

    Ray rw, ro;
    int ri = 0, inst = -1;
    const uint4* nodes = a.tlasNodes;
    const float4* tris = nullptr;
    bool has = false, exhausted = false, found = false, flatW = false, flatO = false;
    int poolNext = 0, poolEnd = 0;
    int band = blockIdx.x % rtd::kBands;   // wave-uniform: band of the work distribution
    int sp = 0, ref = -1, bid = -1, binst = -1, visits = 0, tests = 0;
    int pend = -1;             // postponed BLAS leaf (speculative node phase), -1: none
    float tn = 0.f, best = 0.f, bu = 0.f, bv = 0.f;
    // Uncounted launches postpone BLAS leaves speculatively, as the
    // single-level while-while kernel does; a lane holding a postponed leaf
    // stays inside its instance (it waits at the return marker), so the leaf
    // is tested with that instance's object-space ray.
    const bool spec = a.cntNodes == nullptr;

    auto push = [&](int rf, float t) {
        if (sp < LDSD) {
            s_ref[sp * BLOCK + tid] = rf;
            s_tn[sp * BLOCK + tid] = t;
        } else if (sp < a.maxStack) {
            a.spill[(size_t)(sp - LDSD) * a.spillStride + gtid] = make_int2(rf, __float_as_int(t));
        } else {
            atomicOr(a.status, 1);
            return;
        }
        sp++;
    };

    for (;;) {
        if (!exhausted || poolNext < poolEnd) {
            const uint64_t idle = __ballot(!has);
            if (idle) {
                const int cnt = __popcll(idle);
                const int avail = poolEnd - poolNext;
                int fresh = n;
                if (cnt > avail && !exhausted) {
                    fresh = rtd::take_chunk(a.counter, n, band);
                    if (fresh >= n) exhausted = true;
                }
                const int k = __popcll(idle & ((1ull << lane) - 1ull));
                int w = n;
                if (k < avail) w = poolNext + k;
                else if (fresh < n) w = fresh + (k - avail);
                if (cnt > avail) {
                    if (fresh < n) { poolNext = fresh + (cnt - avail); poolEnd = fresh + 64; }
                    else { poolNext = 0; poolEnd = 0; }
                } else {
                    poolNext += cnt;
                }
                if (!has && w < n) {
                    ri = w;
                    rw.ox = a.ox[ri]; rw.oy = a.oy[ri]; rw.oz = a.oz[ri];
                    rw.dx = a.dx[ri]; rw.dy = a.dy[ri]; rw.dz = a.dz[ri];
                    rw.tmin = a.tmin[ri]; rw.tmax = a.tmax[ri];
                    rtd::ray_setup(rw);
                    flatW = rtd::ray_flat(rw);
                    has = true;
                    sp = 0; ref = 0; tn = -INFINITY; inst = -1; nodes = a.tlasNodes;
                    best = rw.tmax; bu = 0.f; bv = 0.f; bid = -1; binst = -1;
                    visits = 0; tests = 0; found = false;
                }
            }
        }
        if (!__any(has)) {
            if (exhausted && poolNext >= poolEnd) break;
            continue;
        }
        bool fin = false;
        for (;;) {
            if (has && !fin) {
                for (;;) {
                    while (ref == -1 || ref == kReturnMark || (!ANY && tn > best)) {
                        if (ref == kReturnMark) {
                            if (pend != -1) break;           // wait inside the instance
                            inst = -1; nodes = a.tlasNodes; ref = -1;
                            continue;
                        }
                        if (sp == 0) { fin = true; break; }
                        sp--;
                        if (sp < LDSD) {
                            ref = s_ref[sp * BLOCK + tid];
                            tn = s_tn[sp * BLOCK + tid];
                        } else {
                            const int2 e = a.spill[(size_t)(sp - LDSD) * a.spillStride + gtid];
                            ref = e.x; tn = __int_as_float(e.y);
                        }
                    }
                    if (spec && !fin && inst >= 0 && ref < -1 && ref != kReturnMark && pend == -1) {
                        pend = ref; ref = -1;
                        continue;
                    }
                    break;
                }
            }
            // TLAS nodes, TLAS leaves (instance entry) and BLAS nodes are node
            // work; a lane waiting at the return marker with a postponed leaf
            // is not
            const bool atNode = has && !fin && ref != kReturnMark && (ref >= 0 || inst < 0);
            if (!__any(atNode && pend == -1)) break;
            if (atNode) {
                if (ref >= 0) {
                    visits++;
                    const bool w = inst < 0;
                    const Ray& r = w ? rw : ro;
                    visit2w<ANY>(nodes, r, w ? flatW : flatO, ANY ? r.tmax : best, ref, tn, push);
                } else {
                    // TLAS leaf: enter its instance
                    const int enc = -(ref + 2);
                    const int k = __float_as_int(a.tlasTris[3 * (enc >> 3)].w);
                    push(kReturnMark, -INFINITY);
                    inst = k;
                    const InstanceDev& I = a.inst[k];
                    xform(I.w2o, rw, ro);
                    flatO = rtd::ray_flat(ro);
                    const BlasDev& B = a.blas[I.blas];
                    nodes = B.nodes;
                    tris = B.tris;
                    ref = 0;
                    tn = -INFINITY;
                }
            }
        }
        const int leaf = spec ? pend : ((has && !fin) ? ref : -1);
        if (has && leaf < -1) {
            const int enc = -(leaf + 2), ts = enc >> 3, tc = (enc & 7) + 1;
            for (int q = 0; q < tc; q++) {
                const int ti = ts + q;
                tests++;
                const float4 p0 = rtd::ldg_f4(tris + 3 * ti);
                float t, u, v;
                if (!rtd::isect_watertight(ro, p0, rtd::ldg_f4(tris + 3 * ti + 1), rtd::ldg_f4(tris + 3 * ti + 2), t, u, v)) continue;
                if (!(t > ro.tmin) || !(t < ro.tmax)) continue;
                if constexpr (ANY) {
                    found = true;
                    fin = true;
                    break;
                } else {
                    const int id = __float_as_int(p0.w);
                    if (t < best || (t == best && (inst < binst || (inst == binst && id < bid)))) {
                        best = t; bid = id; binst = inst; bu = u; bv = v;
                    }
                }
            }
            if (spec) pend = -1;
            else ref = -1;
        }
        if (has && fin) {
            if constexpr (ANY) {
                a.occ[ri] = found ? 1 : 0;
            } else {
                const bool hit = bid >= 0;
                a.t[ri] = hit ? best : RT_MISS_T;
                if (a.inst_out) a.inst_out[ri] = binst;
                if (a.id) a.id[ri] = bid;
                if (a.u) a.u[ri] = hit ? bu : 0.f;
                if (a.v) a.v[ri] = hit ? bv : 0.f;
            }
            if (a.cntNodes) { a.cntNodes[ri] = visits; a.cntTris[ri] = tests; }
            has = false;
        }
    }
}

// Rays left in a wave when four lanes take each of them over: as many as it
// has quads.
constexpr int kQuadRays2 = 16;

// Stack entry `at` of column `col` beyond the LDS ones. The opaque column keeps
// the compiler from holding its address through the traversal loops.
template <int LDSD>
__device__ __forceinline__ int2* spill2(const Trace2LArgs& a, int at, int col) {
    asm volatile("" : "+v"(col));
    return a.spill + ((size_t)(at - LDSD) * a.spillStride + col);
}
// (a non-temporal load: not merged with the LDS read beside it into a flat load)
__device__ __forceinline__ void unspill2(const int2* p, int& ref, float& tn) {
    typedef int v2i __attribute__((ext_vector_type(2)));
    const v2i e = __builtin_nontemporal_load((const v2i*)p);
    ref = e.x; tn = __int_as_float(e.y);
}

// What a ray of trace2l_wave ends with: its hit so far and, when quads are to
// go on with it (open), its traversal state.
struct Wave2 {
    float t, u, v, tn;
    int id, hinst, ref, inst, sp, steps;
    bool occluded, open;
};

// The rays of a wave through TLAS and BLAS, ending when at most kQuadRays2
// lanes still hold one (Wave2::open). Every lane calls it; `live` lanes hold a
// ray. Culling and tie rule of k_trace2l (any hit may visit children nearest
// first, ORD). Each iteration is one short step per lane — a node visit, an
// instance entry, or the next one or two triangles of the current BLAS leaf
// (leaf cursor; the two fetched together) — so lanes at different kinds of
// step do not wait for whole leaf loops. As in the one-level batch kernel, the
// wave's priority rises one level per 32 steps, so that long walks (grazing
// rays) issue ahead of short ones, and the loop is wave-uniform. r is the
// lane's current ray, in world or object space; the world ray is in s_w, from
// where an instance entry, or the return from one, takes it.
template <bool ANY, bool ORD, int LDSD, int BLOCK>
__device__ __forceinline__ void trace2l_wave(const Trace2LArgs& a, Ray& r, bool live, int* s_ref, float* s_tn,
                                             float* s_w, int tid, int gtid, Wave2& res) {
    int ref = 0, inst = -1, sp = 0, bid = -1, binst = -1;
    int lts = 0, ltc = 0;                   // leaf cursor: next triangle, triangles left
    float tn = -INFINITY, best = r.tmax, bu = 0.f, bv = 0.f;
    bool has = live, found = false, flat = live && rtd::ray_flat(r);
    const uint4* nodes = a.tlasNodes;
    const float4* tris = nullptr;
    auto push = [&](int rf, float t) {
        if (sp < LDSD) {
            s_ref[sp * BLOCK + tid] = rf;
            s_tn[sp * BLOCK + tid] = t;
        } else if (sp < a.maxStack) {
            *spill2<LDSD>(a, sp, gtid) = make_int2(rf, __float_as_int(t));
        } else {
            atomicOr(a.status, 1);   // unreachable: maxStack bounds a DFS of the two levels
            return;
        }
        sp++;
    };
    constexpr int kPrio2 = 32;
    int steps = 0;
    for (;;) {
        if (__popcll(__ballot(has)) <= kQuadRays2) break;
        steps++;
        if (steps == kPrio2) __builtin_amdgcn_s_setprio(1);
        else if (steps == 2 * kPrio2) __builtin_amdgcn_s_setprio(2);
        else if (steps == 3 * kPrio2) __builtin_amdgcn_s_setprio(3);
        if (!has) continue;
        if (ltc == 0) {
            while (ref == -1 || ref == kReturnMark || (!ANY && tn > best)) {
                if (ref == kReturnMark) {
                    inst = -1; nodes = a.tlasNodes; ref = -1;
                    r.ox = s_w[tid]; r.oy = s_w[BLOCK + tid]; r.oz = s_w[2 * BLOCK + tid];
                    r.ix = 1.0f / s_w[3 * BLOCK + tid];
                    r.iy = 1.0f / s_w[4 * BLOCK + tid];
                    r.iz = 1.0f / s_w[5 * BLOCK + tid];
                    flat = rtd::ray_flat(r);
                    continue;
                }
                if (sp == 0) { has = false; break; }
                sp--;
                if (sp < LDSD) {
                    ref = s_ref[sp * BLOCK + tid];
                    tn = s_tn[sp * BLOCK + tid];
                } else {
                    unspill2(spill2<LDSD>(a, sp, gtid), ref, tn);
                }
            }
            if (!has) continue;
            if (ref < 0 && inst >= 0) {         // BLAS leaf: start its cursor
                const int enc = -(ref + 2);
                lts = enc >> 3; ltc = (enc & 7) + 1;
                ref = -1;
            }
        }
        if (ltc > 0) {
            const int ti = lts;
            const bool two = ltc > 1;
            const int tj = two ? ti + 1 : ti;
            const float4 p0 = rtd::ldg_f4(tris + 3 * ti), p1 = rtd::ldg_f4(tris + 3 * ti + 1), p2 = rtd::ldg_f4(tris + 3 * ti + 2);
            const float4 q0 = rtd::ldg_f4(tris + 3 * tj), q1 = rtd::ldg_f4(tris + 3 * tj + 1), q2 = rtd::ldg_f4(tris + 3 * tj + 2);
            lts += two ? 2 : 1;
            ltc -= two ? 2 : 1;
            // leaf order: the first triangle, then the second (a closest-hit
            // update of the first is seen by the second's tie rule)
            auto test = [&](const float4& a0, const float4& a1, const float4& a2) {
                float t, u, v;
                if (rtd::isect_watertight(r, a0, a1, a2, t, u, v) && t > r.tmin) {
                    if constexpr (ANY) return t < r.tmax;
                    // (best starts at tmax with no instance: a hit there is none)
                    const int id = __float_as_int(a0.w);
                    if (t < best || (t == best && (inst < binst || (inst == binst && id < bid)))) {
                        best = t; bid = id; binst = inst; bu = u; bv = v;
                    }
                }
                return false;
            };
            if (test(p0, p1, p2) || (two && test(q0, q1, q2))) { found = true; has = false; }
        } else if (ref >= 0) {
            const uint4* np = nodes + 4 * (size_t)ref;
            const uint4 qc = rtd::ldg_u4(np + 3), nx = rtd::ldg_u4(np), ny = rtd::ldg_u4(np + 1), nz = rtd::ldg_u4(np + 2);
            constexpr bool SLOTS = ANY && !ORD;     // children in slot order
            const float limit = ANY ? r.tmax : best;
            const bool down = __any(flat)
                ? rtd::visit_free<SLOTS, true, LDSD, BLOCK>(r, nx, ny, nz, qc, limit, ref, tn, s_ref, s_tn, tid, sp, push)
                : rtd::visit_free<SLOTS, false, LDSD, BLOCK>(r, nx, ny, nz, qc, limit, ref, tn, s_ref, s_tn, tid, sp, push);
            if (!down) ref = -1;
        } else {
            // TLAS leaf: enter its instance
            const int enc = -(ref + 2);
            const int k = __float_as_int(a.tlasTris[3 * (enc >> 3)].w);
            push(kReturnMark, -INFINITY);
            inst = k;
            const InstanceDev& I = a.inst[k];
            Ray w;
            w.ox = s_w[tid]; w.oy = s_w[BLOCK + tid]; w.oz = s_w[2 * BLOCK + tid];
            w.dx = s_w[3 * BLOCK + tid]; w.dy = s_w[4 * BLOCK + tid]; w.dz = s_w[5 * BLOCK + tid];
            w.tmin = r.tmin; w.tmax = r.tmax;
            xform(I.w2o, w, r);
            flat = rtd::ray_flat(r);
            const BlasDev& B = a.blas[I.blas];
            nodes = B.nodes;
            tris = B.tris;
            ref = 0;
            tn = -INFINITY;
        }
    }
    __builtin_amdgcn_s_setprio(0);
    res.t = best; res.u = bu; res.v = bv; res.id = bid; res.hinst = binst;
    res.occluded = found; res.steps = steps; res.open = has;
    // a leaf cursor as a leaf code, which is not tested against the closest hit again
    res.ref = ltc > 0 ? -((lts << 3) | (ltc - 1)) - 2 : ref;
    res.tn = ltc > 0 ? -INFINITY : tn; res.inst = inst; res.sp = sp;
}

// Rays that a wave has left (lanes with w.open, at most kQuadRays2 of them) go
// on with four lanes each, with their stacks in place and their results
// written from here; the ray is read again. Every lane of the wave calls it.
// Returns the longest quad's steps.
template <bool ANY, int LDSD, int BLOCK>
__device__ __forceinline__ int finish_quads2(const Trace2LArgs& a, const Wave2& w, int ri, int* s_ref, float* s_tn,
                                             const float* s_w, int tid, int gtid) {
    asm volatile("" : "+v"(tid), "+v"(gtid));    // addresses of this phase are not computed ahead of the loop
    const int lane = tid & 63, src = rtq::source_lane(__ballot(w.open), lane), from = src < 0 ? lane : src;
    const int c = lane & 3, sh = lane & 60;
    Quad2 q;
    ri = rtq::take(from, ri);
    q.ref = rtq::take(from, w.ref);
    q.tn = rtq::take(from, w.tn);
    q.sp = rtq::take(from, w.sp);
    const int inst = rtq::take(from, w.inst);
    if constexpr (!ANY) {
        q.best = q.t = rtq::take(from, w.t);
        q.id = rtq::take(from, w.id);
        q.hinst = rtq::take(from, w.hinst);
        q.u = rtq::take(from, w.u); q.v = rtq::take(from, w.v);
    }
    q.col = from - lane;
    q.found = false;
    int steps = 0;
    if (src >= 0) {
        __builtin_amdgcn_s_setprio(3);
        const float* world = s_w + (tid + q.col);
        q.tmin = a.tmin[ri]; q.tmax = a.tmax[ri];
        if (inst < 0) quad_world(q, c, world, BLOCK, a.tlasNodes);
        else quad_enter(q, c, world, BLOCK, inst, a.inst, a.blas);
        auto push = [&](rtq::Ray4& z, int at, int rf, float t) {
            if (at < LDSD) {
                s_ref[at * BLOCK + tid + z.col] = rf;
                s_tn[at * BLOCK + tid + z.col] = t;
            } else {
                *spill2<LDSD>(a, at, gtid + z.col) = make_int2(rf, __float_as_int(t));
            }
        };
        auto pop = [&](rtq::Ray4& z, int at, int& rf, float& t) {
            if (at < LDSD) {
                rf = s_ref[at * BLOCK + tid + z.col];
                t = s_tn[at * BLOCK + tid + z.col];
            } else {
                unspill2(spill2<LDSD>(a, at, gtid + z.col), rf, t);
            }
        };
        steps = quad_trace2<ANY>(q, true, c, sh, world, BLOCK, a.tlasNodes, a.tlasTris, a.inst, a.blas, a.maxStack, a.status,
                                 push, pop);
        __builtin_amdgcn_s_setprio(0);
        if constexpr (!ANY) quad_reduce2(q);
        if (c == 0) {
            if constexpr (ANY) {
                a.occ[ri] = q.found ? 1 : 0;
            } else {
                const bool hit = q.id >= 0;
                a.t[ri] = hit ? q.t : RT_MISS_T;
                if (a.inst_out) a.inst_out[ri] = q.hinst;
                if (a.id) a.id[ri] = q.id;
                if (a.u) a.u[ri] = hit ? q.u : 0.f;
                if (a.v) a.v[ri] = hit ? q.v : 0.f;
            }
        }
    }
    return rtd::wave_max(steps);
}

// Batch schedule: each wave takes 64 rays from its XCD band
// (rtd::take_chunk), one per lane (trace2l_wave), and the last 16 of them with
// four lanes each. When all rays of the launch fit in quads at once, a wave
// takes 16 rays, which start in quads. What bounds a launch is the chain of
// dependent node and triangle fetches of each wave's slowest rays, during
// which most lanes have long finished: with quads for the last 16 rays 1 M
// random rays into 64 instances went from 560 to 450 us (closest) and 440 to
// 380 us (any hit), the camera rays of a 1080p path-traced sample from 700 to
// 570 us and its first bounce from 1,120 to 910 us. Handing over 8 rays
// instead of 16 gave about half of that. Five waves per SIMD: at four (no
// register spilled) the closest-hit launches took 7 % longer.
template <bool ANY, bool ORD, int LDSD, int BLOCK>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(5))) void k_trace2l_batch(Trace2LArgs a) {
    __shared__ int s_ref[LDSD * BLOCK];
    __shared__ float s_tn[LDSD * BLOCK];
    __shared__ float s_w[6 * BLOCK];             // world rays: origins, directions
    const int tid = threadIdx.x, lane = tid & 63;
    const int gtid = blockIdx.x * BLOCK + tid;
    if (a.gate && *a.gate <= a.gateMax) return;
    const int n = a.nDev ? min(*a.nDev, a.n) : a.n;
    const bool direct = n <= (int)gridDim.x * (BLOCK / 64) * kQuadRays2;
    int band = blockIdx.x % rtd::kBands;
    const int nChunks = (n + 63) >> 6;
    for (bool more = true; more;) {
        int ri, chunk = 0;
        bool live;
        if (direct) {
            ri = __builtin_amdgcn_readfirstlane(blockIdx.x * (BLOCK / 64) + (tid >> 6)) * kQuadRays2 + lane;
            live = lane < kQuadRays2 && ri < n;
            more = false;
        } else {
            const int base = rtd::take_chunk(a.counter, n, band);
            if (base >= n) break;
            // chunk c traces chunk c, or chunkOrder[c] in a cost-ordered launch
            chunk = base >> 6;
            if (a.chunkOrder) chunk = a.chunkOrder[chunk];
            ri = chunk * 64 + lane;
            live = (unsigned)chunk < (unsigned)nChunks && ri < n;
        }
        Ray r;
        r.tmax = 0.f;
        if (live) {
            r.ox = a.ox[ri]; r.oy = a.oy[ri]; r.oz = a.oz[ri];
            r.dx = a.dx[ri]; r.dy = a.dy[ri]; r.dz = a.dz[ri];
            r.tmin = a.tmin[ri]; r.tmax = a.tmax[ri];
            r.ix = 1.0f / r.dx; r.iy = 1.0f / r.dy; r.iz = 1.0f / r.dz;
            s_w[tid] = r.ox; s_w[BLOCK + tid] = r.oy; s_w[2 * BLOCK + tid] = r.oz;
            s_w[3 * BLOCK + tid] = r.dx; s_w[4 * BLOCK + tid] = r.dy; s_w[5 * BLOCK + tid] = r.dz;
        }
        Wave2 w;
        trace2l_wave<ANY, ORD, LDSD, BLOCK>(a, r, live, s_ref, s_tn, s_w, tid, gtid, w);
        if (live && !w.open) {
            if constexpr (ANY) {
                a.occ[ri] = w.occluded ? 1 : 0;
            } else {
                const bool hit = w.id >= 0;
                a.t[ri] = hit ? w.t : RT_MISS_T;
                if (a.inst_out) a.inst_out[ri] = w.hinst;
                if (a.id) a.id[ri] = w.id;
                if (a.u) a.u[ri] = hit ? w.u : 0.f;
                if (a.v) a.v[ri] = hit ? w.v : 0.f;
            }
        }
        int qsteps = 0;
        if (__any(w.open)) qsteps = finish_quads2<ANY, LDSD, BLOCK>(a, w, ri, s_ref, s_tn, s_w, tid, gtid);
        // a quad's step is about half as long
        if (!direct && a.chunkCost && lane == 0 && (unsigned)chunk < (unsigned)nChunks)
            a.chunkCost[chunk] = w.steps + qsteps / 2;
    }
}

// Refill schedule: trace2l_wave's one-short-step loop (a node visit, an
// instance entry or one triangle of the current BLAS leaf per iteration),
// with lanes whose ray finished refilled from the wave's pool of 64 rays once
// at least kRefill2Min lanes are idle. Uncounted.
constexpr int kRefill2Min = 16;

template <bool ANY, int LDSD, int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_trace2l_refill(Trace2LArgs a) {
    __shared__ int s_ref[LDSD * BLOCK];
    __shared__ float s_tn[LDSD * BLOCK];
    const int tid = threadIdx.x, lane = tid & 63;
    const int gtid = blockIdx.x * BLOCK + tid;
    if (a.gate && *a.gate <= a.gateMax) return;
    const int n = a.nDev ? min(*a.nDev, a.n) : a.n;

    Ray rw, ro;
    int ri = 0, inst = -1;
    const uint4* nodes = a.tlasNodes;
    const float4* tris = nullptr;
    bool has = false, exhausted = false, flatW = false, flatO = false;
    int poolNext = 0, poolEnd = 0;
    int band = blockIdx.x % rtd::kBands;   // wave-uniform: band of the work distribution
    int sp = 0, ref = -1, bid = -1, binst = -1, lts = 0, ltc = 0;
    float tn = 0.f, best = 0.f, bu = 0.f, bv = 0.f;

    auto push = [&](int rf, float t) {
        if (sp < LDSD) {
            s_ref[sp * BLOCK + tid] = rf;
            s_tn[sp * BLOCK + tid] = t;
        } else if (sp < a.maxStack) {
            a.spill[(size_t)(sp - LDSD) * a.spillStride + gtid] = make_int2(rf, __float_as_int(t));
        } else {
            atomicOr(a.status, 1);
            return;
        }
        sp++;
    };

    for (;;) {
        if (!exhausted || poolNext < poolEnd) {
            const uint64_t idle = __ballot(!has);
            if (idle && (__popcll(idle) >= kRefill2Min || !__any(has))) {
                const int cnt = __popcll(idle);
                const int avail = poolEnd - poolNext;
                int fresh = n;
                if (cnt > avail && !exhausted) {
                    fresh = rtd::take_chunk(a.counter, n, band);
                    if (fresh >= n) exhausted = true;
                }
                const int k = __popcll(idle & ((1ull << lane) - 1ull));
                int w = n;
                if (k < avail) w = poolNext + k;
                else if (fresh < n) w = fresh + (k - avail);
                if (cnt > avail) {
                    if (fresh < n) { poolNext = fresh + (cnt - avail); poolEnd = fresh + 64; }
                    else { poolNext = 0; poolEnd = 0; }
                } else {
                    poolNext += cnt;
                }
                if (!has && w < n) {
                    ri = w;
                    rw.ox = a.ox[ri]; rw.oy = a.oy[ri]; rw.oz = a.oz[ri];
                    rw.dx = a.dx[ri]; rw.dy = a.dy[ri]; rw.dz = a.dz[ri];
                    rw.tmin = a.tmin[ri]; rw.tmax = a.tmax[ri];
                    rtd::ray_setup(rw);
                    flatW = rtd::ray_flat(rw);
                    has = true;
                    sp = 0; ref = 0; tn = -INFINITY; inst = -1; nodes = a.tlasNodes; ltc = 0;
                    best = rw.tmax; bu = 0.f; bv = 0.f; bid = -1; binst = -1;
                }
            }
        }
        if (!__any(has)) {
            if (exhausted && poolNext >= poolEnd) break;
            continue;
        }
        if (!has) continue;
        bool fin = false, found = false;
        if (ltc == 0) {
            while (ref == -1 || ref == kReturnMark || (!ANY && tn > best)) {
                if (ref == kReturnMark) { inst = -1; nodes = a.tlasNodes; ref = -1; continue; }
                if (sp == 0) { fin = true; break; }
                sp--;
                if (sp < LDSD) {
                    ref = s_ref[sp * BLOCK + tid];
                    tn = s_tn[sp * BLOCK + tid];
                } else {
                    const int2 e = a.spill[(size_t)(sp - LDSD) * a.spillStride + gtid];
                    ref = e.x; tn = __int_as_float(e.y);
                }
            }
            if (!fin && ref < 0 && inst >= 0) {      // BLAS leaf: start its cursor
                const int enc = -(ref + 2);
                lts = enc >> 3; ltc = (enc & 7) + 1;
                ref = -1;
            }
        }
        if (!fin) {
            if (ltc > 0) {
                const int ti = lts;
                lts++; ltc--;
                const float4 p0 = rtd::ldg_f4(tris + 3 * ti);
                float t, u, v;
                if (rtd::isect_watertight(ro, p0, rtd::ldg_f4(tris + 3 * ti + 1), rtd::ldg_f4(tris + 3 * ti + 2), t, u, v) && t > ro.tmin &&
                    t < ro.tmax) {
                    if constexpr (ANY) {
                        found = true;
                        fin = true;
                    } else {
                        const int id = __float_as_int(p0.w);
                        if (t < best || (t == best && (inst < binst || (inst == binst && id < bid)))) {
                            best = t; bid = id; binst = inst; bu = u; bv = v;
                        }
                    }
                }
            } else if (ref >= 0) {
                const bool w = inst < 0;
                const Ray& r = w ? rw : ro;
                visit2w<ANY>(nodes, r, w ? flatW : flatO, ANY ? r.tmax : best, ref, tn, push);
            } else {
                // TLAS leaf: enter its instance
                const int enc = -(ref + 2);
                const int k = __float_as_int(a.tlasTris[3 * (enc >> 3)].w);
                push(kReturnMark, -INFINITY);
                inst = k;
                const InstanceDev& I = a.inst[k];
                xform(I.w2o, rw, ro);
                flatO = rtd::ray_flat(ro);
                const BlasDev& B = a.blas[I.blas];
                nodes = B.nodes;
                tris = B.tris;
                ref = 0;
                tn = -INFINITY;
            }
        }
        if (fin) {
            if constexpr (ANY) {
                a.occ[ri] = found ? 1 : 0;
            } else {
                const bool hit = bid >= 0;
                a.t[ri] = hit ? best : RT_MISS_T;
                if (a.inst_out) a.inst_out[ri] = hit ? binst : -1;
                if (a.id) a.id[ri] = hit ? bid : -1;
                if (a.u) a.u[ri] = hit ? bu : 0.f;
                if (a.v) a.v[ri] = hit ? bv : 0.f;
            }
            has = false;
        }
    }
}

constexpr int kBlock2 = 256;

// Zeroes the kBands work-distribution counters (launched with kBands threads).
__global__ void k_reset_counter_2l(uint32_t* c) { c[threadIdx.x * rtd::kBandStride] = 0u; }

template <bool ANY, int LDSD, int SCHED>
static int launch2(Trace2LArgs& a, rt::TraceScratch& sc, int maxStack, int blocksPerCU, hipStream_t s) {
    static rt::KernelInfo ki;
    // SCHED: 0 while-while, 1 batch, 2 batch with nearest-first any hit, 3 refill
    auto kern = SCHED == 0   ? k_trace2l<ANY, LDSD, kBlock2>
                : SCHED == 1 ? k_trace2l_batch<ANY, false, LDSD, kBlock2>
                : SCHED == 2 ? k_trace2l_batch<ANY, true, LDSD, kBlock2>
                             : k_trace2l_refill<ANY, LDSD, kBlock2>;
    rt::note_launch(kern, kBlock2, ki, 0, 0, nullptr);
    int dev = 0, cus = 1;
    hipGetDevice(&dev);
    hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    const int perCU = blocksPerCU > 0 ? std::min(blocksPerCU, ki.maxBlocks) : ki.maxBlocks;
    const int grid = perCU * cus, threads = grid * kBlock2;
    rt::note_launch(kern, kBlock2, ki, perCU, grid, sc.launchInfo);
    a.maxStack = maxStack;
    // only the batch kernels take a chunk order
    if (SCHED != 1 && SCHED != 2) { a.chunkOrder = nullptr; a.chunkCost = nullptr; }
    const int spillDepth = maxStack > LDSD ? maxStack - LDSD : 0;
    const size_t need = (size_t)spillDepth * threads * sizeof(int2);
    if (alloc_scratch(sc) != 0) return -1;
    if (grow_spill(sc, need) != 0) return -1;
    a.spill = (int2*)sc.spill;
    a.spillStride = threads;
    a.counter = sc.counter;
    a.status = sc.status;
    hipLaunchKernelGGL(k_reset_counter_2l, dim3(1), dim3(rtd::kBands), 0, s, sc.counter);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(kBlock2), 0, s, a);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) { rt::set_error("two-level trace launch failed: %s", hipGetErrorString(e)); return -1; }
    return 0;
}

// Stack entries a two-level traversal can need: each visited node pushes at
// most 3 entries along a root-to-leaf path, plus the return marker.
int trace2l_max_stack(const CudaSceneHandle* sc) { return 3 * sc->tlas->depth4 + 4 + 1 + 3 * sc->maxBlasDepth + 4; }

int launch_trace2l(const CudaSceneHandle* sc, rt::TraceScratch& scratch, Trace2LArgs& a, int cls, hipStream_t s) {
    const bool any = cls == 1;
    if (a.n <= 0) return 0;
    a.tlasNodes = (const uint4*)sc->tlas->d_nodes4;
    a.tlasTris = (const float4*)sc->tlas->d_tris;
    a.inst = sc->d_inst;
    a.blas = sc->d_blas;
    const int maxStack = trace2l_max_stack(sc);
    const rt::TraceConfig& c = sc->tune2l[cls >= 0 && cls <= 2 ? cls : 0];
    // counted traces always use the while-while kernel (it keeps the counters)
    const int sched = (a.cntNodes || c.schedule < 0 || c.schedule > 3 || (!any && c.schedule == 2)) ? 0 : c.schedule;
#define RT_L2(D)                                                                                                  \
    if (sched == 0) return any ? launch2<true, D, 0>(a, scratch, maxStack, c.blocksPerCU, s)                     \
                               : launch2<false, D, 0>(a, scratch, maxStack, c.blocksPerCU, s);                   \
    if (sched == 1) return any ? launch2<true, D, 1>(a, scratch, maxStack, c.blocksPerCU, s)                     \
                               : launch2<false, D, 1>(a, scratch, maxStack, c.blocksPerCU, s);                   \
    if (sched == 3) return any ? launch2<true, D, 3>(a, scratch, maxStack, c.blocksPerCU, s)                     \
                               : launch2<false, D, 3>(a, scratch, maxStack, c.blocksPerCU, s);                   \
    return launch2<true, D, 2>(a, scratch, maxStack, c.blocksPerCU, s);
    switch (c.ldsDepth) {
        case 4: { RT_L2(4) }
        case 12: { RT_L2(12) }
        case 16: { RT_L2(16) }
        default: { RT_L2(8) }
    }
#undef RT_L2
}

// World-space geometric normals of closest hits (instance, original
// primitive ID); a miss or an ID outside the scene gives (0, 0, 0).
__global__ void k_hit_normals(const InstanceDev* inst, int numInst, const BlasDev* blas, int n, const int* instId,
                              const int* primId, float* nx, float* ny, float* nz) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float x = 0.0f, y = 0.0f, z = 0.0f;
    const int k = instId[i];
    if (k >= 0 && k < numInst) {
        const InstanceDev& I = inst[k];
        const BlasDev& B = blas[I.blas];
        const int p = primId[i];
        if (p >= 0 && p < B.numTris) world_normal(I, B, B.leafOf[p], x, y, z);
    }
    nx[i] = x; ny[i] = y; nz[i] = z;
}

int launch_hit_normals(const CudaSceneHandle* sc, int n, const int* instId, const int* primId, float* nx, float* ny,
                       float* nz, hipStream_t s) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL(k_hit_normals, dim3((n + 255) / 256), dim3(256), 0, s, sc->d_inst, (int)sc->inst.size(),
                       sc->d_blas, n, instId, primId, nx, ny, nz);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) { rt::set_error("hit normals launch failed: %s", hipGetErrorString(e)); return -1; }
    return 0;
}

}  // namespace rtk
