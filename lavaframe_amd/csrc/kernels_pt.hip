// Wavefront path tracer for gfx950.
//
// One TiledRenderer pass over a tile (renderer.glsl:main + PathTrace,
// pathtrace.glsl:208-295) is split into stages that pass SoA queues through
// HBM:
//   generate  camera rays for the tile pixels and the paths' random-number state;
//             shading of depth 0 starts the rest of the path state
//   extend    closest hit (analytic lights first, then the BVH) per queued ray;
//             one launch per depth takes these and the shadow rays of the depth before
//   shade     miss / emitter / surface shading, next-event candidates, BSDF
//             sampling, Russian roulette; appends continuing rays and shadow
//             rays with one atomic per block (ballot + rank, block offsets in LDS);
//             folds in the next-event terms of the depth before
//   shadow    any hit per shadow ray; clears the candidate when occluded
//   accumulate  pending next-event terms + Kahan-compensated accumulation
// The random-number stream of each path is the reference's: it lives in the
// path state and is consumed in the reference's order; next-event terms are
// evaluated before their shadow test (they consume no random numbers) and
// added after it, in the reference's summation order.
#include "dev_guide.h"
#include "dev_shade.h"
#include "guide_kernels.h"
#include "pt_kernels.h"

namespace lfhd {

LFH_DEV float luminance(V3 c) { return 0.2126f * c.x + 0.7152f * c.y + 0.0722f * c.z; }

// Training record of path p at depth d (only for recorded paths).
LFH_DEV float* guide_rec(const GuideHook& g, int p, int depth) {
    return reinterpret_cast<float*>(g.rec + ((size_t)(p / g.stride) * g.max_depth + depth) * 4);
}

// ---- queue helpers ---------------------------------------------------------------
// Block-aggregated append: every thread of the block calls it at the same point.
// One atomic per block instead of one per wave: all the device's appends to a
// queue hit the same counter, whose atomics serialise across the XCDs.  `lds`
// holds 8 words.  Returns this thread's slot (valid only if `want`).
LFH_DEV uint32_t block_append(uint32_t* counter, bool want, uint32_t* lds) {
    const uint64_t m = __ballot(want);
    const int wave = threadIdx.x >> 6, nw = (int)(blockDim.x >> 6);
    if ((threadIdx.x & 63) == 0) lds[wave] = (uint32_t)__popcll(m);
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t tot = 0;
        for (int w = 0; w < nw; ++w) tot += lds[w];
        uint32_t base = tot ? atomicAdd(counter, tot) : 0u;
        for (int w = 0; w < nw; ++w) {
            const uint32_t c = lds[w];
            lds[w] = base;
            base += c;
        }
    }
    __syncthreads();
    return lds[wave] + (uint32_t)lane_rank(m);
}

// The same for shading's appends: extension rays (`next`) and up to two shadow
// rays per thread, whose counters are the two halves of one 64-bit word, so a
// block takes both ranges with one atomic: shading C0 (4.2M paths) 308 -> 192 us
// per depth on average against an atomic for each.
struct RaySlots {
    uint32_t next, env, light;
};
LFH_DEV RaySlots block_append_rays(uint32_t* counters, bool next, bool env, bool light, uint32_t* lds) {
    const uint64_t mn = __ballot(next), me = __ballot(env), ml = __ballot(light);
    const int wave = threadIdx.x >> 6;
    const uint32_t ne = (uint32_t)__popcll(me);
    if ((threadIdx.x & 63) == 0) {
        lds[wave] = (uint32_t)__popcll(mn);
        lds[4 + wave] = ne + (uint32_t)__popcll(ml);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t a = 0, b = 0;
        for (int w = 0; w < 4; ++w) {
            a += lds[w];
            b += lds[4 + w];
        }
        unsigned long long base = 0;
        if (a | b)
            base = atomicAdd(reinterpret_cast<unsigned long long*>(counters), (unsigned long long)b << 32 | a);
        a = (uint32_t)base;
        b = (uint32_t)(base >> 32);
        for (int w = 0; w < 4; ++w) {
            const uint32_t ca = lds[w], cb = lds[4 + w];
            lds[w] = a;
            lds[4 + w] = b;
            a += ca;
            b += cb;
        }
    }
    __syncthreads();
    RaySlots r;
    r.next = lds[wave] + (uint32_t)lane_rank(mn);
    r.env = lds[4 + wave] + (uint32_t)lane_rank(me);
    r.light = lds[4 + wave] + ne + (uint32_t)lane_rank(ml);
    return r;
}

LFH_DEV float4 f4(V3 v, float w) { return make_float4(v.x, v.y, v.z, w); }

// Counter set d: the counts of the rays that traversal d takes (the extension
// rays of depth d, the shadow rays of depth d - 1) and their fetch counters.
LFH_HD uint32_t* set_counts(uint32_t* counts, int d) { return counts + 2 * (d % kQueueSets); }
LFH_HD unsigned long long* set_fetch(unsigned long long* work, int d) { return work + (size_t)(d % kQueueSets) * 2 * kFetchWords; }

// Adds a set's ray counts to the running totals and clears the set (threads
// 0 .. 2 kFetchSlices - 1 of one block).
LFH_DEV void retire_set(uint32_t* counts, unsigned long long* fetch, unsigned long long* totals, int t) {
    if (t < 2) {
        totals[t] += counts[t];
        counts[t] = 0u;
    }
    if (t < 2 * kFetchSlices) fetch[t * kFetchStride] = 0ull;
}

__global__ void k_pt_reset(uint32_t* counts, unsigned long long* work) {
    for (int d = 0; d < kQueueSets; ++d)
        retire_set(set_counts(counts, d), set_fetch(work, d), work + kWorkTotals, (int)threadIdx.x);
}

// generate: one thread per tile pixel (MULTI: per pixel of every job).
// unshaded: no depth will be shaded (path depth 0), so the radiance starts here and
// no ray is queued: nothing would trace it, and a queue's count goes to the ray totals.
// whole: every path has a pixel (tiles inside the frame), so path p's ray goes to
// slot p.  Tiles that stick out of the frame append their rays, one atomic per
// block; on whole frames those bound the kernel (4.2M paths 194 -> 59 us,
// 16.6M 800 -> 215 us).
template <bool MULTI>
__global__ __launch_bounds__(256) void k_generate(CamParams cam1, const JobDev* __restrict__ jobs, int njobs,
                                                  int total, PathBufs pb, float4* __restrict__ rayq,
                                                  uint32_t* __restrict__ count, int unshaded, int whole) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    int lp = p, j = 0;
    CamParams cam = cam1;
    bool inrange = p < total;
    if (MULTI && inrange) {
        while (j + 1 < njobs && jobs[j + 1].path_offset <= p) ++j;
        cam = jobs[j].cam;
        lp = p - jobs[j].path_offset;
        pb.job[p] = j;
    }
    const int P = cam.tile_w * cam.tile_h;
    if (cam.batch > 1 && inrange) {
        const int k = lp / P;   // sample k of the batch: the frame after k passes
        lp -= k * P;
        cam.frame += k;
    }
    bool valid = false;
    int lx = 0, ly = 0;
    if (inrange && lp < P) {
        lx = lp % cam.tile_w;
        ly = lp / cam.tile_w;
        valid = cam.preview ||
                ((cam.tileX * cam.tile_w + lx < cam.width) && (cam.tileY * cam.tile_h + ly < cam.height));
    }
    V3 o = v3(0.f, 0.f, 0.f), d = v3(0.f, 0.f, 1.f);
    uint4 seed = make_uint4(0, 0, 0, 0);
    if (valid) {
        if (cam.preview)
            camera_ray_preview(cam, lx, ly, o, d, seed);
        else
            camera_ray(cam, lx, ly, o, d, seed);
        // shading of depth 0 starts the rest of the path state
        pb.rng[p] = seed;
        if (unshaded) pb.rad[p] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    if (unshaded) return;   // of the whole launch
    uint32_t slot = (uint32_t)p;
    if (whole) {
        if (p == 0) *count = (uint32_t)total;
    } else {
        __shared__ uint32_t app[8];
        slot = block_append(count, valid, app);
    }
    if (valid) {
        rayq[(size_t)slot * 2] = f4(o, __int_as_float(p));
        rayq[(size_t)slot * 2 + 1] = f4(d, 0.f);
    }
}

// generate from caller-given rays and seeds (lfh_path_trace_rays)
__global__ __launch_bounds__(256) void k_generate_rays(const float* __restrict__ rays6, const uint4* __restrict__ seeds,
                                                       int n, PathBufs pb, float4* __restrict__ rayq,
                                                       uint32_t* __restrict__ count, int unshaded) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    bool valid = p < n;
    if (valid) {
        pb.rng[p] = seeds[p];
        if (unshaded) pb.rad[p] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    if (unshaded) return;   // as in k_generate
    if (p == 0) *count = (uint32_t)n;
    if (valid) {
        const float* r = rays6 + (size_t)p * 6;
        rayq[(size_t)p * 2] = make_float4(r[0], r[1], r[2], __int_as_float(p));
        rayq[(size_t)p * 2 + 1] = make_float4(r[3], r[4], r[5], 0.f);
    }
}

// ---- extend: closest hit, lights first (closest_hit.glsl:7-67) ---------------------
LFH_DEV void light_closest(const ShadeScene& sc, V3 o, V3 d, float& t, int& light, float& lpdf) {
    for (int i = 0; i < sc.num_lights; ++i) {
        const float4* lp = sc.lights + (size_t)i * kLightF4;
        float4 a = lp[0], b = lp[1], c = lp[2];
        float type = a.w, area = b.w, radius = c.w;
        if (type == 0.0f) {
            V3 normal = ld3(lp[4]);
            if (dot(normal, d) > 0.0f) continue;
            float dd = rect_hit(lp, o, d);
            if (dd < 0.0f) dd = kInfinity;
            if (dd < t) {
                t = dd;
                float cosTheta = dot(-d, normal);
                lpdf = (t * t) / (area * cosTheta);
                light = i;
            }
        }
        if (type == 1.0f) {
            float dd = sphere_hit(radius, ld3(a), o, d);
            if (dd < 0.0f) dd = kInfinity;
            if (dd < t) {
                t = dd;
                lpdf = (t * t) / area;
                light = i;
            }
        }
    }
}

LFH_DEV bool light_any(const ShadeScene& sc, V3 o, V3 d, float maxDist) {
    for (int i = 0; i < sc.num_lights; ++i) {
        const float4* lp = sc.lights + (size_t)i * kLightF4;
        float4 a = lp[0], c = lp[2];
        if (a.w == 0.0f) {
            float dd = rect_hit(lp, o, d);
            if (dd > 0.0f && dd < maxDist) return true;
        }
        if (a.w == 1.0f) {
            float dd = sphere_hit(c.w, ld3(a), o, d);
            if (dd > 0.0f && dd < maxDist) return true;
        }
    }
    return false;
}

// One wave's share of a ray queue: extension rays write hit records, shadow
// rays clear the weight of their next-event term when they are occluded.
template <bool SHADOW, bool MULTI>
LFH_DEV void trace_queue(const ShadeScene& sc, const JobDev* __restrict__ jobs, const float4* __restrict__ q,
                         int64_t n, float4* __restrict__ hitq, const PathBufs& pb, LaneStack& st,
                         unsigned long long* __restrict__ work, int block, float cull, int* __restrict__ err) {
    const int lane = threadIdx.x & 63;
    WaveFetch fetch;
    fetch.init(n, (int)gridDim.x, kTraceBlock / 64, block, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6));
    if (fetch.idle()) return;   // wave-uniform; the kernel has no block barrier
    TraceState s;
    bool active = false;
    int64_t rid = 0;
    int light = -1;
    float lpdf = 0.f;
    TraceScene ts = sc.tr;
    for (;;) {
        const bool need = !active;
        const uint64_t mask = __ballot(need);
        if (mask) {
            const int64_t id = fetch.next(work, mask, lane, n, (int)gridDim.x, kTraceBlock / 64);
            if (need) {
                rid = id;
                if (rid < n) {
                    float4 a = q[rid * 2], b = q[rid * 2 + 1];
                    V3 o = v3(a.x, a.y, a.z), d = v3(b.x, b.y, b.z);
                    const uint32_t tag = __float_as_uint(a.w);
                    const int pth = SHADOW ? (int)(tag >> 1) : (int)tag;
                    const ShadeScene& S = MULTI ? jobs[pb.job[pth]].sc : sc;
                    ts = S.tr;
                    if (SHADOW) {
                        float maxd = b.w;
                        trace_init(s, st, o, d, 0.0f, maxd, ts.root);
                        if (light_any(S, o, d, maxd)) {
                            s.occluded = true;
                            s.cur = kRefSentinel;  // finishes at once
                        }
                    } else {
                        float t = kInfinity;
                        light = -1;
                        lpdf = 0.f;
                        light_closest(S, o, d, t, light, lpdf);
                        trace_init(s, st, o, d, 0.0f, t, ts.root);
                    }
                    active = true;
                }
            }
        }
        if (__ballot(active) == 0) break;
        if (active) {
            bool done = trace_run<SHADOW, false>(ts, s, st, cull, SHADOW ? kAnySlice : kTraceSlice, nullptr);
            if (done) {
                if (st.overflow) atomicOr(err, 1);
                if (SHADOW) {
                    if (s.occluded) {
                        float4 a = q[rid * 2];
                        uint32_t tag = __float_as_uint(a.w);
                        uint32_t p = tag >> 1, kind = tag & 1u;
                        pb.nee[(size_t)kind * pb.stride + p].w = 0.0f;
                    }
                } else {
                    float4 h0, h1;
                    if (s.bestPrim >= 0) {
                        h0 = make_float4(s.tbest, s.bu, s.bv, __int_as_float(s.bestSlot));
                        h1 = make_float4(__int_as_float(s.bestInst), __int_as_float(s.bestMat), 0.f, __int_as_float(-1));
                    } else {
                        h0 = make_float4(s.tbest, 0.f, 0.f, __int_as_float(-1));
                        h1 = make_float4(__int_as_float(-1), __int_as_float(-1), lpdf, __int_as_float(light));
                    }
                    hitq[rid * 2] = h0;
                    hitq[rid * 2 + 1] = h1;
                }
                active = false;
            }
        }
    }
}

// Extension rays of one depth and shadow rays of the depth before, which do
// not depend on each other, in one launch: a wave that finds no more extension
// rays goes on with shadow rays, so the slowest extension rays and the shadow
// traversal share the chip without a second stream.  The shadow queue's first
// rays go to the waves in reverse order, so that in small wavefronts other
// waves take them.
#ifndef LFH_QUEUE_WAVES
#define LFH_QUEUE_WAVES 6   // queue traversal register budget, waves per SIMD: 7 / 6 / 5: C0 2.84 / 2.41 / 2.39 ms, instanced 1080p frame 22.6 / 19.0 / 19.8 ms, guiding room 7.43 / 6.25 / 6.39 ms, textured tiles 4.53 / 4.13 / 3.93 ms
#endif
template <bool MULTI>
__global__ __launch_bounds__(kTraceBlock, LFH_QUEUE_WAVES) void k_trace_queues(ShadeScene sc, const JobDev* __restrict__ jobs,
                                                              const float4* __restrict__ rayq, const uint32_t* __restrict__ rays,
                                                              unsigned long long* __restrict__ ray_work,
                                                              float4* __restrict__ hitq,
                                                              const float4* __restrict__ shadowq,
                                                              const uint32_t* __restrict__ shadows,
                                                              unsigned long long* __restrict__ shadow_work, PathBufs pb,
                                                              uint32_t* __restrict__ spill, float cull,
                                                              int* __restrict__ err) {
    __shared__ uint32_t stk[kTraceBlock / 64][kLdsStack][64];
    LaneStack st;
    st.lds = (LdsWord*)&stk[threadIdx.x >> 6][0][threadIdx.x & 63];
    st.spill = (GlobalWord*)(spill + ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * kSpillStride);
    st.reset();
    const int block = (int)blockIdx.x;
    trace_queue<false, MULTI>(sc, jobs, rayq, (int64_t)*rays, hitq, pb, st, ray_work, block, cull, err);
    trace_queue<true, MULTI>(sc, jobs, shadowq, (int64_t)*shadows, hitq, pb, st, shadow_work,
                             (int)gridDim.x - 1 - block, cull, err);
}

// ---- shade ------------------------------------------------------------------------
// State word of a path (rad.w): the last surface's material, whether a
// Beer-Lambert coefficient is stored, and which next-event terms of the last
// vertex wait for their shadow rays.
constexpr uint32_t kStateMat = 0x1FFFFFFFu, kStateLight = 1u << 29, kStateEnv = 1u << 30, kStateAbsorb = 1u << 31;

// Adds the last vertex's next-event terms (weight 0 once their shadow ray met
// something).  A vertex with one term stores it times the throughput; one
// with both stores them as they are, and the throughput.
struct NeeTerms {
    float4 env, light, thr;
};
LFH_DEV void load_nee(const PathBufs& pb, int p, uint32_t word, NeeTerms& t) {
    const float4* env = pb.nee + p;
    const float4* light = env + pb.stride;
    if (word & kStateEnv) t.env = *env;
    if (word & kStateLight) t.light = *light;
    if ((word & kStateEnv) && (word & kStateLight)) t.thr = light[pb.stride];
}
LFH_DEV void add_nee(const NeeTerms& t, uint32_t word, V3& rad) {
    if ((word & kStateEnv) && (word & kStateLight)) {
        V3 Li = v3(0.f, 0.f, 0.f);
        if (t.env.w != 0.0f) Li = Li + ld3(t.env);
        if (t.light.w != 0.0f) Li = Li + ld3(t.light);
        rad = rad + Li * ld3(t.thr);
    } else if (word & (kStateEnv | kStateLight)) {
        const float4 c = word & kStateEnv ? t.env : t.light;
        if (c.w != 0.0f) rad = rad + ld3(c);
    }
}
LFH_DEV void combine_nee(const PathBufs& pb, int p, uint32_t word, V3& rad) {
    NeeTerms t = {};
    load_nee(pb, p, word, t);
    add_nee(t, word, rad);
}

// GUIDED: the variant for guided wavefronts (guide sampling, MIS with the
// guide's pdf, training records); unguided wavefronts run the variant without
// that code, which would otherwise hold registers they never use.
//
// Bound by the path state's and the queues' traffic on full queues and by one
// chain of dependent loads and arithmetic on small ones.  Per path and bounce
// of a scene with lights only and no media it moves 144 B in and up to 144 B
// out (192 and 208 B with every array read and written, and 128 B per path
// more by generation): C0 3.07 -> 2.88 ms, guiding room 8.20 -> 7.53 ms,
// instanced 1080p 22.0 -> 20.7 ms, guided frame 14.0 -> 12.7 ms.  Budgeted for
// 3 waves per SIMD (142-167 VGPRs).  Blocks that loop over the queue
// (1536-8192 of them, sparing late depths their empty blocks) need 168 VGPRs with
// spills: C0 2.91-2.95 ms, instanced 21.0-21.2 ms.
#ifndef LFH_SHADE_WAVES
#define LFH_SHADE_WAVES 3
#endif
template <bool MULTI, bool GUIDED>
__global__ __launch_bounds__(256, LFH_SHADE_WAVES) void k_shade(ShadeScene sc1, const JobDev* __restrict__ jobs, int depth,
                                               const float4* __restrict__ rayq,
                                               const float4* __restrict__ hitq, const uint32_t* __restrict__ count,
                                               float4* __restrict__ nextq, float4* __restrict__ shadowq,
                                               uint32_t* __restrict__ next_counts, PathBufs pb, GuideHook gh,
                                               uint32_t* __restrict__ done_counts,
                                               unsigned long long* __restrict__ done_fetch,
                                               unsigned long long* __restrict__ totals) {
    const uint32_t n = *count;
    // the counters of the traversal before the last are read by nothing any more
    if (blockIdx.x == 0) retire_set(done_counts, done_fetch, totals, (int)threadIdx.x);
    __shared__ uint32_t app[8];
    const uint32_t base = blockIdx.x * 256u;
    if (base >= n) return;   // block-uniform
    const uint32_t i = base + threadIdx.x;
    const bool live = i < n;
    bool cont = false;
    bool shEnv = false, shLight = false;
    V3 nextO = v3(0.f, 0.f, 0.f), nextD = v3(0.f, 0.f, 0.f);
    V3 shO = v3(0.f, 0.f, 0.f), shEnvD = v3(0.f, 0.f, 0.f), shLightD = v3(0.f, 0.f, 0.f);
    float shLightMax = 0.f;
    int p = 0;
    if (live) {
        float4 r0 = rayq[(size_t)i * 2], r1 = rayq[(size_t)i * 2 + 1];
        p = __float_as_int(r0.w);
        const ShadeScene& sc = MULTI ? jobs[pb.job[p]].sc : sc1;
        V3 ro = ld3(r0), rd = ld3(r1);
        float4 h0 = hitq[(size_t)i * 2], h1 = hitq[(size_t)i * 2 + 1];
        // a path starts with no radiance and throughput 1
        V3 rad = v3(0.f, 0.f, 0.f), thr = v3(1.f, 1.f, 1.f);
        float prevPdf = 0.f;
        uint32_t word = 0u;
        float2 texc = make_float2(0.f, 0.f);   // last surface's texture coordinate
        if (depth > 0) {
            const float4 r4 = pb.rad[p], t4 = pb.thr[p];
            rad = ld3(r4);
            thr = ld3(t4);
            prevPdf = t4.w;
            word = __float_as_uint(r4.w);
            if (sc.tex) texc = pb.texc[p];
            combine_nee(pb, p, word, rad);
        }
        const bool recorded = GUIDED && gh.train && (p % gh.stride) == gh.phase;
        if (recorded && depth > 0) guide_rec(gh, p, depth - 1)[11] = luminance(rad);
        const int lastMat = (int)(word & kStateMat);
        uint32_t nextWord = 0u;
        const float t = h0.x;
        const int light = __float_as_int(h1.w);
        const int slot = __float_as_int(h0.w);
        if (t == kInfinity) {
            // miss (pathtrace.glsl:223-244)
            if (sc.const_bg) {
                rad = rad + v3(sc.bg[0], sc.bg[1], sc.bg[2]) * thr;
            } else if (sc.use_env) {
                float misWeight = 1.0f;
                float u = (kPi + atan2f(rd.z, rd.x)) * (1.0f / kTwoPi);
                float v = acosf(rd.y) * (1.0f / kPi);
                if (depth > 0) {
                    float lightPdf = EnvPdf(sc, rd);
                    misWeight = powerHeuristic(prevPdf, lightPdf);
                }
                rad = rad + misWeight * tex_linear(sc.hdr_cols, sc.hdr_w, sc.hdr_h, u, v) * thr * sc.hdr_mult;
            }
        } else if (slot < 0 && light >= 0) {
            // analytic light is the closest hit (pathtrace.glsl:246-260): the
            // material fetched is the last surface's (state is not refreshed),
            // its emission map read at that surface's texture coordinate
            Mat m = load_material(sc.materials, lastMat);
            rad = rad + textured_emission(sc, lastMat, texc, m.emission) * thr;
            V3 em = ld3(sc.lights[(size_t)light * kLightF4 + 1]);
            V3 Le = (depth == 0) ? em : powerHeuristic(prevPdf, h1.z) * em;
            rad = rad + Le * thr;
        } else {
            const int inst = __float_as_int(h1.x);
            const int matId = __float_as_int(h1.y);
            float u = h0.y, v = h0.z;
            float w = 1.0f - u - v;
            // hit point: object-space ray point, then the instance transform
            // (closest_hit.glsl:140-143)
            const float4* ip = sc.tr.insts + (size_t)inst * 4;
            float4 i0 = ip[0], i1 = ip[1], i2 = ip[2];
            V3 oo = xform_inv(i0, i1, i2, ro, 1.0f);
            V3 od = xform_inv(i0, i1, i2, rd, 0.0f);
            V3 po = oo + od * t;
            const float4* xp = sc.xforms + (size_t)inst * 4;
            float4 c0 = xp[0], c1 = xp[1], c2 = xp[2], c3 = xp[3];
            V3 fhp = v3(c0.x * po.x + c1.x * po.y + c2.x * po.z + c3.x * 1.0f,
                        c0.y * po.x + c1.y * po.y + c2.y * po.z + c3.y * 1.0f,
                        c0.z * po.x + c1.z * po.y + c2.z * po.z + c3.z * 1.0f);
            // shading normal (pathtrace.glsl:16-37)
            int4 vi = sc.vidx[slot];
            V3 n1 = ld3(sc.normals[vi.x]), n2 = ld3(sc.normals[vi.y]), n3 = ld3(sc.normals[vi.z]);
            V3 nrm = normalize(n1 * w + n2 * u + n3 * v);
            const float4* np = sc.nmats + (size_t)inst * 3;
            float4 m0 = np[0], m1 = np[1], m2 = np[2];
            nrm = normalize(v3(m0.x * nrm.x + m0.y * nrm.y + m0.z * nrm.z, m1.x * nrm.x + m1.y * nrm.y + m1.z * nrm.z,
                               m2.x * nrm.x + m2.y * nrm.y + m2.z * nrm.z));
            Mat m = load_material(sc.materials, matId);
            if (sc.tex) {
                const float2 t1 = sc.uvs[vi.x], t2 = sc.uvs[vi.y], t3 = sc.uvs[vi.z];
                texc = make_float2(t1.x * w + t2.x * u + t3.x * v, t1.y * w + t2.y * u + t3.y * v);
                apply_textures(sc, matId, texc, m, nrm);
            }
            Frame fr;
            fr.N = dot(nrm, rd) <= 0.0f ? nrm : nrm * -1.0f;
            onb(nrm, fr.T, fr.B);
            fr.eta = dot(rd, nrm) < 0.0f ? (1.0f / m.ior) : m.ior;
            // a stored coefficient is not zero; a zero one multiplies by exactly 1
            V3 absorb = v3(0.f, 0.f, 0.f);
            rad = rad + m.emission * thr;
            if ((word & kStateAbsorb) && !(dot(nrm, fr.N) > 0.0f)) {
                absorb = ld3(pb.absorb[p]);
                thr = thr * v3(expf(-absorb.x * t), expf(-absorb.y * t), expf(-absorb.z * t));
            }
            nextWord = (uint32_t)matId;
            uint4 rng = pb.rng[p];
            const float4* lob = gh.lobes + i;
            const size_t lst = (size_t)gh.lobe_stride;
            // the strategy choice depends only on the lobes, never on a sample
            const bool guided = GUIDED && gh.enabled != 0 && gh.sample != 0 && guide_valid(lob, lst);
            // next-event estimation (pathtrace.glsl:126-204)
            const V3 V = -rd;
            // the reference offsets along the unflipped normal (pathtrace.glsl:130), so
            // from behind a one-sided surface its shadow rays start on the far side;
            // the consistent estimator offsets to the side the ray came from
            V3 surfacePos = fhp + (sc.estimator == 1 ? fr.N : nrm) * kEps;
            shO = surfacePos;
            float4 e4 = make_float4(0.f, 0.f, 0.f, 0.f), l4 = make_float4(0.f, 0.f, 0.f, 0.f);
            if (sc.use_env) {
                V3 color, ldir;
                float lightPdf;
                EnvSample(sc, rng, color, ldir, lightPdf);
                float bp;
                V3 f = DisneyEval(m, fr.eta, V, fr.N, ldir, bp);
                if (bp > 0.0f) {
                    const float qp = guided ? (1.0f - kGuideFrac) * bp + kGuideFrac * guide_pdf(lob, ldir, lst) : bp;
                    float mw = powerHeuristic(lightPdf, qp);
                    if (mw > 0.0f) {
                        V3 c = mw * f * fabsf(dot(ldir, fr.N)) * color / lightPdf;
                        e4 = f4(c, 1.0f);
                        shEnv = true;
                        shEnvD = ldir;
                    }
                }
            }
            if (sc.num_lights > 0) {
                int index = (int)(rnd(rng) * (float)sc.num_lights);
                if (index >= sc.num_lights) index = sc.num_lights - 1;
                LightRec lr;
                sampleOneLight(sc, index, surfacePos, lr, rng);
                if (dot(lr.direction, lr.normal) < 0.0f) {
                    float bp;
                    V3 f = DisneyEval(m, fr.eta, V, fr.N, lr.direction, bp);
                    float area = sc.lights[(size_t)index * kLightF4 + 1].w;
                    float weight = 1.0f;
                    if (area > 0.0f)
                        weight = powerHeuristic(
                            lr.pdf, guided ? (1.0f - kGuideFrac) * bp + kGuideFrac * guide_pdf(lob, lr.direction, lst) : bp);
                    if (bp > 0.0f) {
                        V3 c = weight * f * fabsf(dot(fr.N, lr.direction)) * lr.emission / lr.pdf;
                        l4 = f4(c, 1.0f);
                        shLight = true;
                        shLightD = lr.direction;
                        shLightMax = lr.dist - kEps;
                    }
                }
            }
            {
                float4* nee = pb.nee + p;
                if (shEnv && shLight) {
                    nee[0] = e4;
                    nee[pb.stride] = l4;
                    nee[2 * pb.stride] = f4(thr, 1.0f);
                } else if (shEnv) {
                    nee[0] = f4(ld3(e4) * thr, 1.0f);
                } else if (shLight) {
                    nee[pb.stride] = f4(ld3(l4) * thr, 1.0f);
                }
                nextWord |= (shEnv ? kStateEnv : 0u) | (shLight ? kStateLight : 0u);
            }
            // BSDF sampling (pathtrace.glsl:268-291)
            V3 L;
            float pdf, misPdf;
            V3 f;
            if (guided) {
                // one-sample MIS of the guide and the BSDF: the direction comes
                // from either, weighted by the mixture density q = (1-a) p_bsdf + a p_guide
                bool ok = true;
                if (rnd(rng) < kGuideFrac) {
                    const float u0 = rnd(rng), u1 = rnd(rng), u2 = rnd(rng);
                    L = guide_sample(lob, u0, u1, u2, lst);
                } else {
                    float pl;
                    DisneySample(m, fr, V, L, pl, rng);
                    ok = pl > 0.0f;
                }
                float bp;
                f = DisneyEval(m, fr.eta, V, fr.N, L, bp);
                pdf = ok ? (1.0f - kGuideFrac) * bp + kGuideFrac * guide_pdf(lob, L, lst) : 0.0f;
                misPdf = pdf;
            } else {
                f = DisneySample(m, fr, V, L, pdf, rng);
                misPdf = pdf;
                if (sc.estimator == 1 && pdf > 0.0f) {
                    // consistent MIS: the BSDF strategy's density is the lobe
                    // mixture's (disney.glsl:289-290), as in the light-sample weights
                    float bp;
                    DisneyEval(m, fr.eta, V, fr.N, L, bp);
                    misPdf = bp;
                }
            }
            if (dot(fr.N, L) < 0.0f)
                absorb = v3(-logf(m.extinction.x) / m.atDistance, -logf(m.extinction.y) / m.atDistance,
                            -logf(m.extinction.z) / m.atDistance);
            bool alive = pdf > 0.0f;
            const V3 thrBefore = thr;
            if (alive) thr = thr * ((f * fabsf(dot(fr.N, L))) / pdf);
            if (alive && sc.rr && depth >= sc.rr_depth) {
                float q = fminf(fmaxf(thr.x, fmaxf(thr.y, thr.z)) + 0.001f, 0.95f);
                if (rnd(rng) > q) alive = false;
                else thr = thr / q;
            }
            if (alive && depth + 1 < sc.max_depth) {
                cont = true;
                nextD = L;
                nextO = fhp + L * kEps;
            }
            if (recorded) {
                float* r = guide_rec(gh, p, depth);
                r[3] = cont ? 1.0f : 0.0f;
                r[7] = luminance(thrBefore);
                reinterpret_cast<float4*>(r)[3] = make_float4(L.x, L.y, L.z, 0.0f);
            }
            if (cont) {   // a path that ends here is shaded no more
                pb.rng[p] = rng;
                pb.thr[p] = f4(thr, misPdf);
                if (!(absorb.x == 0.0f && absorb.y == 0.0f && absorb.z == 0.0f)) {
                    pb.absorb[p] = f4(absorb, 0.f);
                    nextWord |= kStateAbsorb;
                }
                if (sc.tex) pb.texc[p] = texc;
            }
        }
        pb.rad[p] = f4(rad, __uint_as_float(nextWord));
    }
    const RaySlots slot_of = block_append_rays(next_counts, cont, shEnv, shLight, app);
    const uint32_t s = slot_of.next, se = slot_of.env, sl = slot_of.light;
    if (cont) {
        nextq[(size_t)s * 2] = f4(nextO, __int_as_float(p));
        nextq[(size_t)s * 2 + 1] = f4(nextD, 0.f);
    }
    if (shEnv) {
        shadowq[(size_t)se * 2] = f4(shO, __uint_as_float(((uint32_t)p << 1) | 0u));
        shadowq[(size_t)se * 2 + 1] = f4(shEnvD, kInfinity - kEps);
    }
    if (shLight) {
        shadowq[(size_t)sl * 2] = f4(shO, __uint_as_float(((uint32_t)p << 1) | 1u));
        shadowq[(size_t)sl * 2 + 1] = f4(shLightD, shLightMax);
    }
}

// ---- accumulate: pending NEE + Kahan sum into the frame -----------------------------
template <bool MULTI>
__global__ __launch_bounds__(256) void k_accumulate(PathBufs pb, int total, CamParams cam1, float4* accum1,
                                                    float4* comp1, int kahan1, const JobDev* __restrict__ jobs, int keep) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= total) return;
    CamParams cam = cam1;
    float4* accum = accum1;
    float4* comp = comp1;
    int kahan = kahan1, lp = p;
    if (MULTI) {
        const JobDev& J = jobs[pb.job[p]];
        cam = J.cam;
        accum = J.accum;
        comp = J.comp;
        kahan = J.kahan;
        lp = p - J.path_offset;
    }
    if (lp >= cam.tile_w * cam.tile_h) return;
    const int lx = lp % cam.tile_w, ly = lp / cam.tile_w;
    const int gx = cam.tileX * cam.tile_w + lx, gy = cam.tileY * cam.tile_h + ly;
    if (gx >= cam.width || gy >= cam.height) return;
    const size_t pix = (size_t)gy * cam.width + gx;
    float4 s = accum[pix];
    float4 c = kahan ? comp[pix] : make_float4(0.f, 0.f, 0.f, 0.f);
    // the batch's samples of this pixel, added in frame order as separate passes would
    const int nb = cam.batch > 1 ? cam.batch : 1;
    const int P = cam.tile_w * cam.tile_h;
    // Bound by the chain of a thread's own loads where pixels are few (256 x 256 at 64 samples is one wave per
    // SIMD, 94 % of its time waiting), so four samples' loads are in flight together: 73 -> 54 us, C0 frame 2.30 ->
    // 2.27 ms, 1080p the same.  That takes 84 VGPRs, 5 waves per SIMD instead of 8, which costs more than it gives
    // where pixels are many: 18 passes of a served 720p frame 146 -> 163 us.  A server's wavefronts hold the pixels
    // of all its jobs, so they take one sample at a time.
    constexpr int kAhead = MULTI ? 1 : 4;
    for (int k0 = 0; k0 < nb; k0 += kAhead) {
        const int m = nb - k0 < kAhead ? nb - k0 : kAhead;
        float4 r4[kAhead];
        NeeTerms nee[kAhead];
#pragma unroll
        for (int j = 0; j < kAhead; ++j)
            if (j < m) r4[j] = pb.rad[p + (k0 + j) * P];
#pragma unroll
        for (int j = 0; j < kAhead; ++j)
            if (j < m) load_nee(pb, p + (k0 + j) * P, __float_as_uint(r4[j].w), nee[j]);
#pragma unroll
        for (int j = 0; j < kAhead; ++j) {
            if (j >= m) break;
            V3 rad = ld3(r4[j]);
            add_nee(nee[j], __float_as_uint(r4[j].w), rad);
            if (keep) pb.rad[p + (k0 + j) * P] = f4(rad, 0.f);   // final path radiance (guide training targets)
            if (kahan) {
                float yx = rad.x - c.x, yy = rad.y - c.y, yz = rad.z - c.z;
                float tx = s.x + yx, ty = s.y + yy, tz = s.z + yz;
                c.x = (tx - s.x) - yx;
                c.y = (ty - s.y) - yy;
                c.z = (tz - s.z) - yz;
                s = make_float4(tx, ty, tz, s.w + 1.0f);
            } else {
                s = make_float4(s.x + rad.x, s.y + rad.y, s.z + rad.z, s.w + 1.0f);
            }
        }
    }
    if (kahan) comp[pix] = c;
    accum[pix] = s;
}

// radiance out for lfh_path_trace_rays
__global__ void k_collect(PathBufs pb, int n, float* __restrict__ out) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const float4 r4 = pb.rad[p];
    V3 rad = ld3(r4);
    combine_nee(pb, p, __float_as_uint(r4.w), rad);
    out[(size_t)p * 3] = rad.x;
    out[(size_t)p * 3 + 1] = rad.y;
    out[(size_t)p * 3 + 2] = rad.z;
}

// linear HDR output: (sum - compensation) / samples, bottom-up rows
__global__ void k_output(const float4* __restrict__ accum, const float4* __restrict__ comp, int64_t npix, float inv,
                         float* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= npix) return;
    float4 s = accum[i], c = comp[i];
    out[i * 3] = (s.x - c.x) * inv;
    out[i * 3 + 1] = (s.y - c.y) * inv;
    out[i * 3 + 2] = (s.z - c.z) * inv;
}

__global__ void k_clear_flag(int* f) {
    if (threadIdx.x == 0) f[0] = 0;
}

__global__ void k_clear4(float4* a, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = make_float4(0.f, 0.f, 0.f, 0.f);
}

// ---- per-stage parity kernels ---------------------------------------------------------
LFH_DEV void load_frame(const float* fr, Frame& f, V3& V, int& mat) {
    f.N = v3(fr[0], fr[1], fr[2]);
    f.T = v3(fr[3], fr[4], fr[5]);
    f.B = v3(fr[6], fr[7], fr[8]);
    V = v3(fr[9], fr[10], fr[11]);
    f.eta = fr[12];
    mat = (int)fr[13];
}

__global__ void k_eval_bsdf(ShadeScene sc, const float* frames, const float* L, int n, float* f, float* pdf) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    Frame fr;
    V3 V;
    int mat;
    load_frame(frames + (size_t)i * 16, fr, V, mat);
    Mat m = load_material(sc.materials, mat);
    float p;
    V3 r = DisneyEval(m, fr.eta, V, fr.N, v3(L[i * 3], L[i * 3 + 1], L[i * 3 + 2]), p);
    f[i * 3] = r.x;
    f[i * 3 + 1] = r.y;
    f[i * 3 + 2] = r.z;
    pdf[i] = p;
}

__global__ void k_sample_bsdf(ShadeScene sc, const float* frames, uint4* seeds, int n, float* Lo, float* f,
                              float* pdf) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    Frame fr;
    V3 V;
    int mat;
    load_frame(frames + (size_t)i * 16, fr, V, mat);
    Mat m = load_material(sc.materials, mat);
    uint4 s = seeds[i];
    V3 L = v3(0.f, 0.f, 0.f);
    float p;
    V3 r = DisneySample(m, fr, V, L, p, s);
    seeds[i] = s;
    Lo[i * 3] = L.x;
    Lo[i * 3 + 1] = L.y;
    Lo[i * 3 + 2] = L.z;
    f[i * 3] = r.x;
    f[i * 3 + 1] = r.y;
    f[i * 3 + 2] = r.z;
    pdf[i] = p;
}

__global__ void k_sample_light(ShadeScene sc, const float* pos, uint4* seeds, int n, float* dir, float* nrm,
                               float* em, float* dist, float* pdf) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint4 s = seeds[i];
    int index = (int)(rnd(s) * (float)sc.num_lights);
    if (index >= sc.num_lights) index = sc.num_lights - 1;
    LightRec r;
    sampleOneLight(sc, index, v3(pos[i * 3], pos[i * 3 + 1], pos[i * 3 + 2]), r, s);
    seeds[i] = s;
    dir[i * 3] = r.direction.x; dir[i * 3 + 1] = r.direction.y; dir[i * 3 + 2] = r.direction.z;
    nrm[i * 3] = r.normal.x; nrm[i * 3 + 1] = r.normal.y; nrm[i * 3 + 2] = r.normal.z;
    em[i * 3] = r.emission.x; em[i * 3 + 1] = r.emission.y; em[i * 3 + 2] = r.emission.z;
    dist[i] = r.dist;
    pdf[i] = r.pdf;
}

__global__ void k_sample_env(ShadeScene sc, uint4* seeds, int n, float* dir, float* pdf, float* col) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint4 s = seeds[i];
    V3 c, d;
    float p;
    EnvSample(sc, s, c, d, p);
    seeds[i] = s;
    dir[i * 3] = d.x; dir[i * 3 + 1] = d.y; dir[i * 3 + 2] = d.z;
    col[i * 3] = c.x; col[i * 3 + 1] = c.y; col[i * 3 + 2] = c.z;
    pdf[i] = p;
}

__global__ void k_env_pdf(ShadeScene sc, const float* dir, int n, float* pdf) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    pdf[i] = EnvPdf(sc, v3(dir[i * 3], dir[i * 3 + 1], dir[i * 3 + 2]));
}

}  // namespace lfhd

// ===========================================================================
// host launchers
// ===========================================================================
using namespace lfhd;

static inline int nblk(int64_t n, int b = 256) { return (int)((n + b - 1) / b); }

hipError_t pt_reset(uint32_t* counters, unsigned long long* work, hipStream_t s) {
    hipLaunchKernelGGL(k_pt_reset, dim3(1), dim3(64), 0, s, counters, work);
    return hipGetLastError();
}

hipError_t pt_generate(const CamParams& cam, int max_depth, const PathBufs& pb, float4* rayq, uint32_t* count,
                       hipStream_t s) {
    int P = cam.tile_w * cam.tile_h * (cam.batch > 1 ? cam.batch : 1);
    const int whole = cam.preview || ((cam.tileX + 1) * cam.tile_w <= cam.width && (cam.tileY + 1) * cam.tile_h <= cam.height);
    hipLaunchKernelGGL(k_generate<false>, dim3(nblk(P)), dim3(256), 0, s, cam, (const JobDev*)nullptr, 1, P, pb, rayq,
                       count, max_depth <= 0, whole);
    return hipGetLastError();
}

hipError_t pt_generate_multi(const JobDev* jobs, int njobs, int total, int max_depth, const PathBufs& pb, float4* rayq,
                             uint32_t* count, hipStream_t s) {
    CamParams dummy{};
    hipLaunchKernelGGL(k_generate<true>, dim3(nblk(total)), dim3(256), 0, s, dummy, jobs, njobs, total, pb, rayq,
                       count, max_depth <= 0, 1);   // every job renders its whole frame
    return hipGetLastError();
}

hipError_t pt_generate_rays(const float* rays6, const uint4* seeds, int n, int max_depth, const PathBufs& pb, float4* rayq,
                            uint32_t* count, hipStream_t s) {
    hipLaunchKernelGGL(k_generate_rays, dim3(nblk(n)), dim3(256), 0, s, rays6, seeds, n, pb, rayq, count,
                       max_depth <= 0);
    return hipGetLastError();
}

namespace {

// One wavefront's bounces: per depth one traversal launch (this depth's
// extension rays, the last depth's shadow rays), guide inference for guided
// wavefronts, and shading; a last traversal takes the last shadow rays.
template <bool MULTI>
hipError_t bounces(const ShadeScene& sc, const JobDev* jobs, int max_depth, const PtQueues& q, const PathBufs& pb,
                   const GuideHook& gh, const lfhd::GuideDev* gd, const ShadeScene& guide_sc, hipStream_t s) {
    if (max_depth <= 0) return hipSuccess;
    for (int d = 0;; ++d) {
        uint32_t* counts = set_counts(q.counts, d);
        unsigned long long* fetch = set_fetch(q.work, d);
        hipLaunchKernelGGL((k_trace_queues<MULTI>), dim3(q.grid_blocks), dim3(kTraceBlock), 0, s, sc, jobs,
                           q.rayq[d & 1], counts, fetch, q.hitq, q.shadowq, counts + 1, fetch + kFetchWords, pb,
                           q.spill, q.cull, q.err);
        if (d == max_depth) break;
        if (gh.enabled) {
            hipError_t e = guide_infer_queue(*gd, guide_sc, q.rayq[d & 1], q.hitq, counts, q.maxq, gh, d,
                                             const_cast<float4*>(gh.lobes), s);
            if (e != hipSuccess) return e;
        }
        const auto shade = gh.enabled ? k_shade<MULTI, true> : k_shade<MULTI, false>;
        const int done = d + kQueueSets - 1;   // the set of traversal d - 1
        hipLaunchKernelGGL(shade, dim3(nblk(q.maxq)), dim3(256), 0, s, sc, jobs, d, q.rayq[d & 1], q.hitq, counts,
                           q.rayq[(d + 1) & 1], q.shadowq, set_counts(q.counts, d + 1), pb, gh,
                           set_counts(q.counts, done), set_fetch(q.work, done), q.work + kWorkTotals);
    }
    return hipGetLastError();
}

}  // namespace

hipError_t pt_bounces(const ShadeScene& sc, int max_depth, const PtQueues& q, const PathBufs& pb, const GuideHook& gh,
                      const lfhd::GuideDev* gd, hipStream_t s) {
    return bounces<false>(sc, nullptr, max_depth, q, pb, gh, gd, sc, s);
}

hipError_t pt_bounces_multi(const JobDev* jobs, int max_depth, const PtQueues& q, const PathBufs& pb,
                            const GuideHook& gh, const lfhd::GuideDev* gd, const ShadeScene* guide_sc,
                            hipStream_t s) {
    // every job of a guided wavefront draws on one scene (the guide's)
    const ShadeScene none{};
    return bounces<true>(none, jobs, max_depth, q, pb, gh, gd, guide_sc ? *guide_sc : none, s);
}

hipError_t pt_accumulate_multi(const JobDev* jobs, int total, const PathBufs& pb, bool keep_radiance, hipStream_t s) {
    CamParams dummy{};
    hipLaunchKernelGGL(k_accumulate<true>, dim3(nblk(total)), dim3(256), 0, s, pb, total, dummy, (float4*)nullptr,
                       (float4*)nullptr, 0, jobs, keep_radiance ? 1 : 0);
    return hipGetLastError();
}

hipError_t pt_accumulate(const PathBufs& pb, const CamParams& cam, float4* accum, float4* comp, int kahan,
                         bool keep_radiance, hipStream_t s) {
    int P = cam.tile_w * cam.tile_h;
    hipLaunchKernelGGL(k_accumulate<false>, dim3(nblk(P)), dim3(256), 0, s, pb, P, cam, accum, comp, kahan,
                       (const JobDev*)nullptr, keep_radiance ? 1 : 0);
    return hipGetLastError();
}

hipError_t pt_collect(const PathBufs& pb, int n, float* out, hipStream_t s) {
    hipLaunchKernelGGL(k_collect, dim3(nblk(n)), dim3(256), 0, s, pb, n, out);
    return hipGetLastError();
}

hipError_t pt_output(const float4* accum, const float4* comp, int64_t npix, float inv, float* out, hipStream_t s) {
    hipLaunchKernelGGL(k_output, dim3(nblk(npix)), dim3(256), 0, s, accum, comp, npix, inv, out);
    return hipGetLastError();
}

hipError_t pt_clear4(float4* a, int64_t n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_clear4, dim3(nblk(n)), dim3(256), 0, s, a, n);
    return hipGetLastError();
}

hipError_t pt_clear_flag(int* flag, hipStream_t s) {
    hipLaunchKernelGGL(k_clear_flag, dim3(1), dim3(64), 0, s, flag);
    return hipGetLastError();
}

int pt_trace_grid_blocks() {
    static int blocks = 0;
    if (blocks == 0) {
        int dev = 0, a = 0, b = 0;
        hipGetDevice(&dev);
        hipDeviceProp_t prop;
        hipGetDeviceProperties(&prop, dev);
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&a, (const void*)k_trace_queues<true>, kTraceBlock, 0) !=
                hipSuccess || a <= 0)
            a = 4;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, (const void*)k_trace_queues<false>, kTraceBlock, 0) !=
                hipSuccess || b <= 0)
            b = 4;
        blocks = (a > b ? a : b) * prop.multiProcessorCount;
    }
    return blocks;
}

hipError_t stage_eval_bsdf(const ShadeScene& sc, const float* fr, const float* L, int n, float* f, float* pdf,
                           hipStream_t s) {
    hipLaunchKernelGGL(k_eval_bsdf, dim3(nblk(n)), dim3(256), 0, s, sc, fr, L, n, f, pdf);
    return hipGetLastError();
}
hipError_t stage_sample_bsdf(const ShadeScene& sc, const float* fr, uint4* seeds, int n, float* L, float* f,
                             float* pdf, hipStream_t s) {
    hipLaunchKernelGGL(k_sample_bsdf, dim3(nblk(n)), dim3(256), 0, s, sc, fr, seeds, n, L, f, pdf);
    return hipGetLastError();
}
hipError_t stage_sample_light(const ShadeScene& sc, const float* pos, uint4* seeds, int n, float* dir, float* nrm,
                              float* em, float* dist, float* pdf, hipStream_t s) {
    hipLaunchKernelGGL(k_sample_light, dim3(nblk(n)), dim3(256), 0, s, sc, pos, seeds, n, dir, nrm, em, dist, pdf);
    return hipGetLastError();
}
hipError_t stage_sample_env(const ShadeScene& sc, uint4* seeds, int n, float* dir, float* pdf, float* col,
                            hipStream_t s) {
    hipLaunchKernelGGL(k_sample_env, dim3(nblk(n)), dim3(256), 0, s, sc, seeds, n, dir, pdf, col);
    return hipGetLastError();
}
hipError_t stage_env_pdf(const ShadeScene& sc, const float* dir, int n, float* pdf, hipStream_t s) {
    hipLaunchKernelGGL(k_env_pdf, dim3(nblk(n)), dim3(256), 0, s, sc, dir, n, pdf);
    return hipGetLastError();
}
