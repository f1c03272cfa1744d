// Device-side layouts and helpers shared by the gfx950 kernels.
//
// All device code is compiled with -ffp-contract=off: traversal and
// intersection arithmetic is evaluated in exactly the order written (one IEEE
// rounding per operation), which is what makes hit ids bit-exact against the
// CPU restatement of shaders/common/closest_hit.glsl.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define LFH_DEV __device__ __forceinline__
#define LFH_HD __host__ __device__ __forceinline__

namespace lfhd {

constexpr float kInfinity = 1000000.0f;   // globals.glsl:8
constexpr float kEps = 0.001f;            // globals.glsl:9
constexpr float kPi = 3.14159265358979323f;
constexpr float kTwoPi = 6.28318530717958648f;

// ---- child references (32 bit) ---------------------------------------------
//   internal node : index (< 2^30)
//   BLAS leaf     : 0x80000000 | (count << 28) | first triangle slot (< 2^28)
//   TLAS leaf     : 0x40000000 | instance index (< 2^30)
//   sentinel      : 0xFFFFFFFF (absent child; end marker of the stack)
//   return marker : 0xFFFFFFFE (on the stack below a BLAS; no leaf has this ref:
//                   7 triangles from slot 2^28 - 2)
constexpr uint32_t kRefSentinel = 0xFFFFFFFFu;
constexpr uint32_t kRefReturn = 0xFFFFFFFEu;
constexpr uint32_t kRefLeafBit = 0x80000000u;
constexpr uint32_t kRefInstBit = 0x40000000u;
LFH_HD bool ref_is_node(uint32_t r) { return r < kRefInstBit; }
LFH_HD bool ref_is_leaf(uint32_t r) { return (r & kRefLeafBit) != 0; }
LFH_HD bool ref_is_inst(uint32_t r) { return (r & 0xC0000000u) == kRefInstBit; }
LFH_HD uint32_t leaf_first(uint32_t r) { return r & 0x0FFFFFFFu; }
LFH_HD uint32_t leaf_count(uint32_t r) { return (r >> 28) & 0x7u; }
LFH_HD uint32_t make_leaf(uint32_t first, uint32_t count) { return kRefLeafBit | (count << 28) | first; }
LFH_HD uint32_t make_inst(uint32_t inst) { return kRefInstBit | inst; }

// ---- packed layouts ------------------------------------------------------------
// Internal BVH4 node, 128 B (one L2 line), the four child boxes in the parent
// as structure of arrays, child k in lane k of each float4:
//   f4[0..2] = min.x, min.y, min.z    f4[3..5] = max.x, max.y, max.z
//   f4[6]    = as_float(child refs)   f4[7]    = 0
//   an absent child has ref kRefSentinel and the empty box (+inf, -inf), which
//   no ray with finite nonzero inv enters.
// (Host intermediate: the BVH2 node of 64 B with both child boxes,
//  (lmin, lmax, rmin, rmax, left ref, right ref), collapsed into BVH4 nodes.)
// Triangle, 48 B, in vert_indices slot order:
//   f4[0] = (v0.xyz, as_float(prim)),  f4[1] = (e0 = v1 - v0, as_float(slot)),
//   f4[2] = (e1 = v2 - v0, 0)
// Instance, 64 B: rows 0..2 of inverse(M) as (inv[0][r], inv[1][r], inv[2][r],
//   inv[3][r]) and (as_float(blas ref), as_float(material), as_float(index), 0).

// Traversal stack: the first kLdsStack entries of a lane live in LDS, deeper
// ones in a per-lane global area of kSpillStride entries.
#ifndef LFH_LDS_STACK
#define LFH_LDS_STACK 16   // 24 entries: any hit 2207 against 2116 us (8.4M incoherent rays), closest hit the same
#endif
#ifndef LFH_TRACE_WAVES
// Waves per SIMD the ray-batch closest-hit kernel is register-budgeted for (87 VGPRs, no
// spills).  16.8M rays, 1M-triangle soup: 5 waves 6.22 ms, 6 waves 6.23 ms.
#define LFH_TRACE_WAVES 5
#endif
#ifndef LFH_ANYHIT_WAVES
// the same for any hit (80 VGPRs): 5 and 6 waves 0.794 ms for 2.1M rays
#define LFH_ANYHIT_WAVES 6
#endif
// Work counters of the persistent traversal kernels: a queue's ray ids are
// split into kFetchSlices contiguous slices, each with its own counter
// kFetchStride 64-bit words (256 B) from the next.  A wavefront keeps
// kQueueSets sets of queue counters in turn, traversal d using set
// d % kQueueSets: the ray counts (extension, shadow) and both queues' fetch
// counters; two running ray totals follow the fetch counters at kWorkTotals.
#ifndef LFH_FETCH_SLICES
#define LFH_FETCH_SLICES 8
#endif
constexpr int kFetchSlices = LFH_FETCH_SLICES;
constexpr int kFetchStride = 32;
constexpr int kFetchWords = kFetchSlices * kFetchStride;
constexpr int kQueueSets = 3;
constexpr int kWorkTotals = kQueueSets * 2 * kFetchWords;
constexpr int kWorkWords = kWorkTotals + 8;
#ifndef LFH_TRACE_SLICE
// 16 / 24 / 32 / 48 steps: 16.8M closest hits 5.90 / 5.92 / 5.92 / 6.09 ms, instanced 1080p frame
// 22.0 / 22.1 / 22.3 / 22.6 ms, C0 3.14 / 3.10 / 3.10 / 3.09 ms, served mix 5.04 / 4.93 / 4.98 / 4.94 ms
#define LFH_TRACE_SLICE 24
#endif
constexpr int kTraceSlice = LFH_TRACE_SLICE;  // traversal steps between refills of a wave's idle lanes
#ifndef LFH_ANY_SLICE
// the same for any-hit queries: 8 / 12 / 16 / 24 / 32 steps 1003 / 798 / 794 / 797 / 989 us for 2.1M rays
#define LFH_ANY_SLICE 16
#endif
constexpr int kAnySlice = LFH_ANY_SLICE;
constexpr int kLdsStack = LFH_LDS_STACK;  // LDS entries per lane
constexpr int kTraceBlock = 256;        // threads per traversal block (4 wave64)
constexpr uint32_t kSpillStride = 128;  // global entries per lane; the most a scene's traversal may need

struct TraceScene {
    const float4* nodes;
    const float4* tris;
    const float4* insts;
    uint32_t root;
    uint32_t spill_stride;   // entries per lane in the spill area
};

struct V3 {
    float x, y, z;
};
LFH_HD V3 v3(float x, float y, float z) { return V3{x, y, z}; }
LFH_HD V3 operator+(V3 a, V3 b) { return v3(a.x + b.x, a.y + b.y, a.z + b.z); }
LFH_HD V3 operator-(V3 a, V3 b) { return v3(a.x - b.x, a.y - b.y, a.z - b.z); }
LFH_HD V3 operator-(V3 a) { return v3(-a.x, -a.y, -a.z); }
LFH_HD V3 operator*(V3 a, V3 b) { return v3(a.x * b.x, a.y * b.y, a.z * b.z); }
LFH_HD V3 operator*(V3 a, float s) { return v3(a.x * s, a.y * s, a.z * s); }
LFH_HD V3 operator*(float s, V3 a) { return v3(s * a.x, s * a.y, s * a.z); }
LFH_HD V3 operator/(V3 a, float s) { return v3(a.x / s, a.y / s, a.z / s); }
LFH_HD V3 operator/(V3 a, V3 b) { return v3(a.x / b.x, a.y / b.y, a.z / b.z); }
// dot(a, b) = (a.x*b.x + a.y*b.y) + a.z*b.z
LFH_HD float dot(V3 a, V3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
LFH_HD V3 cross(V3 a, V3 b) {
    return v3(a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x);
}
#if defined(__HIP__)
// normalize(v) = v / sqrt(dot(v, v))
LFH_DEV V3 normalize(V3 a) {
    float l = sqrtf(dot(a, a));
    return v3(a.x / l, a.y / l, a.z / l);
}
LFH_DEV float length(V3 a) { return sqrtf(dot(a, a)); }
#endif
LFH_HD V3 xyz(float4 f) { return v3(f.x, f.y, f.z); }

#if defined(__HIP__)
LFH_DEV float as_f(uint32_t u) { return __uint_as_float(u); }
LFH_DEV uint32_t as_u(float f) { return __float_as_uint(f); }

// ---- slab test (intersection.glsl:56-72) -------------------------------------
// Order key of a box the ray enters in front of its origin (AABBIntersect > 0)
// at a distance t0 <= lim, infinity for any other box.  min/max are IEEE
// minNum/maxNum.  Both lower limits go into max(t0, the least positive float),
// for closest hit both upper ones into min(t1, lim), so one comparison
// decides (two for any hit).  min(t1, lim) also asks for a positive lim, so for
// closest hit lim is at least the least positive float: at best distance 0 a
// box around the origin still passes.
//
// The key decides how many nodes a ray visits, not what it hits:
//   closest hit  t0, also where it is negative: of the boxes around the origin
//                the one reaching furthest back goes first.  Ordering those by
//                their exit t1 (AABBIntersect's value) costs an incoherent ray
//                twice the visits: 8.4M rays 9.01 ms against 3.81 ms, and 3.85 ms
//                with all of them at key 0.
//   any hit      the longest stretch inside the box first, where a hit is
//                likeliest: 8.4M rays 2.20 ms against 3.13 ms by t0, 2.79 ms by
//                AABBIntersect's value, 3.47 ms by t1, 2.53 ms by -t1.
constexpr float kLeastPositive = 1.401298464e-45f;
template <bool ANY>
LFH_DEV float slab_entry(float nx, float ny, float nz, float fx, float fy, float fz, float lim) {
    const float t0 = fmaxf(nx, fmaxf(ny, nz));
    const float none = __builtin_inff();
    if (ANY) {
        const float c0 = fmaxf(t0, kLeastPositive);
        const float t1 = fminf(fx, fminf(fy, fz));
        return t1 >= c0 && c0 <= lim ? c0 - t1 : none;
    }
    const float t1 = fminf(fx, fminf(fy, fminf(fz, lim)));
    return t1 >= fmaxf(t0, kLeastPositive) ? t0 : none;
}
// The near and far plane of each axis already chosen by the ray's octant
// (finite inv): the same t0 / t1, bit for bit, without the per-axis min / max.
template <bool ANY>
LFH_DEV float slab_octant(V3 bnear, V3 bfar, V3 o, V3 inv, float lim) {
    return slab_entry<ANY>((bnear.x - o.x) * inv.x, (bnear.y - o.y) * inv.y, (bnear.z - o.z) * inv.z,
                      (bfar.x - o.x) * inv.x, (bfar.y - o.y) * inv.y, (bfar.z - o.z) * inv.z, lim);
}
template <bool ANY>
LFH_DEV float slab(V3 bmin, V3 bmax, V3 o, V3 inv, float lim) {
    const float fx = (bmax.x - o.x) * inv.x, fy = (bmax.y - o.y) * inv.y, fz = (bmax.z - o.z) * inv.z;
    const float nx = (bmin.x - o.x) * inv.x, ny = (bmin.y - o.y) * inv.y, nz = (bmin.z - o.z) * inv.z;
    return slab_entry<ANY>(fminf(fx, nx), fminf(fy, ny), fminf(fz, nz), fmaxf(fx, nx), fmaxf(fy, ny), fmaxf(fz, nz), lim);
}

// ---- Moller-Trumbore as written in closest_hit.glsl:119-134 ------------------
// No epsilons; uvt.xyz / det as three IEEE divisions; w = (1 - u) - v.
// Returns true and fills (t, u, v) when u, v, w, t >= 0.
LFH_DEV bool tri_test(V3 o, V3 d, V3 v0, V3 e0, V3 e1, float* t, float* u, float* v) {
    V3 pv = cross(d, e1);
    float det = dot(e0, pv);
    V3 tv = o - v0;
    V3 qv = cross(tv, e0);
    float nu = dot(tv, pv);
    float nv = dot(d, qv);
    float nt = dot(e1, qv);
    float uu = nu / det, vv = nv / det, tt = nt / det;
    float ww = 1.0f - uu - vv;
    *t = tt;
    *u = uu;
    *v = vv;
    return uu >= 0.f && vv >= 0.f && tt >= 0.f && ww >= 0.f;
}

// Ray into instance space: inverse(M) * vec4(p, w) with the product summed
// column by column: ((c0*x + c1*y) + c2*z) + c3*w.
LFH_DEV V3 xform_inv(const float4& r0, const float4& r1, const float4& r2, V3 p, float w) {
    return v3(r0.x * p.x + r0.y * p.y + r0.z * p.z + r0.w * w,
              r1.x * p.x + r1.y * p.y + r1.z * p.z + r1.w * w,
              r2.x * p.x + r2.y * p.y + r2.z * p.z + r2.w * w);
}

LFH_DEV V3 rcp3(V3 d) { return v3(1.0f / d.x, 1.0f / d.y, 1.0f / d.z); }
#endif  // __HIP__

}  // namespace lfhd
