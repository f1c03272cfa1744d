// Two-level BVH traversal for gfx950: closest hit and any hit.
//
// Visit order and acceptance follow ClosestHit / AnyHit
// (shaders/common/closest_hit.glsl:69-201, anyhit.glsl:48-170):
//   * start at the top-level node without testing its box;
//   * at an internal node test the child boxes, descend into the nearest one
//     and push the others (the nodes are a BVH4 collapsed from the
//     reference's binary tree with the same boxes, so the same triangles are
//     reached);
//   * at a TLAS leaf move the ray into instance space with the inverse
//     transform, push a return marker and continue at the BLAS root;
//   * at a BLAS leaf run Moller-Trumbore on each triangle.
// Differences, all result-preserving:
//   * child boxes whose entry distance exceeds the current best t (times a
//     safety factor `cull`, default 1 + 2^-10) are skipped; the reference
//     visits them and rejects all their triangles;
//   * exact-t ties between triangles go to the lowest (instance, prim) pair
//     instead of the first one found, so the answer does not depend on visit
//     order;
//   * the per-lane stack keeps its first kLdsStack entries in LDS and deeper
//     ones in a per-lane global area.
#pragma once
#include "dev_common.h"

namespace lfhd {


// Entry e of a lane's stack is in LDS for e < kLdsStack (at lds[e * 64]) and in
// the lane's global area above that.  Entry 0 is the end marker kRefSentinel.
// The address spaces are part of the types: a pop that selects between two
// generic pointers becomes one flat load, which waits for both memories.
typedef __attribute__((address_space(3))) uint32_t LdsWord;
typedef __attribute__((address_space(1))) uint32_t GlobalWord;
struct LaneStack {
    LdsWord* lds;       // this lane's LDS column
    GlobalWord* spill;  // this lane's global area
    int sp;           // entries
    bool overflow;
    LFH_DEV void reset() {
        lds[0] = kRefSentinel;
        sp = 1;
        overflow = false;
    }
    LFH_DEV void push(uint32_t v) {
        if (sp < kLdsStack) lds[sp * 64] = v;
        else if (sp < kLdsStack + (int)kSpillStride) spill[sp - kLdsStack] = v;
        else { overflow = true; return; }
        sp++;
    }
    LFH_DEV uint32_t pop() {
        sp--;
        uint32_t r = lds[(sp < kLdsStack ? sp : 0) * 64];
        if (__builtin_expect(sp >= kLdsStack, 0)) r = spill[sp - kLdsStack];
        return r;
    }
};

// Work fetch of the persistent traversal kernels.  A queue's ids are split
// into kFetchSlices contiguous slices; a wave belongs to slice blockIdx.x %
// kFetchSlices (blocks go to the XCDs in turn, so each XCD starts on its own
// run of neighbouring rays).
//
// A wave's first ids are its own by position, without an atomic.  In a queue
// of at most kFetchChunk ids per wave of the launch every wave owns the even
// share, at least kFetchMin ids: such queues (late bounces, small frames,
// small ray batches) take no atomics at all and spread over as many waves as
// they can, so that few lanes of a wave diverge.  In a larger queue every wave
// owns one chunk in each of the first `rounds` rounds over its slice, so the
// waves of an XCD still sweep the slice together.
// The ids behind the owned ones are handed out dynamically, kFetchChunk at a
// time, by a counter per slice (kFetchStride words apart): atomics to one
// counter serialise across the XCDs, at about 11 ns each, and a wave waits for
// the round trip of its own.  When a slice runs out the wave moves to the
// next one, looking at its counter before the first addition to it, and after
// finding every slice exhausted it has no more work.  Counters only grow, so a
// slice once exhausted stays so, and every id below n is handed out exactly
// once.
#ifndef LFH_FETCH_CHUNK
// 64 / 128 / 192 / 256: 16.8M-ray closest hit 5.95 / 5.59 / 5.44 / 5.41 ms, 2M-ray any hit 765 / 749 / 781 / 787 us,
// 8.4M incoherent rays 3.50 / 3.52 / 3.57 / 3.58 ms, C0 2.41 / 2.31 / 2.33 / 2.32 ms, viewer 720p 9.52 / 9.31 / 9.42 /
// 9.52 ms, served mix 4.68 / 4.56 / 4.61 / 4.65 ms: longer chunks save atomics, and leave the waves that end a queue
// with more rays each.
// The length is also the line between queues that are all owned and queues with dynamic fetches (closest hit: 328k
// rays at 64, 655k at 128; any hit 393k and 786k).  Batches of incoherent / pinhole rays, 1M triangles, closest hit,
// 64 against 128:
//   300k          293 / 196 us against 293 / 206    both lengths all owned
//   400k          361 / 275 against 340 / 252       between the lines
//   650k          472 / 323 against 437 / 339
//   780k          508 / 369 against 569 / 418       just past the longer line: few waves end with a chunk more
//   1.3M          725 / 487 against 724 / 501
//   2M            986 / 653 against 1012 / 680
//   from 3.2M on  equal to 1 %
// Any hit 0.95-1.10 times its time with 128 between the lines, 0.92-1.05 up to 2M.  128 for all, because the
// path tracer's queues prefer it at every depth (64: C0 2.37 against 2.27 ms, viewer 9.70 against 9.28, and 2 %
// longer in both with 64 only for queues of one to four times the line).
#define LFH_FETCH_CHUNK 128
#endif
#ifndef LFH_FETCH_MIN
// at least 1 / 4 / 16 rays per wave, closest hit, 1M triangles: 1k incoherent rays 93 / 123 / 137 us, 5k 118 / 128 /
// 155, 20k 179 / 179 / 187, 50k 195 / 195 / 189; 20k triangles, pinhole: 1k 57 / 73 / 74, 20k 71 / 71 / 61, 50k 88 / 88 /
// 73 (coherent rays of a wave cost little more than one).  A pick of 1021 rays 67 / 77 / 92 us, textured 128 x 128
// tiles 172 / 165 / 164 us per pass, viewer 9.28 / 9.24 / 9.37 ms: 1 for the smallest calls.
#define LFH_FETCH_MIN 1
#endif
#ifndef LFH_FETCH_OWNED
// eighths of a large queue owned by position: 0 / 4 / 6: viewer 9.36 / 9.22 / 9.30 ms, C0 2.27 / 2.27 / 2.28; batches of
// 0.9M-8.4M rays the same with 0, 2 and 4, and up to 6 % longer with 6 (8.4M pinhole rays, 20k triangles 1.53 ->
// 1.62 ms: owned chunks are never passed on)
#define LFH_FETCH_OWNED 4
#endif
constexpr int kFetchChunk = LFH_FETCH_CHUNK;
constexpr int kFetchMin = LFH_FETCH_MIN;

// Lane 0's value in a scalar register.
LFH_DEV unsigned long long wave_first(unsigned long long v) {
    const uint32_t lo = __builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
    return (unsigned long long)hi << 32 | lo;
}
// Set bits of `mask` below this lane.
LFH_DEV int lane_rank(uint64_t mask) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

struct WaveFetch {
    int64_t base = 0;   // next id of the wave's reservation (same in every lane)
    int64_t own = 0;    // first id of the wave's next owned chunk
    int left = 0;       // ids left in the reservation
    int rounds = 0;     // owned chunks not yet taken
    int slice = 0;      // current slice
    int tried = 0;      // slices found exhausted
    int owned = 0;      // ids each wave of the launch owns
    bool probe = false; // look at the slice's counter before adding to it

    static LFH_HD int waves_of(int s, int blocks, int waves) { return (blocks - s + kFetchSlices - 1) / kFetchSlices * waves; }
    // blocks x waves: the launch; block, wave: this wave's place in it
    LFH_DEV void init(int64_t n, int blocks, int waves, int block, int wave) {
        const int64_t all = (int64_t)blocks * waves;
        slice = block % kFetchSlices;
        const int64_t lo = n * slice / kFetchSlices, hi = n * (slice + 1) / kFetchSlices;
        const int64_t idx = (int64_t)(block / kFetchSlices) * waves + wave;
        if (n <= all * kFetchChunk) {
            const int share = (int)((n + all - 1) / all);
            owned = share < kFetchMin ? kFetchMin : share;
            base = lo + idx * owned;
            left = base >= hi ? 0 : (hi - base < owned ? (int)(hi - base) : owned);
            // equal waves in every slice: nothing is left to fetch
            if (blocks % kFetchSlices == 0) tried = kFetchSlices;
        } else {
            const int64_t r = n / (all * kFetchChunk) * LFH_FETCH_OWNED / 8;
            rounds = r < 1 ? 1 : (r > (1 << 20) ? 1 << 20 : (int)r);
            owned = rounds * kFetchChunk;
            own = lo + idx * kFetchChunk;
        }
    }
    // Nothing owned and nothing to fetch.
    LFH_DEV bool idle() const { return left == 0 && rounds == 0 && tried == kFetchSlices; }
    // Ids for the lanes in `mask` (nonzero; called by every lane of the wave),
    // in rank order within the mask; n (no work) for lanes left without one.
    LFH_DEV int64_t next(unsigned long long* ctr, uint64_t mask, int lane, int64_t n, int blocks, int waves) {
        const int want = __popcll(mask);
        const int rank = lane_rank(mask);
        if (left >= want) {
            const int64_t id = base + rank;
            base += want;
            left -= want;
            return id;
        }
        const int old = left;
        int64_t id = rank < old ? base + rank : n;
        left = 0;
        while (rounds > 0 || tried < kFetchSlices) {
            const int64_t lo = n * slice / kFetchSlices, hi = n * (slice + 1) / kFetchSlices;
            int64_t start;
            if (rounds > 0) {
                start = own;
                own += (int64_t)waves_of(slice, blocks, waves) * kFetchChunk;
                --rounds;
                if (start >= hi) {
                    rounds = 0;
                    continue;
                }
            } else {
                start = lo + (int64_t)waves_of(slice, blocks, waves) * owned;
                if (start < hi) {
                    unsigned long long* c = ctr + (size_t)slice * kFetchStride;
                    unsigned long long nb = 0;
                    if (lane == 0) {
                        if (probe) nb = __hip_atomic_load(c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        if (start + (int64_t)nb < hi) nb = atomicAdd(c, (unsigned long long)kFetchChunk);
                    }
                    start += (int64_t)wave_first(nb);
                }
                if (start >= hi) {
                    slice = slice + 1 == kFetchSlices ? 0 : slice + 1;
                    ++tried;
                    probe = true;
                    continue;
                }
                probe = false;
            }
            const int avail = hi - start < kFetchChunk ? (int)(hi - start) : kFetchChunk;
            const int used = want - old < avail ? want - old : avail;
            if (rank >= old && rank < old + used) id = start + (rank - old);
            base = start + used;
            left = avail - used;
            break;
        }
        return id;
    }
};

struct TraceStats {
    int nint, ntri, ninst;
};

// Per-lane traversal state, resumable (the persistent kernels run it in
// bounded slices so idle lanes can be refilled).
struct TraceState {
    V3 O, D, invD;      // world ray
    V3 o, d, inv;       // current-space ray
    float tmin, tbest;
    uint32_t cur;
    int curInst, curMat;
    int bestPrim, bestInst, bestMat, bestSlot;
    float bu, bv;
    bool occluded;
    uint32_t oct;   // near-plane byte offsets x | y << 8 | z << 16, bit 24: inv has an infinite or zero component
};

// The near-side plane of each axis follows from the sign of inv: min at
// bytes 0/16/32 of a node, max at 48/64/80.  For finite inv the near plane's
// distance equals the per-axis min of the two (t = (b - o) inv is monotonic
// in b), bit for bit; an infinite component (d = +-0) can make one of them
// 0 * inf = NaN, which the min/max form resolves differently, so such rays
// take the min/max form (and so do rays with a zero component of inv, whose
// distances to the infinite planes of an absent child would be NaN).
LFH_DEV void set_octant(TraceState& s) {
    const uint32_t nx = signbit(s.inv.x) ? 48u : 0u, ny = signbit(s.inv.y) ? 64u : 16u,
                   nz = signbit(s.inv.z) ? 80u : 32u;
    const float big = fmaxf(fmaxf(fabsf(s.inv.x), fabsf(s.inv.y)), fabsf(s.inv.z));
    const float small = fminf(fminf(fabsf(s.inv.x), fabsf(s.inv.y)), fabsf(s.inv.z));
    const bool inf = !(big < __builtin_inff() && small > 0.0f);
    s.oct = nx | (ny << 8) | (nz << 16) | (inf ? 1u << 24 : 0u);
}
LFH_DEV bool octant_inf(const TraceState& s) { return (s.oct >> 24) != 0; }
LFH_DEV uint32_t near_x(const TraceState& s) { return s.oct & 0xFFu; }
LFH_DEV uint32_t near_y(const TraceState& s) { return (s.oct >> 8) & 0xFFu; }
LFH_DEV uint32_t near_z(const TraceState& s) { return (s.oct >> 16) & 0xFFu; }

LFH_DEV void trace_init(TraceState& s, LaneStack& st, V3 O, V3 D, float tmin, float tmax, uint32_t root) {
    s.O = O;
    s.D = D;
    s.invD = rcp3(D);
    s.o = O;
    s.d = D;
    s.inv = s.invD;
    s.tmin = tmin;
    s.tbest = tmax;
    s.cur = root;
    s.curInst = -1;
    s.curMat = 0;
    s.bestPrim = -1;
    s.bestInst = -1;
    s.bestMat = -1;
    s.bestSlot = -1;
    s.bu = 0.f;
    s.bv = 0.f;
    s.occluded = false;
    set_octant(s);
    st.reset();
}

// Triangle tests of BLAS leaf `ref` (in the current instance's space).
// Returns true when an any-hit query found its hit.
template <bool ANY, bool STATS>
LFH_DEV bool leaf_test(const TraceScene& sc, TraceState& s, uint32_t ref, TraceStats* stats) {
    const uint32_t first = leaf_first(ref), count = leaf_count(ref);
    for (uint32_t k = 0; k < count; ++k) {
        const float4* tp = sc.tris + (size_t)(first + k) * 3;
        float4 a = tp[0], b = tp[1], c = tp[2];
        float t, u, v;
        if (STATS) stats->ntri++;
        bool h = tri_test(s.o, s.d, xyz(a), xyz(b), xyz(c), &t, &u, &v);
        if (ANY) {
            if (h && t >= s.tmin && t < s.tbest) {
                s.occluded = true;
                return true;
            }
        } else if (h && t >= s.tmin) {
            int prim = (int)as_u(a.w);
            bool better = t < s.tbest ||
                          (t == s.tbest && (s.curInst < s.bestInst ||
                                            (s.curInst == s.bestInst && prim < s.bestPrim)));
            if (better) {
                s.tbest = t;
                s.bestPrim = prim;
                s.bestSlot = (int)as_u(b.w);
                s.bestInst = s.curInst;
                s.bestMat = s.curMat;
                s.bu = u;
                s.bv = v;
            }
        }
    }
    return false;
}

// TLAS leaf: move the ray into instance space and continue at the BLAS root.
template <bool STATS>
LFH_DEV void enter_instance(const TraceScene& sc, TraceState& s, LaneStack& st, uint32_t cur, TraceStats* stats) {
    const uint32_t inst = cur & 0x3FFFFFFFu;
    const float4* ip = sc.insts + (size_t)inst * 4;
    float4 r0 = ip[0], r1 = ip[1], r2 = ip[2], meta = ip[3];
    if (STATS) stats->ninst++;
    s.o = xform_inv(r0, r1, r2, s.O, 1.0f);
    s.d = xform_inv(r0, r1, r2, s.D, 0.0f);
    s.inv = rcp3(s.d);
    set_octant(s);
    st.push(kRefReturn);
    s.curInst = (int)inst;
    s.curMat = (int)as_u(meta.y);
    s.cur = as_u(meta.x);
}

// A node's near planes (a, b, c), far planes (d, e, f) and child refs.
struct NodeRec {
    float4 a, b, c, d, e, f, rf;
};
// near and far planes read by per-lane offsets: the per-axis min/max drop out
LFH_DEV void load_node(const TraceScene& sc, const TraceState& s, uint32_t cur, NodeRec& n) {
    const char* nb = reinterpret_cast<const char*>(sc.nodes);
    const uint32_t off = cur * 128u;
    const uint32_t ox = near_x(s), oy = near_y(s), oz = near_z(s);
    n.a = *reinterpret_cast<const float4*>(nb + (off + ox));
    n.b = *reinterpret_cast<const float4*>(nb + (off + oy));
    n.c = *reinterpret_cast<const float4*>(nb + (off + oz));
    n.d = *reinterpret_cast<const float4*>(nb + (off + (48u - ox)));
    n.e = *reinterpret_cast<const float4*>(nb + (off + (80u - oy)));
    n.f = *reinterpret_cast<const float4*>(nb + (off + (112u - oz)));
    n.rf = *reinterpret_cast<const float4*>(nb + (off + 96u));
}

// BVH4 node: slab-test the four child boxes, push the hit children last in
// order first.  Returns the first one, or kRefSentinel when none is hit.
//
// Bound by VALU issue (83 % busy on 16.8M mixed rays, 40 % of the lanes active
// on average) and close behind it by node traffic: 43 % of the requests hit L2,
// and the rest moves 22.9 GB per launch at 4.1-4.2 TB/s, 86 % of what a copy
// reaches.  The test is 17 instructions per child, the sort 25, the pushes
// 12 without a branch per child.  With one pop per step for all lanes and the
// order keys of slab_entry the 1M-triangle soup's closest hit went from 1650 to
// 2840 Mrays/s (incoherent half 1037 -> 2380), any hit from 3270 to 3960;
// with 128-ray reservations they are 3010-3070 and 4720-4850.
// Loading the nodes of a step before its leaf tests, to overlap the two
// latencies, spills (6.24 against 5.95 ms; any hit 6.9 against 2.2 ms).
template <bool ANY, bool STATS>
LFH_DEV uint32_t visit_node(const NodeRec& nd, bool plain, TraceState& s, LaneStack& st, float cull,
                            TraceStats* stats) {
    if (STATS) stats->nint++;
    // a closest hit at distance 0 (a ray from a mesh vertex) leaves the boxes around the origin
    // open: the triangle its tie goes to may be in one of them
    const float lim = ANY ? s.tbest * cull : fmaxf(s.tbest * cull, kLeastPositive);
    const float none = __builtin_inff();
    float h[4];      // order key of a hit child, infinity otherwise
    uint32_t r[4] = {as_u(nd.rf.x), as_u(nd.rf.y), as_u(nd.rf.z), as_u(nd.rf.w)};
    const float4 nx = nd.a, ny = nd.b, nz = nd.c, fx = nd.d, fy = nd.e, fz = nd.f;
    if (plain) {
        h[0] = slab_octant<ANY>(v3(nx.x, ny.x, nz.x), v3(fx.x, fy.x, fz.x), s.o, s.inv, lim);
        h[1] = slab_octant<ANY>(v3(nx.y, ny.y, nz.y), v3(fx.y, fy.y, fz.y), s.o, s.inv, lim);
        h[2] = slab_octant<ANY>(v3(nx.z, ny.z, nz.z), v3(fx.z, fy.z, fz.z), s.o, s.inv, lim);
        h[3] = slab_octant<ANY>(v3(nx.w, ny.w, nz.w), v3(fx.w, fy.w, fz.w), s.o, s.inv, lim);
    } else {
        h[0] = slab<ANY>(v3(nx.x, ny.x, nz.x), v3(fx.x, fy.x, fz.x), s.o, s.inv, lim);
        h[1] = slab<ANY>(v3(nx.y, ny.y, nz.y), v3(fx.y, fy.y, fz.y), s.o, s.inv, lim);
        h[2] = slab<ANY>(v3(nx.z, ny.z, nz.z), v3(fx.z, fy.z, fz.z), s.o, s.inv, lim);
        h[3] = slab<ANY>(v3(nx.w, ny.w, nz.w), v3(fx.w, fy.w, fz.w), s.o, s.inv, lim);
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (r[k] == kRefSentinel) h[k] = none;
    }
    // first in order first, absent / culled children last
#define LFH_CSWAP(a, b)                                              \
    {                                                                \
        const bool sw = h[b] < h[a];                                 \
        const float lo = sw ? h[b] : h[a], hi = sw ? h[a] : h[b];    \
        const uint32_t rl = sw ? r[b] : r[a], rh = sw ? r[a] : r[b]; \
        h[a] = lo; h[b] = hi;                                        \
        r[a] = rl; r[b] = rh;                                        \
    }
    LFH_CSWAP(0, 1) LFH_CSWAP(2, 3) LFH_CSWAP(0, 2) LFH_CSWAP(1, 3) LFH_CSWAP(1, 2)
#undef LFH_CSWAP
    if (__builtin_expect(st.sp <= kLdsStack - 3, 1)) {
        // room for three: each write lands on the slot the last valid one left
        LdsWord* p = st.lds + st.sp * 64;
        int n = 0;
        p[0] = r[3];
        n += h[3] < none ? 64 : 0;
        p[n] = r[2];
        n += h[2] < none ? 64 : 0;
        p[n] = r[1];
        n += h[1] < none ? 64 : 0;
        st.sp += n / 64;
    } else {
        if (h[3] < none) st.push(r[3]);
        if (h[2] < none) st.push(r[2]);
        if (h[1] < none) st.push(r[1]);
    }
    return h[0] < none ? r[0] : kRefSentinel;
}

// Runs up to `budget` loop steps; returns true when the traversal finished.
// A step is a node visit, a leaf or an instance entry, then one pop for all
// the lanes that have nothing left below.
template <bool ANY, bool STATS>
LFH_DEV bool trace_run(const TraceScene& sc, TraceState& s, LaneStack& st, float cull, int budget,
                       TraceStats* stats) {
    if (s.cur == kRefSentinel) return true;
    for (int it = 0; it < budget; ++it) {
        const uint32_t cur = s.cur;
        uint32_t next = kRefSentinel;
        if (ref_is_node(cur)) {
            NodeRec nd;
            load_node(sc, s, cur, nd);
            next = visit_node<ANY, STATS>(nd, __ballot(octant_inf(s)) == 0, s, st, cull, stats);
        } else if (ref_is_leaf(cur)) {
            if (leaf_test<ANY, STATS>(sc, s, cur, stats)) return true;
        } else {
            enter_instance<STATS>(sc, s, st, cur, stats);
            next = s.cur;
        }
        if (next == kRefSentinel) {
            next = st.pop();
            if (next == kRefReturn) {
                s.o = s.O;
                s.d = s.D;
                s.inv = s.invD;
                set_octant(s);
                next = st.pop();
            }
            if (next == kRefSentinel) return true;
        }
        s.cur = next;
        if (st.overflow) return true;
    }
    return false;
}

}  // namespace lfhd
