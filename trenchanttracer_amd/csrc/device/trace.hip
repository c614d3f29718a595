// Closest-hit / any-hit traversal of the SBVH on gfx950 (wave64).
//
// k_trace_wide walks the four-child tree of wide.hip (48-byte nodes, planes quantised to
// 8 bits, always outwards) and tests every triangle with the reference's arithmetic. Its
// results are those of the reference intersect() (include/geometry/IntersectKernel.cuh:
// 78-296) on the two-child tree, which walk_exact and k_trace restate:
//   - ray precompute idir / ood with the 2^-80 clamp                (:92-101)
//   - two child boxes per 64-byte node, slab entry/exit as 3-operand integer
//     min/max of the float bit patterns (v_min3_i32 / v_max3_i32 restate the
//     PTX vmin/vmax.s32 forms), traverse iff entry <= exit, entry >= tmin,
//     entry <= 1e20                                                  (:126-147)
//   - near child first, far child pushed                             (:149-167)
//   - Moeller-Trumbore on v0 and the two edges, front faces only with
//     |det| > 1e-5, tmin < t < best                                  (:230-257)
// Arithmetic of these is unfused (fp contract off) and division IEEE, so for a given
// visiting order every decision is bit-identical to the host restatement.
//
// Why the wide walk gives the same hits. The two-child walk tests the triangles of the
// leaves whose boxes the ray enters (a leaf's box lies inside every ancestor's, checked
// when the wide tree is built, and rounding is monotone, so passing the leaf's slab test
// implies passing its ancestors'). The wide boxes contain the two-child ones by more
// than the rounding of both slab tests, so the wide walk tests at least those triangles.
// When a ray is done its winner's leaf box is put through the two-child slab test at the
// distance of the nearest other triangle (next_t): if it passes, the two-child walk enters
// that leaf whatever its best distance was by then, and no tested triangle is nearer. If it
// does not pass (a hit within rounding of its box's edge), or two triangles tie exactly
// (the first one visited wins there) unless one is the other's twin (wide.hip), or the ray is one the quantised arithmetic does not
// cover (non-finite or overflowing terms, negative tmin, a full stack), the lane walks the
// two-child tree. An any-hit ray applies the leaf test to every triangle it would accept.
// That rests on a culled box holding no triangle nearer than the best distance. In exact
// arithmetic a hit lies in its triangle's box; a computed one can lie far off it, as |det|
// goes down to 1e-5. For variant 0 with the reference's test (EXACT) boxes are widened by as much as it can (kNoise), so
// that at any t the ray is inside every box down to one of the triangle's leaves and the
// triangle is tested unless t is past the best distance (with the two-sided test, which
// accepts any det but 0, variant 0 takes the two-child loop). Variant 1 culls with 2^-10 of
// the distance to spare instead: of 5M rays aimed within 1e-8 to 1e-2 of the planes
// of triangles 5 to 20 units wide, 8 got another hit than the single-lane order's (the
// speculative two-child loop: 4); of 9M at |e1||e2| up to 1 from up to 1000 units away, 3.
//
// Stack: the lowest S entries of each lane live in LDS ([entry][lane] so the lanes of a
// wave hit distinct banks), deeper entries in per-lane scratch.
//
// k_trace is the two-child while-while loop of Aila & Laine ("Understanding the Efficiency
// of Ray Traversal on GPUs", HPG 2009): for scenes without a four-child tree, and, with
// recording, for the node-fetch probe.
#include <type_traits>

#include "dev_common.h"

#pragma clang fp contract(off)

namespace tt {
namespace {

__device__ __forceinline__ int fb(float f) { return __float_as_int(f); }
__device__ __forceinline__ float bf(int i) { return __int_as_float(i); }

// fminf / fmaxf of the slab code with -0 < +0 (v_minimum3_f32 / v_maximum3_f32).
__device__ __forceinline__ float fmn(float a, float b) { return __builtin_elementwise_minimum(a, b); }
__device__ __forceinline__ float fmx(float a, float b) { return __builtin_elementwise_maximum(a, b); }

// spanBeginKepler / spanEndKepler (IntersectKernel.cuh:54-60).
__device__ __forceinline__ float span_begin(float a0, float a1, float b0, float b1, float c0, float c1, float d) {
    int z = max(min(fb(c0), fb(c1)), fb(d));
    return bf(max(max(fb(fmn(a0, a1)), fb(fmn(b0, b1))), z));
}
__device__ __forceinline__ float span_end(float a0, float a1, float b0, float b1, float c0, float c1, float d) {
    int z = min(max(fb(c0), fb(c1)), fb(d));
    return bf(min(min(fb(fmx(a0, a1)), fb(fmx(b0, b1))), z));
}

// The overflow array lives outside the struct: a struct that holds a dynamically
// indexed array is kept in scratch as a whole, and then every push and pop would
// load and store sp and the LDS pointer through scratch as well.
template <int S>
struct Stack {
    int *lds;       // this lane's column: lds[k * stride]
    int stride;
    int sp;         // entries held (the sentinel lies below entry 0)
    int off;        // sp * stride, kept by additions (no multiply per push / pop)
    int *spill;     // this lane's private overflow, kStackCap - S entries

    __device__ __forceinline__ void push(int v) {
        if (sp < S) {
            lds[off] = v;
        } else if (sp < kStackCap) {
            spill[sp - S] = v;
        }
        sp++;
        off += stride;
    }
    __device__ __forceinline__ int pop() {
        if (sp <= 0) return kSentinel;
        sp--;
        off -= stride;
        if (sp < S) return lds[off];
        if (sp < kStackCap) return spill[sp - S];
        return kSentinel;
    }
};

// One child box of a two-child node against a ray (IntersectKernel.cuh:126-147).
struct RayTerms {
    float idirx, idiry, idirz, oodx, oody, oodz, tmin;
};
__device__ __forceinline__ bool slab(float4 xy, float zlo, float zhi, const RayTerms &r, float hit_t, float *entry) {
    const float lox = xy.x * r.idirx - r.oodx, hix = xy.y * r.idirx - r.oodx;
    const float loy = xy.z * r.idiry - r.oody, hiy = xy.w * r.idiry - r.oody;
    const float loz = zlo * r.idirz - r.oodz, hiz = zhi * r.idirz - r.oodz;
    const float cmin = span_begin(lox, hix, loy, hiy, loz, hiz, r.tmin);
    const float cmax = span_end(lox, hix, loy, hiy, loz, hiz, hit_t);
    const float ray_tmax = 1e20f;
    *entry = cmin;
    return (cmin <= cmax) && (cmin >= r.tmin) && (cmin <= ray_tmax);
}

// Moeller-Trumbore, IntersectKernel.cuh:230-254 (edges precomputed: same bits): whether
// the triangle is crossed at a t in (tmin, tbest], with that t and the barycentrics.
template <int TRI>
__device__ __forceinline__ bool tri_test(float4 A, float4 B, float4 C, float ox, float oy, float oz, float dx, float dy,
                                         float dz, float tmin, float tbest, float *t_out, float *u_out, float *v_out) {
    const float tvx = ox - A.x, tvy = oy - A.y, tvz = oz - A.z;
    const float pvx = dy * C.z - dz * C.y;
    const float pvy = dz * C.x - dx * C.z;
    const float pvz = dx * C.y - dy * C.x;
    const float det = B.x * pvx + B.y * pvy + B.z * pvz;
    const float inv = 1.0f / det;
    const float u = (tvx * pvx + tvy * pvy + tvz * pvz) * inv;
    const float qvx = tvy * B.z - tvz * B.y;
    const float qvy = tvz * B.x - tvx * B.z;
    const float qvz = tvx * B.y - tvy * B.x;
    const float v = (dx * qvx + dy * qvy + dz * qvz) * inv;
    const float t = (C.x * qvx + C.y * qvy + C.z * qvz) * inv;
    // bitwise: every lane takes the same instructions (short-circuit branches cost more
    // than the comparisons they skip)
    bool ok;
    if (TRI == kTriReference) {
        const float EPS = 0.00001f;
        // the reference's back-face bounds (IntersectKernel.cuh:248-250) have their
        // comparisons reversed, !(u > 0 || u < 1) && !(v > 0 || u + v < 1): they hold for
        // a NaN u alone
        ok = (bool)(((int)(det > EPS) & (int)!(u < 0.0f) & (int)!(u > 1.0f) & (int)!(v < 0.0f) & (int)!((u + v) > 1.0f)) |
                    ((int)(det < -EPS) & (int)(u != u) & (int)!(v > 0.0f)));
    } else {
        ok = (bool)((int)(det != 0.0f) & (int)(u >= 0.0f) & (int)(u <= 1.0f) & (int)(v >= 0.0f) & (int)((u + v) <= 1.0f));
    }
    *t_out = t;
    *u_out = u;
    *v_out = v;
    return (bool)((int)ok & (int)(tmin < t) & (int)(t <= tbest));
}

// ------------------------------------------------------------------ the traversal
// Stack of a lane: entries of E (closest hit: entry distance and child, so that a popped
// subtree past the best hit is dropped unread; any hit: the child alone), the lowest S in
// LDS ([entry][lane]: the lanes of a wave hit distinct banks), deeper ones in per-lane
// scratch. Entries past kWideCap are not kept: push tells, and the lane walks the two-child
// tree instead. The LDS pointers keep their address space: through a generic one the
// compiler merges the two reads of pop into one flat load of a selected address.
#define TT_LDS __attribute__((address_space(3)))
template <class E, int S>
struct WideStack {
    TT_LDS E *bottom, *top;   // the lane's column; the first free LDS entry
    int stride;
    int over;                 // entries in scratch
    E *spill;
    __device__ __forceinline__ bool empty() const { return top == bottom; }
    __device__ __forceinline__ void clear() {
        top = bottom;
        over = 0;
    }
    // up to three entries, the last valid one on top: written unconditionally, each over
    // the one before where that was not valid (some lane of a wave nearly always pushes,
    // so branches around the writes save nothing). False: one was not kept.
    __device__ __forceinline__ bool push3(E a, bool va, E b, bool vb, E c, bool vc) {
        if (top <= bottom + (S - 3) * stride) {
            top[0] = a;
            top += va ? stride : 0;
            top[0] = b;
            top += vb ? stride : 0;
            top[0] = c;
            top += vc ? stride : 0;
            return true;
        }
        bool kept = true;
        if (va) kept = push(a);
        if (vb) kept = push(b) && kept;
        if (vc) kept = push(c) && kept;
        return kept;
    }
    __device__ __forceinline__ bool push(E v) {
        if (top < bottom + S * stride) {
            top[0] = v;
            top += stride;
        } else if (over < kWideCap - S) {
            spill[over++] = v;
        } else {
            return false;
        }
        return true;
    }
    __device__ __forceinline__ E pop() {   // not empty
        E e = top[-stride];
        if (over == 0) top -= stride;
        else e = spill[--over];
        return e;
    }
};

struct HitState {
    float t, u, v;
    int id;
};

// The two-child walk of one ray in the single-lane order, on the lane's own stack memory.
template <bool ANY, int S, int TRI>
__device__ __forceinline__ void walk_exact(const TraceArgs &a, int root, float ox, float oy, float oz, float dx, float dy,
                                           float dz, const RayTerms &r, float tmax, int *lds, int stride, int *spill,
                                           HitState &h) {
    Stack<S> st{lds, stride, 0, 0, spill};
    h = HitState{tmax, 0.0f, 0.0f, -1};
    int node = root, leaf = 0;
    while (node != kSentinel) {
        while (node >= 0 && node != kSentinel) {
            const float4 *np = a.nodes + (int64_t)node * 4;
            const float4 n0 = np[0], n1 = np[1], nz = np[2];
            const int2 ch = reinterpret_cast<const int2 *>(np + 3)[0];
            float e0, e1;
            const bool t0 = slab(n0, nz.x, nz.y, r, h.t, &e0);
            const bool t1 = slab(n1, nz.z, nz.w, r, h.t, &e1);
            if (!t0 && !t1) {
                node = st.pop();
            } else {
                int far = ch.y;
                node = t0 ? ch.x : ch.y;
                if (t0 && t1) {
                    if (e1 < e0) {
                        far = node;
                        node = ch.y;
                    }
                    st.push(far);
                }
            }
            if (node < 0) {
                leaf = node;
                node = st.pop();
                break;
            }
        }
        while (leaf < 0) {
            for (int tri = ~leaf;; ++tri) {
                const float4 *tp = a.tris + (int64_t)tri * 3;
                const float4 A = tp[0], B = tp[1], C = tp[2];
                float t, u, v;
                if (tri_test<TRI>(A, B, C, ox, oy, oz, dx, dy, dz, r.tmin, h.t, &t, &u, &v) && t < h.t) {
                    h = HitState{t, u, v, fb(A.w)};
                    if (ANY) return;
                }
                if (fb(C.w) != 0) break;
            }
            leaf = node;
            if (node < 0) node = st.pop();
        }
    }
}

// Whether the two-child walk enters a leaf (its place: node * 2 + child, below two other bits)
// at best distance hit_t.
__device__ __forceinline__ bool in_leaf(const TraceArgs &a, int place, const RayTerms &r, float hit_t) {
    const float4 *np = a.nodes + (int64_t)((place & 0x3FFFFFFF) >> 1) * 4;
    const float4 xy = np[place & 1];
    const float2 z = reinterpret_cast<const float2 *>(np + 2)[place & 1];
    float e;
    return slab(xy, z.x, z.y, r, hit_t, &e);
}

// Whether the two-child walk reaches the triangle of a record, found in the leaf at
// `place`, while its best distance is t or more, through any of its leaves: the records of
// one triangle form a ring (a spatial split puts a triangle in several leaves, and the one
// it was found in here may be one whose own box the ray misses: 1-3% of the soup's rays).
// Longer rings than the limit go to the full walk, which a lane alone takes some 150 us for:
// with a limit of 16, exact camera rays on soup of 250k triangles took 418 or 585 us by the
// rings' order, which differs from one build of the tree to the next; with 64, 415.
__device__ __forceinline__ bool reached(const TraceArgs &a, int rec, int place, int chain, const RayTerms &r, float t,
                                        float near) {
    if (in_leaf(a, place, r, t)) return true;
    // (where another triangle as near is what keeps it out, that would do so elsewhere too)
    if (t < near && in_leaf(a, place, r, near)) return false;
    const auto word = [&](int at, int k) { return fb(reinterpret_cast<const float4 *>(a.wide + (uint32_t)at)[k].w); };
    // the leaf where the triangle was met last, if more than once
    if (chain != rec && word(chain, 0) == word(rec, 0) && in_leaf(a, word(chain, 1), r, t)) return true;
    int at = rec;
    for (int i = 0; i < 64; ++i) {
        at = word(at, 2) & 0x7FFFFFFF;
        if (at == rec) return false;
        if (in_leaf(a, word(at, 1), r, t)) return true;
    }
    return false;
}

// EXACT: what boxes are widened by for the sake of hits at t or nearer. Such a hit's |o - v0|
// is at most t |d|, the triangle's longer edge and the hit's own displacement; the size codes
// hold the last two for directions of about unit length (wide.hip), others are not narrowed.
__device__ __forceinline__ float noise_to(const TraceArgs &a, float dx, float dy, float dz, float t) {
    const float len = sqrtf(dx * dx + dy * dy + dz * dz);
    return len <= kUnitLength ? a.wide_noise * len * (t * len + a.wide_grain) : INFINITY;
}

// The counts of the queue traced, uniform, and the slot of its r-th position (-1: none).
struct SegmentCounts {
    int32_t n0 = 0, n1 = 0, n2 = 0, n3 = 0;   // (an array would go to scratch memory)
    static_assert(kSegs == 4, "one count each");
    __device__ __forceinline__ int32_t read(const TraceArgs &a) {
        n0 = __builtin_amdgcn_readfirstlane(*a.n_dev);
        if (!a.seg) return n0;
        n1 = __builtin_amdgcn_readfirstlane(a.n_dev[kSegStride]);
        n2 = __builtin_amdgcn_readfirstlane(a.n_dev[2 * kSegStride]);
        n3 = __builtin_amdgcn_readfirstlane(a.n_dev[3 * kSegStride]);
        return (max(max(n0, n1), max(n2, n3)) + 63) / 64 * (64 * kSegs);
    }
    __device__ __forceinline__ int32_t slot(const TraceArgs &a, int32_t r) const {
        if (!a.seg) return r;
        const int s = segment_of(r);
        const int32_t i = entry_of(r), lo = s & 1 ? n1 : n0, hi = s & 1 ? n3 : n2;
        return i < (s & 2 ? hi : lo) ? s * a.seg + i : -1;
    }
};
__device__ __forceinline__ void reset_counts(const TraceArgs &a, int tid) {
    if (blockIdx.x == 0 && tid < kSegs) {
        if (a.reset0) a.reset0[tid * kSegStride] = 0;
        if (a.reset1) a.reset1[tid * kSegStride] = 0;
    }
}

// log2 of the rays of a group (TraceArgs::spread), uniform.
__device__ __forceinline__ int group_bits(uint32_t n, int32_t spread) {
    if (!spread || n == 0u) return 6;
    const uint32_t full = (n - 1u) >> spread;
    return full ? min(6, 32 - __clz((int)full)) : 0;
}

// EXACT widens boxes as kNoise asks (9 instructions a node, 78 VGPRs as held to 6 waves per
// SIMD, 87 without): whole calls of 1.2M rays, soup of 250k triangles, 720 us as variant 1, 746
// exact, of 20k 378 and 383.
//
// Four-child walk. What bounds it: VALU issue first, vector memory lane loads second. On
// the 1M-triangle soup (8.3M rays in Morton order) the two-child while-while loop kept VALU
// issue 90% and the address path 82% busy, with 32% of the lanes active: 1.85e9 VALU
// instructions, 1.53e9 cache accesses and 4.0 ms a launch. Visiting four boxes with 3 loads
// instead of 8, and taking node visits and triangle tests by the vote below (59% of the
// lanes active), takes 1.43e9, 0.90e9 and 3.0 ms; each alone gains little, as the other
// limit holds (four children in the while-while loop: 6.6 ms, slower).
template <bool ANY, int S, int TRI, bool EXACT>
__global__ __launch_bounds__(256, ANY ? 1 : 6) void k_trace_wide(TraceArgs a) {
    static_assert(!EXACT || (!ANY && TRI == kTriReference), "kNoise is the reference test's");
    using E = typename std::conditional<ANY, int, uint64_t>::type;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    // XCD-contiguous order: the hardware hands blocks to the 8 XCDs round-robin, so
    // block b runs on XCD b % 8; renumbering b -> (b % 8) * q + b / 8 (for the first
    // 8q blocks, q = blocks / 8; the tail keeps its number) is a bijection that gives
    // each XCD's L2 one contiguous range of waves
    unsigned vb = blockIdx.x;
    if (a.xcd_order) {
        const unsigned q = gridDim.x >> 3;
        if (vb < (q << 3)) vb = (vb & 7u) * q + (vb >> 3);
    }
    uint32_t n = (uint32_t)a.n;   // below 2^31 (launch_trace)
    SegmentCounts in;
    if (a.n_dev) n = min((uint32_t)max(0, in.read(a)), n);
    reset_counts(a, tid);
    // Launch forms. One wave per 64-ray group; persistent waves (Aila & Laine's persistent
    // threads with ray replacement): the grid holds about as many waves as the chip keeps
    // resident, and wave w of W owns the groups w, w + W, w + 2W, ... in that order, so that
    // all waves sweep the ray range together (the rays in flight at any moment lie in a
    // window of about 2W groups, as with one wave per group, which keeps coherent rays'
    // nodes in cache); and sweeps: the same over one part of the range after another, W
    // waves and a.sweep groups each per part, so that the waves cannot drift apart over a
    // long range and the dispatcher evens out their loads. A lane whose ray is done takes
    // the next ray of its wave's sequence (ballot and prefix count, no atomics): the lanes
    // stay busy until the sequence runs out, instead of idling behind the wave's longest
    // ray. Each ray's traversal is the same as with one ray per lane. The wave's number is
    // read from its first lane, so that everything uniform stays in scalar registers and
    // the loops below branch on scalars.
    const int gs = group_bits(n, a.spread);
    const uint32_t groups = (uint32_t)(((uint64_t)n + (1u << gs) - 1u) >> gs);
    const uint32_t w = vb * (blockDim.x >> 6) + (uint32_t)__builtin_amdgcn_readfirstlane(tid >> 6);
    uint32_t waves = max(1u, min(gridDim.x * (blockDim.x >> 6), groups)), first = w, last = groups;
    if (a.sweep) {
        waves = (uint32_t)a.sweep_waves;
        const uint32_t part = w / waves, size = waves * (uint32_t)a.sweep;
        first = part * size + (w - part * waves);
        last = min(groups, (part + 1u) * size);
    }
    // whole waves only: nothing below synchronises the block
    if (first >= last || (!a.sweep && w >= waves)) return;
    const uint32_t total = ((last - first + waves - 1u) / waves) << gs;   // the wave's sequence positions
    const unsigned long long below = (1ull << lane) - 1ull;

    // one private array serves both walks
    constexpr int kWideWords = (kWideCap - S) * (int)(sizeof(E) / 4);
    constexpr int kSpillWords = kWideWords > kStackCap - S ? kWideWords : kStackCap - S;
    __align__(8) int spill[kSpillWords];
    WideStack<E, S> st;
    st.bottom = (TT_LDS E *)lds_raw + tid;
    st.stride = blockDim.x;
    st.clear();
    st.spill = reinterpret_cast<E *>(spill);

    int rid = -1;              // the lane's ray (-1: none)
    uint32_t cursor = 0;       // next sequence position (uniform)
    float ox = 0.0f, oy = 0.0f, oz = 0.0f, tmin = 0.0f, dx = 0.0f, dy = 0.0f, dz = 1.0f;
    float idirx = 0.0f, idiry = 0.0f, idirz = 0.0f;
    float nearx = 0.0f, neary = 0.0f, nearz = 0.0f;   // -(o idir) less the rounding allowance
    float farx = 0.0f, fary = 0.0f, farz = 0.0f;      // -(o idir) plus it
    float noise = 0.0f;        // EXACT: what a node's boxes are widened by, over its size code squared
    int node = kSentinel;      // inner node to visit; sign set: a leaf waiting for room; kSentinel: none
    int leaf = 0, leaf2 = 0;   // sign set: next record of the leaf being tested, first of the one after it
    float hit_t = 0.0f;
    int cull = 0;              // bits of the distance boxes are culled against (hit_t and a share to spare)
    float spare = 0.0f;
    // the winner's record (-1: none; any hit: 0 once occluded). Its id and barycentrics go
    // straight to the ray's hit record when it is accepted, which frees their registers.
    int hit_rec = -1, hit_place = 0;   // (and the place of its leaf)
    // A triangle tested after the winner wherever it is cannot take the ray from it, so its
    // distance does not count: one whose twin (two bits of its record) is the winner, or was
    // found to be so (chain). Otherwise every hit on coincident triangles would be a tie that
    // ends in a full walk (1.2M rays on soup of 50k triangles, each twice: 2811 us, with this
    // 599, once each 531; path tracing one with faces on both sides 5818 and 3589; two-child loop
    // 823 and 3544). Also the winner itself where it was met again, in another leaf.
    int chain = 0;
    float next_t = 0.0f;       // no other accepted triangle lies below this (at most where boxes are culled)
    bool redo = false;         // not for the wide walk

    for (;;) {
        const bool done = node == kSentinel && st.empty() && leaf >= 0;
        if (done && rid >= 0) {
            const RayTerms r{idirx, idiry, idirz, ox * idirx, oy * idiry, oz * idirz, tmin};
            bool walk = redo;
            if (!ANY && !walk && hit_rec >= 0)
                walk = !(hit_t < next_t) ||
                       !reached(a, hit_rec, hit_place, chain, r, fminf(next_t, bf(cull)), hit_t * 1.00001f);
            if (walk) {
                HitState h;
                walk_exact<ANY, S, TRI>(a, a.roots ? a.roots[a.ray_root ? a.ray_root[rid] : 0] : 0, ox, oy, oz, dx, dy, dz,
                                        r, a.rays[rid].tmax, reinterpret_cast<int *>(lds_raw) + tid * (int)(sizeof(E) / 4),
                                        st.stride * (int)(sizeof(E) / 4), spill, h);
                if (ANY) hit_rec = h.id == -1 ? -1 : 0;
                else *reinterpret_cast<float4 *>(a.hits + rid) = make_float4(bf(h.id), h.t, h.u, h.v);
            }
            if (ANY) a.flags[rid] = hit_rec >= 0 ? 1 : 0;
            else if (!walk && hit_rec < 0)
                *reinterpret_cast<float4 *>(a.hits + rid) = make_float4(bf(-1), hit_t, 0.0f, 0.0f);
            rid = -1;
        }
        const unsigned long long m = __ballot(done);
        // new rays once enough lanes are idle (all idle always qualifies, so the
        // wave cannot wait on itself)
        const bool take = (int32_t)__popcll(m) >= a.refill;
        if (take && done) {
            const uint32_t q = cursor + (uint32_t)__popcll(m & below);
            if (q < total) {
                const uint32_t r = (((q >> gs) * waves + first) << gs) + (q & ((1u << gs) - 1u));
                if (r < n) rid = a.order ? (int)a.order[r] : in.slot(a, (int)r);
            }
            if (rid >= 0) {
                const float4 *rp = reinterpret_cast<const float4 *>(a.rays + rid);
                const float4 r0 = rp[0], r1 = rp[1];
                ox = r0.x;
                oy = r0.y;
                oz = r0.z;
                tmin = r0.w;
                dx = r1.x;
                dy = r1.y;
                dz = r1.z;
                const float tmax = r1.w;
                const float ooeps = 0x1p-80f;
                idirx = 1.0f / (fabsf(dx) > ooeps ? dx : copysignf(ooeps, dx));
                idiry = 1.0f / (fabsf(dy) > ooeps ? dy : copysignf(ooeps, dy));
                idirz = 1.0f / (fabsf(dz) > ooeps ? dz : copysignf(ooeps, dz));
                // allowance for the rounding of both slab tests (wide.hip's planes are exact
                // to 2^-53): the two-child test's terms are off by at most
                // 2.01 (B + |o|) |idir| 2^-24 and this one's by 4.1 of the same, B the largest
                // coordinate of a plane; 8 covers the two
                // (EXACT: 32 instead, for what kNoise leaves out: besides this slab test's 4.1, 9 for
                // the test's unamplified roundings, 2 for the edges', 9 for a spatial split's clipped
                // boxes)
                constexpr float kSlack = EXACT ? 0x1p-19f : 0x1p-21f;
                const float sx = (fabsf(ox) + a.wide_bound) * fabsf(idirx) * kSlack;
                const float sy = (fabsf(oy) + a.wide_bound) * fabsf(idiry) * kSlack;
                const float sz = (fabsf(oz) + a.wide_bound) * fabsf(idirz) * kSlack;
                nearx = -(ox * idirx) - sx;
                neary = -(oy * idiry) - sy;
                nearz = -(oz * idirz) - sz;
                farx = sx - ox * idirx;
                fary = sy - oy * idiry;
                farz = sz - oz * idirz;
                // rays the wide walk covers: all terms finite (NaN compares false), the allowance
                // far above what denormal terms lose (directions past about 2^79 of the scene's
                // size do not), distances that compare as integers
                constexpr float kLeast = 0x1p-100f;
                bool fits = sx > kLeast && sy > kLeast && sz > kLeast && sx < 1e30f && sy < 1e30f &&
                            sz < 1e30f && fb(tmin) >= 0 && tmin < 1e30f && fb(tmax) >= 0 && tmax <= INFINITY;
                // To the scenes' far corner. Distances are culled with 2^-10 to spare, from far away
                // 2^-8 of the scenes' diagonal, but 2^-16 at least: 2^-10 of 1000 diagonals is all
                // of the scene, as is 2^-16 of 2^15, where closest hits take the full walk. (4M
                // rays on the unit cube of 50k triangles from 100, 1000, 10000 away, with 2^-10
                // throughout 1336, 4374, 4398 us, with this 1067, 1115, 1688; two-child loop 2001.)
                const float ax = fabsf(ox - a.wide_mid[0]) + a.wide_half[0];
                const float ay = fabsf(oy - a.wide_mid[1]) + a.wide_half[1];
                const float az = fabsf(oz - a.wide_mid[2]) + a.wide_half[2];
                spare = min(max(a.wide_grain * 0x1p-6f / (ax + ay + az), 0x1p-16f), 0x1p-10f);
                fits = fits && (ANY || ax + ay + az < a.wide_grain * 0x1p17f);
                if constexpr (EXACT) {
                    const float dd = dx * dx + dy * dy + dz * dz;
                    const float across = sqrtf(dd) * sqrtf(ax * ax + ay * ay + az * az);
                    noise = min(a.wide_noise * across, noise_to(a, dx, dy, dz, tmax));
                    const float most = noise * (255.0f * 255.0f);
                    fits = fits && across <= a.wide_reach && dd > 1e-30f && most * fabsf(idirx) < 1e30f &&
                           most * fabsf(idiry) < 1e30f && most * fabsf(idirz) < 1e30f;
                }
                st.clear();
                redo = !fits;
                leaf = leaf2 = 0;
                node = fits ? a.wide_step * (a.ray_root ? a.ray_root[rid] : 0) : kSentinel;
                hit_t = next_t = tmax;
                hit_rec = -1;
                cull = fb(tmax + tmax * spare);
            }
        }
        if (take) cursor += (uint32_t)__popcll(m);
        // ends once the sequence is used up and no lane holds a ray (only the last
        // group of the range can be partial)
        if (cursor >= total && __ballot(rid >= 0) == 0) break;
        const int quit = cursor < total ? a.refill : 64;   // idle lanes at which the wave retires rays

        // Each round the wave visits a node or tests a triangle, whichever more of its lanes
        // are ready for (a node visit takes about twice a test's instructions, so it needs
        // 1.4 times the lanes). Lanes hold up to two leaves, so most are ready for either.
        // Simulated wave utilisation on Morton-sorted incoherent rays of 1M-triangle soup:
        // 0.69 / 0.49 (node / triangle rounds) against 0.42 / 0.33 for the while-while loop,
        // which runs each phase until its slowest lane is through.
        for (;;) {
            if (node == kSentinel && !st.empty()) {
                const E e = st.pop();
                if constexpr (ANY) node = e;
                else node = (int)(e >> 32) <= cull ? (int)(uint32_t)e : kSentinel;
            }
            {
                // a waiting leaf moves up where there is room
                const bool move = (int)(node < 0) & (int)(leaf2 >= 0), first = leaf >= 0;
                const int moved = node;
                node = move ? kSentinel : node;
                leaf2 = move ? (first ? 0 : moved) : leaf2;
                leaf = (int)move & (int)first ? moved : leaf;
            }
            // records are 16-byte units below 2^30: an inner node compares below, kSentinel
            // and leaves (sign set) above
            const bool at_node = (uint32_t)node < (1u << 30), at_leaf = leaf < 0;
            const unsigned long long mn = __ballot(at_node), mt = __ballot(at_leaf);
            // (a lane that popped a stale entry counts as idle for this round)
            if (64 - (int)__popcll(mn | mt) >= quit) break;
            if ((int)__popcll(mn) * 5 >= (int)__popcll(mt) * 7) {
                if (at_node) {
                    const uint4 *np = a.wide + (uint32_t)node;
                    const uint4 q0 = np[0], q1 = np[1], q2 = np[2];
                    // plane scales 2^code, codes signed bytes
                    const float kx = ldexpf(idirx, __builtin_amdgcn_sbfe((int)q1.y, 0, 8));
                    const float ky = ldexpf(idiry, __builtin_amdgcn_sbfe((int)q1.y, 8, 8));
                    const float kz = ldexpf(idirz, __builtin_amdgcn_sbfe((int)q1.y, 16, 8));
                    const float bx = bf((int)q0.x), by = bf((int)q0.y), bz = bf((int)q0.z);
                    float nx = __builtin_fmaf(bx, idirx, nearx), fx = __builtin_fmaf(bx, idirx, farx);
                    float ny = __builtin_fmaf(by, idiry, neary), fy = __builtin_fmaf(by, idiry, fary);
                    float nz = __builtin_fmaf(bz, idirz, nearz), fz = __builtin_fmaf(bz, idirz, farz);
                    if constexpr (EXACT) {
                        const float code = (float)(q1.y >> 24), pad = noise * code * code;
                        nx = __builtin_fmaf(-pad, fabsf(idirx), nx);
                        fx = __builtin_fmaf(pad, fabsf(idirx), fx);
                        ny = __builtin_fmaf(-pad, fabsf(idiry), ny);
                        fy = __builtin_fmaf(pad, fabsf(idiry), fy);
                        nz = __builtin_fmaf(-pad, fabsf(idirz), nz);
                        fz = __builtin_fmaf(pad, fabsf(idirz), fz);
                    }
                    const bool px = idirx >= 0.0f, py = idiry >= 0.0f, pz = idirz >= 0.0f;
                    const uint32_t nwx = px ? q1.z : q1.w, fwx = px ? q1.w : q1.z;
                    const uint32_t nwy = py ? q2.x : q2.y, fwy = py ? q2.y : q2.x;
                    const uint32_t nwz = pz ? q2.z : q2.w, fwz = pz ? q2.w : q2.z;
                    // per slot: entry distance with 8 times the slot in its low five bits (all
                    // ones: not entered)
                    uint32_t key[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const float tnx = __builtin_fmaf((float)((nwx >> (8 * k)) & 255u), kx, nx);
                        const float tny = __builtin_fmaf((float)((nwy >> (8 * k)) & 255u), ky, ny);
                        const float tnz = __builtin_fmaf((float)((nwz >> (8 * k)) & 255u), kz, nz);
                        const float tfx = __builtin_fmaf((float)((fwx >> (8 * k)) & 255u), kx, fx);
                        const float tfy = __builtin_fmaf((float)((fwy >> (8 * k)) & 255u), ky, fy);
                        const float tfz = __builtin_fmaf((float)((fwz >> (8 * k)) & 255u), kz, fz);
                        // bits compare as the floats do: the entry is at least tmin >= +0, and a
                        // negative exit stays negative
                        const int en = max(max(fb(tnx), fb(tny)), max(fb(tnz), fb(tmin)));
                        const int ex = min(min(fb(tfx), fb(tfy)), min(fb(tfz), cull));
                        key[k] = en <= ex ? ((uint32_t)en & ~31u) | (uint32_t)(8 * k) : 0xFFFFFFFFu;
                    }
                    // nearest first
                    const auto order2 = [&](int i, int j) {
                        const uint32_t lo = min(key[i], key[j]), hi = max(key[i], key[j]);
                        key[i] = lo;
                        key[j] = hi;
                    };
                    order2(0, 1);
                    order2(2, 3);
                    order2(0, 2);
                    order2(1, 3);
                    order2(1, 2);
                    // the slot's byte: unit offset from the node's child block, sign: a leaf
                    const auto child = [&](uint32_t key_k) -> int {
                        return (int)((uint32_t)__builtin_amdgcn_sbfe((int)q1.x, key_k, 8) & 0x8000007Fu) + (int)q0.w;
                    };
                    const auto entry = [&](uint32_t key_k) -> E {
                        if constexpr (ANY) return child(key_k);
                        else return (uint64_t)key_k << 32 | (uint32_t)child(key_k);
                    };
                    redo |= !st.push3(entry(key[3]), key[3] != 0xFFFFFFFFu, entry(key[2]), key[2] != 0xFFFFFFFFu,
                                      entry(key[1]), key[1] != 0xFFFFFFFFu);
                    node = key[0] != 0xFFFFFFFFu ? child(key[0]) : kSentinel;
                }
            } else if (at_leaf) {
                const uint32_t rec = (uint32_t)leaf & 0x7FFFFFFFu;
                const float4 *tp = reinterpret_cast<const float4 *>(a.wide + rec);
                const float4 A = tp[0], B = tp[1], C = tp[2];
                float t, u, v;
                const bool end = fb(C.w) < 0;
                leaf = end ? leaf2 : leaf + a.wide_step;
                leaf2 = end ? 0 : leaf2;
                if (tri_test<TRI>(A, B, C, ox, oy, oz, dx, dy, dz, tmin, ANY ? hit_t : bf(cull), &t, &u, &v)) {
                    if (ANY) {
                        const RayTerms r{idirx, idiry, idirz, ox * idirx, oy * idiry, oz * idirz, tmin};
                        if (t < hit_t && in_leaf(a, fb(B.w), r, hit_t)) {
                            hit_rec = 0;
                            redo = false;
                            st.clear();
                            node = kSentinel;
                            leaf = leaf2 = 0;
                        }
                    } else if (t < hit_t) {
                        *reinterpret_cast<float4 *>(a.hits + rid) = make_float4(A.w, t, u, v);
                        next_t = hit_t;
                        hit_t = t;
                        hit_rec = (int)rec;
                        hit_place = fb(B.w);
                        chain = (int)rec;
                        cull = fb(t + t * spare);
                        if constexpr (EXACT) noise = min(noise, noise_to(a, dx, dy, dz, bf(cull)));
                    } else if (hit_rec >= 0 && t < next_t) {
                        // (without a winner a triangle at or past tmax is no hit, and next_t is tmax)
                        const int id = fb(reinterpret_cast<const float4 *>(a.wide + (uint32_t)hit_rec)->w);
                        const uint32_t twin = (uint32_t)fb(B.w) >> 30;
                        const int at = (int)(rec - (twin & 1 ? a.wide_step : 0) - (twin & 2 ? 2 * a.wide_step : 0));
                        if (fb(A.w) == id ||
                            (twin && (at == chain ||
                                      fb(reinterpret_cast<const float4 *>(a.wide + (uint32_t)at)->w) == id)))
                            chain = (int)rec;
                        else next_t = fminf(next_t, t);
                    }
                }
            }
        }
    }
}

// The two-child while-while loop: for scenes without a four-child tree (wide.hip) and for
// the node-fetch probe. VARIANT 0 (exact): a lane leaves the node loop as soon as it holds
// a leaf, the single-lane order; VARIANT 1 (speculative): lanes keep descending until no
// lane of the wave is still searching for its first leaf (__any ballot, :192-203); results
// can differ only where a triangle lies on a box boundary within rounding of the current
// hit distance.
// REC (closest hit only; the probe): 1 counts each ray's node visits, triangle tests and
// leaf visits; 2 records at every node visit the slab test's outcome as a 4-bit code (bit
// 0: child 0 entered, bit 1: child 1 entered, bit 2: both, child 1 first); 3 replays: the
// same loop, stack, leaf postponement, ballots and refills, every node and triangle record
// fetched, but each node's outcome read from the record instead of computed and no
// triangle arithmetic.
template <int VARIANT, bool ANY, int S, int TRI, int REC = 0>
__global__ __launch_bounds__(256) void k_trace(TraceArgs a) {
    static_assert(REC == 0 || !ANY, "fetch recording follows the closest-hit loop");
    extern __shared__ int lds_stack[];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    // XCD-contiguous order: the hardware hands blocks to the 8 XCDs round-robin, so
    // block b runs on XCD b % 8; renumbering b -> (b % 8) * q + b / 8 (for the first
    // 8q blocks, q = blocks / 8; the tail keeps its number) is a bijection that gives
    // each XCD's L2 one contiguous range of waves
    unsigned vb = blockIdx.x;
    if (a.xcd_order) {
        const unsigned q = gridDim.x >> 3;
        if (vb < (q << 3)) vb = (vb & 7u) * q + (vb >> 3);
    }
    int64_t n = a.n;
    SegmentCounts in;
    if (a.n_dev) n = min((int64_t)in.read(a), n);
    reset_counts(a, tid);
    // the launch form of k_trace_wide
    const int gs = group_bits((uint32_t)max((int64_t)0, n), a.spread);
    const int64_t groups = (n + (1 << gs) - 1) >> gs;
    const int64_t waves_all = (int64_t)gridDim.x * (blockDim.x >> 6);
    const int64_t waves = max((int64_t)1, min(waves_all, groups));
    const int64_t w = (int64_t)vb * (blockDim.x >> 6) + (tid >> 6);
    if (w >= waves) return;   // whole waves only: nothing below synchronises the block
    const int64_t total = ((groups - w + waves - 1) / waves) << gs;   // the wave's sequence positions
    const unsigned long long below = (1ull << lane) - 1ull;

    int spill[kStackCap - S];
    Stack<S> st;
    st.lds = lds_stack + tid;
    st.stride = blockDim.x;
    st.sp = 0;
    st.off = 0;
    st.spill = spill;

    int64_t rid = -1;          // the lane's ray (-1: none)
    int64_t cursor = 0;        // next sequence position (uniform)
    float ox = 0.0f, oy = 0.0f, oz = 0.0f, tmin = 0.0f, dx = 0.0f, dy = 0.0f, dz = 1.0f;
    float idirx = 0.0f, idiry = 0.0f, idirz = 0.0f, oodx = 0.0f, oody = 0.0f, oodz = 0.0f;
    int leaf_addr = 0;
    int node_addr = kSentinel;
    float hit_t = 0.0f, hit_u = 0.0f, hit_v = 0.0f;
    int hit_id = -1;
    int rec_n = 0, rec_t = 0, rec_l = 0;   // node visits, triangle tests, leaf visits of the lane's ray (REC)
    int64_t rec_base = 0, rec_cap = 0;     // the ray's words of outcome codes (REC 2, 3)
    uint32_t rec_word = 0;                 // codes of the current 8 visits
    uint32_t rec_next = 0;                 // codes of the next 8 (REC 3: loaded a word ahead)
    uint32_t tok = 0;                      // every fetched word folded in (REC 3)

    for (;;) {
        const bool done = node_addr == kSentinel;
        if (done && rid >= 0) {
            if (REC == 1) {
                a.rec_nodes[rid] = rec_n;
                a.rec_tris[rid] = rec_t;
                a.rec_leaves[rid] = rec_l;
            } else if (REC == 2) {
                if ((rec_n & 7) != 0 && (rec_n >> 3) < rec_cap) a.rec_log[rec_base + (rec_n >> 3)] = (int32_t)rec_word;
            } else if (REC == 3) {
                *reinterpret_cast<float4 *>(a.hits + rid) = make_float4(bf((int)tok), 0.0f, 0.0f, 0.0f);
            } else if (ANY) {
                a.flags[rid] = hit_id != -1 ? 1 : 0;
            } else {
                *reinterpret_cast<float4 *>(a.hits + rid) = make_float4(bf(hit_id), hit_t, hit_u, hit_v);
            }
            rid = -1;
        }
        const unsigned long long m = __ballot(done);
        // new rays once enough lanes are idle (all idle always qualifies, so the
        // wave cannot wait on itself)
        const bool take = (int32_t)__popcll(m) >= a.refill;
        if (take && done) {
            const int64_t q = cursor + __popcll(m & below);
            if (q < total) {
                const int64_t r = (((q >> gs) * waves + w) << gs) + (q & ((1 << gs) - 1));
                if (r < n) rid = a.order ? (int64_t)a.order[r] : in.slot(a, (int)r);
            }
            if (rid >= 0) {
                const float4 *rp = reinterpret_cast<const float4 *>(a.rays + rid);
                const float4 r0 = rp[0], r1 = rp[1];
                ox = r0.x;
                oy = r0.y;
                oz = r0.z;
                tmin = r0.w;
                dx = r1.x;
                dy = r1.y;
                dz = r1.z;
                const float ooeps = 0x1p-80f;
                idirx = 1.0f / (fabsf(dx) > ooeps ? dx : copysignf(ooeps, dx));
                idiry = 1.0f / (fabsf(dy) > ooeps ? dy : copysignf(ooeps, dy));
                idirz = 1.0f / (fabsf(dz) > ooeps ? dz : copysignf(ooeps, dz));
                oodx = ox * idirx;
                oody = oy * idiry;
                oodz = oz * idirz;
                st.sp = 0;
                st.off = 0;
                leaf_addr = 0;
                node_addr = a.num_nodes > 0 ? (a.roots ? a.roots[a.ray_root ? a.ray_root[rid] : 0] : 0) : kSentinel;
                hit_t = r1.w;
                hit_u = 0.0f;
                hit_v = 0.0f;
                hit_id = -1;
                rec_n = 0;
                rec_t = 0;
                rec_l = 0;
                rec_word = 0;
                if (REC >= 2) {
                    rec_base = a.rec_off[rid];
                    rec_cap = a.rec_off[rid + 1] - rec_base;
                }
                if (REC == 3) {
                    tok = __float_as_uint(r0.x) ^ __float_as_uint(r1.w);
                    rec_next = rec_cap > 0 ? (uint32_t)a.rec_log[rec_base] : 0u;
                }
            }
        }
        if (take) cursor += __popcll(m);
        // ends once the sequence is used up and no lane holds a ray (only the last
        // group of the range can be partial)
        if (cursor >= total && !__any(rid >= 0)) break;

        while (node_addr >= 0 && node_addr != kSentinel) {
            const float4 *np = a.nodes + (int64_t)node_addr * 4;
            const float4 n0xy = np[0];
            const float4 n1xy = np[1];
            const float4 nz = np[2];
            const int2 ch = reinterpret_cast<const int2 *>(np + 3)[0];
            bool t0, t1, c1_first;
            if (REC == 3) {
                // the recorded outcome; the box words are still fetched and used
                if ((rec_n & 7) == 0) {
                    // the next word is requested 8 visits before it is needed
                    rec_word = rec_next;
                    const int64_t wn = (rec_n >> 3) + 1;
                    rec_next = wn < rec_cap ? (uint32_t)a.rec_log[rec_base + wn] : 0u;
                }
                const uint32_t code = (rec_word >> ((rec_n & 7) * 4)) & 15u;
                ++rec_n;
                t0 = (code & 1u) != 0;
                t1 = (code & 2u) != 0;
                c1_first = (code & 4u) != 0;
                tok ^= (__float_as_uint(n0xy.x) ^ __float_as_uint(n0xy.y) ^ __float_as_uint(n0xy.z) ^
                        __float_as_uint(n0xy.w)) ^
                       (__float_as_uint(n1xy.x) ^ __float_as_uint(n1xy.y) ^ __float_as_uint(n1xy.z) ^
                        __float_as_uint(n1xy.w)) ^
                       (__float_as_uint(nz.x) ^ __float_as_uint(nz.y) ^ __float_as_uint(nz.z) ^ __float_as_uint(nz.w));
            } else {

            const RayTerms r{idirx, idiry, idirz, oodx, oody, oodz, tmin};
            float c0min, c1min;
            t0 = slab(n0xy, nz.x, nz.y, r, hit_t, &c0min);
            t1 = slab(n1xy, nz.z, nz.w, r, hit_t, &c1min);
            c1_first = c1min < c0min;
            if (REC == 2) {
                const uint32_t code = (t0 ? 1u : 0u) | (t1 ? 2u : 0u) | ((t0 && t1 && c1_first) ? 4u : 0u);
                rec_word |= code << ((rec_n & 7) * 4);
                if ((rec_n & 7) == 7) {
                    if ((rec_n >> 3) < rec_cap) a.rec_log[rec_base + (rec_n >> 3)] = (int32_t)rec_word;
                    rec_word = 0;
                }
            }
            if (REC) ++rec_n;
            }
            // the child indices are used only when a child is entered; without a use on
            // every path the compiler issues their load there, after the slab tests,
            // which makes it a second dependent fetch per visited node. This empty
            // statement uses them here, so all 64 bytes of the node are fetched at once.
            asm volatile("" : : "v"(ch.x), "v"(ch.y));

            if (!t0 && !t1) {
                node_addr = st.pop();
            } else {
                int far = ch.y;
                node_addr = t0 ? ch.x : ch.y;
                if (t0 && t1) {
                    if (c1_first) {
                        int tmp = node_addr;
                        node_addr = far;
                        far = tmp;
                    }
                    st.push(far);
                }
            }
            if (node_addr < 0 && leaf_addr >= 0) {
                leaf_addr = node_addr;
                node_addr = st.pop();
            }
            if (VARIANT == 0) {
                if (leaf_addr < 0) break;
            } else {
                if (!__any(leaf_addr >= 0)) break;
            }
        }

        while (leaf_addr < 0) {
            int tri = ~leaf_addr;
            if (REC) ++rec_l;
            for (;;) {
                if (REC) ++rec_t;
                const float4 *tp = a.tris + (int64_t)tri * 3;
                const float4 A = tp[0];
                const float4 B = tp[1];
                const float4 C = tp[2];
                if (REC == 3) {
                    // the record is fetched and its words used; no test
                    tok ^= (__float_as_uint(A.x) ^ __float_as_uint(A.y) ^ __float_as_uint(A.z) ^ __float_as_uint(A.w)) ^
                           (__float_as_uint(B.x) ^ __float_as_uint(B.y) ^ __float_as_uint(B.z) ^ __float_as_uint(B.w)) ^
                           (__float_as_uint(C.x) ^ __float_as_uint(C.y) ^ __float_as_uint(C.z));
                    if (fb(C.w) != 0) break;
                    ++tri;
                    continue;
                }
                float t, u, v;
                if (tri_test<TRI>(A, B, C, ox, oy, oz, dx, dy, dz, tmin, hit_t, &t, &u, &v) && t < hit_t) {
                    hit_t = t;
                    hit_u = u;
                    hit_v = v;
                    hit_id = fb(A.w);
                    if (ANY) {
                        node_addr = kSentinel;
                        break;
                    }
                }
                if (fb(C.w) != 0) break;
                ++tri;
            }
            leaf_addr = node_addr;
            if (node_addr < 0) node_addr = st.pop();
        }
    }
}

// Persistent launch: as many blocks as the CUs hold at once (occupancy of this
// instantiation at this block size and LDS), and for a known ray count no more
// blocks than 64-ray groups. Otherwise one wave per 64-ray group (every wave's
// sequence is its one group): the hardware dispatcher then balances the waves,
// which wins where rays are coherent or the count is known. With a.sweep (a known count)
// the range is traced in parts of that many groups per resident wave; a range of at most
// one group per wave is a launch of one wave per group.
template <class K>
hipError_t launch_k(K kernel, TraceArgs a, bool persistent, int block, size_t lds, int num_cus, hipStream_t s) {
    // lanes of a group, as the kernel sets them (group_bits)
    int64_t rays = 64;
    while (a.spread && rays > 1 && a.n <= (rays / 2) << a.spread) rays /= 2;
    int64_t grid = ((a.n + rays - 1) / rays + block / 64 - 1) / (block / 64);
    if (persistent) {
        int per_cu = 0;
        hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, block, lds);
        if (e != hipSuccess) return e;
        const int64_t resident = (int64_t)std::max(1, per_cu) * std::max(1, num_cus);
        const int64_t groups = (a.n + rays - 1) / rays, waves = resident * (block / 64);
        if (a.sweep && groups > waves) {
            a.sweep_waves = (int32_t)waves;
            const int64_t part = waves * a.sweep;
            grid = (groups + part - 1) / part * resident;
        } else if (a.sweep) {
            a.sweep = 0;
            a.refill = 64;
        } else {
            grid = a.n_dev ? resident : std::min<int64_t>(resident, groups);
        }
    }
    grid = std::max<int64_t>(1, grid);
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(block), lds, s, a);
    return hipGetLastError();
}

template <bool ANY, int TRI, bool EXACT>
hipError_t launch_wide(const TraceArgs &a, bool persistent, int S, int block, int num_cus, hipStream_t s) {
    // S entries for any-hit launches (4 bytes each), 3/4 S for closest-hit ones (8 bytes)
    const size_t lds = (ANY ? (size_t)S * 4 : (size_t)S * 6) * block;
    switch (S) {
        case 8: return launch_k(k_trace_wide<ANY, ANY ? 8 : 6, TRI, EXACT>, a, persistent, block, lds, num_cus, s);
        case 16: return launch_k(k_trace_wide<ANY, ANY ? 16 : 12, TRI, EXACT>, a, persistent, block, lds, num_cus, s);
        case 24: return launch_k(k_trace_wide<ANY, ANY ? 24 : 18, TRI, EXACT>, a, persistent, block, lds, num_cus, s);
        case 32: return launch_k(k_trace_wide<ANY, ANY ? 32 : 24, TRI, EXACT>, a, persistent, block, lds, num_cus, s);
        default: return hipErrorInvalidValue;
    }
}

template <int V, bool ANY, int TRI>
hipError_t launch_s(const TraceArgs &a, bool persistent, int S, int block, int num_cus, hipStream_t s) {
    const size_t lds = (size_t)S * block * sizeof(int);
    switch (S) {
        case 8: return launch_k(k_trace<V, ANY, 8, TRI>, a, persistent, block, lds, num_cus, s);
        case 16: return launch_k(k_trace<V, ANY, 16, TRI>, a, persistent, block, lds, num_cus, s);
        case 24: return launch_k(k_trace<V, ANY, 24, TRI>, a, persistent, block, lds, num_cus, s);
        case 32: return launch_k(k_trace<V, ANY, 32, TRI>, a, persistent, block, lds, num_cus, s);
        default: return hipErrorInvalidValue;
    }
}

// The four-child walk where the scene has that tree (wide.hip builds it where it pays),
// the two-child loop of the asked variant elsewhere.
template <bool ANY, int TRI>
hipError_t launch_v(const TraceArgs &a, bool persistent, int variant, int S, int block, int num_cus, hipStream_t s) {
    // exact closest hits: by the reference's test, on scenes where kNoise's widened boxes pay
    // (wide_reach: build_wide); the two-sided test accepts any det but 0, which bounds nothing
    constexpr bool kBounded = !ANY && TRI == kTriReference;
    const bool exact = !ANY && variant == 0;
    if (a.wide && !(exact && !(kBounded && a.wide_reach > 0.0f))) {
        // refill 0 and the count known here: sweeps of 4 groups per wave, taking rays at 32
        // idle lanes. Against one wave per group and one persistent range (us): 1M shadow
        // rays 556 / 386, with sweeps 389; 1.8M rays in 250k triangles 960 / 846, 846, its
        // camera half 425 / 383, 385; 8.3M unsorted rays in 1M triangles 3915 / 4028, 3783.
        // (2 groups: 470, 882, 3736; 8 groups: 386, 837, 3904.) A renderer's camera rays,
        // many through one pixel, are the exception: 1080p at 64 samples 102.7 ms with one
        // wave per group, 105.3 in sweeps, 110.1 persistent; their count is on the device.
        TraceArgs b = a;
        if (!persistent && !a.n_dev) {
            b.sweep = 4;
            b.refill = 32;
        }
        if (exact) return launch_wide<ANY, TRI, kBounded>(b, persistent || b.sweep, S, block, num_cus, s);
        return launch_wide<ANY, TRI, false>(b, persistent || b.sweep, S, block, num_cus, s);
    }
    if (variant == 0) return launch_s<0, ANY, TRI>(a, persistent, S, block, num_cus, s);
    if (variant == 1) return launch_s<1, ANY, TRI>(a, persistent, S, block, num_cus, s);
    return hipErrorInvalidValue;
}

}  // namespace

hipError_t launch_trace_record(const TraceArgs &a, int variant, int pass, int block, int refill, int num_cus,
                               hipStream_t s) {
    if (a.n <= 0) return hipSuccess;
    if (block < 64 || block > 256 || block % 64 != 0) return hipErrorInvalidValue;
    TraceArgs b = a;
    b.xcd_order = 0;
    const bool persistent = refill > 0;
    b.refill = persistent ? (refill > 64 ? 64 : refill) : 64;
    const size_t lds = (size_t)16 * block * sizeof(int);
#define TT_REC(V, P) \
    if (variant == V && pass == P) return launch_k(k_trace<V, false, 16, kTriReference, P>, b, persistent, block, lds, num_cus, s);
    TT_REC(0, 1) TT_REC(0, 2) TT_REC(0, 3) TT_REC(1, 1) TT_REC(1, 2) TT_REC(1, 3)
#undef TT_REC
    return hipErrorInvalidValue;
}

hipError_t launch_trace(const TraceArgs &a, int variant, bool any, int lds_stack, int block, int xcd_order,
                        int refill, int num_cus, hipStream_t s, int tri_mode) {
    if (a.n <= 0) return hipSuccess;
    if (block < 64 || block > 256 || block % 64 != 0) return hipErrorInvalidValue;
    TraceArgs b = a;
    b.xcd_order = xcd_order ? 1 : 0;
    // refill 0: one wave per 64-ray group; 1..64: persistent waves with that threshold
    const bool persistent = refill > 0;
    b.refill = persistent ? (refill > 64 ? 64 : refill) : 64;
    // Few rays are spread over the chip: with fewer than 64 for each of 8 waves per CU a group
    // shrinks: a wave takes as many rounds as its rays ask for in turn, fewer rays ask for
    // fewer, and there is room for more waves. Any-hit rays in 223k records,
    // closest-hit rays in 550k, us, groups of 64 / 4 waves per CU / 8 / 16 / 32: 1000 rays 113
    // / 75 / 73 / 76 / 73 and 143 / 97 / 96 / 102 / 98; 10000: 138 / 123 / 116 / 117 / 125 and
    // 212 / 180 / 181 / 163 / 164; 50000: 190 / 188 / 181 / 175 / 182 and 273 / 272 / 281 / 266
    // / 268; 200000 (64 rays at 8 waves): 245 / 248 / 247 / 247 / 261 and 321 / 322 / 320 / 321
    // / 337. Guided render 12.75 / 12.58 / 12.58 / 12.69 / 13.29 ms, room of 20 triangles 2089
    // / 2091 / 2096 / 2106 / 2143 us.
    for (b.spread = 0; 8LL * std::max(1, num_cus) >> (b.spread + 1);) ++b.spread;
    // ray indices are 32-bit in the kernel: more rays go in several launches, but one with a
    // device-side count or an order, which have fewer
    constexpr int64_t kMost = ((int64_t)1 << 31) - 1;
    const bool whole = a.n_dev || a.order;
    if (whole && a.n > kMost) return hipErrorInvalidValue;
    const int64_t part = whole ? a.n : (int64_t)1 << 30;
    for (int64_t at = 0; at < a.n; at += part) {
        b.n = std::min(part, a.n - at);
        b.rays = a.rays + at;
        if (a.hits) b.hits = a.hits + at;
        if (a.flags) b.flags = a.flags + at;
        if (a.ray_root) b.ray_root = a.ray_root + at;
        hipError_t e = hipErrorInvalidValue;
        if (tri_mode == kTriReference)
            e = any ? launch_v<true, kTriReference>(b, persistent, variant, lds_stack, block, num_cus, s)
                    : launch_v<false, kTriReference>(b, persistent, variant, lds_stack, block, num_cus, s);
        else if (tri_mode == kTriTwoSided)
            e = any ? launch_v<true, kTriTwoSided>(b, persistent, variant, lds_stack, block, num_cus, s)
                    : launch_v<false, kTriTwoSided>(b, persistent, variant, lds_stack, block, num_cus, s);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace tt
