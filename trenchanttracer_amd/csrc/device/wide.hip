// The four-child tree k_trace_wide walks, built on the GPU from the two-child SBVH when a
// scene is created.
//
// One array of records, nodes and triangles alike: 48 bytes (three 16-byte units) of
// content, 48 or 64 bytes apart (by the tree's size: build_wide); a
// reference is a unit index below 2^30, with the sign bit set for a leaf. The scenes'
// roots come first; a node's children lie together, inner nodes first, then the leaves'
// triangle records. The walk is bound by VALU issue and by vector memory lane loads, so a
// node is as few loads as four boxes and their children fit in, in the form that decodes
// with the fewest operations:
//   unit 0: origin x, y, z (floats), first unit of the child block
//   unit 1: per slot a byte {leaf, unit offset in the block}; the plane scales' exponents (x, y,
//           z as signed bytes), size code; x low planes (one byte per slot), x high planes
//   unit 2: y low, y high, z low, z high planes
// A plane is origin + byte * 2^exponent, rounded outwards. Slots hold the inner children,
// then the leaves by rising triangle count (which keeps the offsets small), then empty
// boxes. An empty box that the rounding allowance lets a ray enter leads to a leaf of the
// node once more, or, where it has none, to a record no ray hits: never to a node.
// The size code is for exact closest hits, whose boxes are widened by kNoise (dev_common.h)
// times |e1||e2||d||w|. For a hit at t, |w| is at most t |d| + M + the hit's own displacement,
// M the longer edge, so with |d| up to kUnitLength at most
//   (t |d| + grain) max(1, M / grain) / (1 - kNoise kUnitLength |e1||e2|);
// a triangle's size is |e1||e2| times the last two factors, and code^2 / 255^2 of the scene's
// largest bounds the sizes below the node. (A grain of 1/4 of the scenes' diagonal leaves the
// factors of all but large triangles at 1. 1/32, 1/16, 1/8, 1/4, 1 of it: camera rays in soup of
// 20k triangles 522, 323, 300, 287, 286 us, incoherent ones 430, 328, 329, 311, 317.)
// Children: starting from a two-child node's two, the inner child with the largest box is
// replaced by its own two while they fit (simulated on 1M-triangle soup: 24.2 visits of 3
// loads per incoherent ray against 50.6 of 4; eight children with 80-byte nodes: 16.7
// visits of 5). Triangle records are copied so that a node's leaves lie together; the
// second word's w is the leaf's place in the two-child tree (node * 2 + child), the third's
// the next record of the same triangle (a ring over its leaves), negative at a leaf's end.
// Above the place, two bits: 1 to 3 for a triangle that has a twin, which in each of its leaves
// lies that many records before it (another number in another leaf), so that the twin is tested
// before it, always. Triangles with equal centres, coincident ones, are made twins.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "../host/tt_host.h"
#include "dev_common.h"
#include "scene_dev.h"

namespace tt {
namespace {

constexpr int kMaxOffset = 127;   // largest unit offset of a slot
constexpr int32_t kNone = -2;               // no triangle id
constexpr float kMaxSize = 1e30f;           // of sizes that exact hits are widened for
constexpr int32_t kRingEnd = 0x7FFFFFFF;   // no unit index
constexpr float kGrain = 0.25f;
// Reaches at which the cost of boxes widened for exact hits is measured, in diagonals of the
// scenes' box (rule in build_wide)
constexpr int kReaches = 7;
__host__ __device__ constexpr float reach_of(int k) { return (float)(1 << k); }   // 1 ... 64

struct WideState {
    int32_t nodes, records;   // listed, allocated
    int32_t unfit;            // set: the tree does not fit
    int32_t built;            // nodes k_wide_top has built
    float most;               // the scenes' largest size (k_wide_sizes)
    int32_t pad;
    // Boxes entered per line through the scenes' box (sums of the boxes' areas over its own),
    // 32 fractional bits (whole numbers: the same sum in any order): [0] the boxes as they are,
    // [1] widened by the walk's rounding allowance, [2 + k] for exact hits up to reach_of(k)
    unsigned long long cost[2 + kReaches];
};

struct WideBuild {
    const float4 *nodes;
    const float4 *tris;
    const int32_t *roots;   // two-child roots of the scenes
    int32_t nroots;
    uint4 *wide;            // [step * record]
    int32_t step;           // units from one record to the next
    // breadth-first list of the nodes: record, and place in the two-child tree (node * 2 +
    // child; roots: unused)
    int2 *list;
    int32_t *parent;        // of a listed node, its parent's place in the list (roots: -1)
    int32_t *size;          // ... bits of its triangles' largest size (-1: no triangle)
    int32_t *last_of;       // [triangle id]: first unit of its record linked last, or -1
    int32_t *twin;          // ... the one before it, kNone where its leaves have none or others, or -1
    int32_t ids;            // triangle ids below this have a ring; others stand alone
    WideState *state;
    int32_t node_cap, rec_cap;
    float diagonal, area;     // of the scenes' box: length, half its surface
    float slack;              // what the rounding allowance adds to a box's extents
    float per_grain;
};

struct Child {
    float lo[3], hi[3];
    int32_t ref;      // two-child index: node, or ~first record
    int32_t place;    // node * 2 + child
    int32_t count;    // triangle records of a leaf (0: inner child)
    int32_t ref2, count2, place2;   // a second leaf merged into the slot (count2 0: none)
};

__device__ void box_of(const float4 *nodes, int32_t node, int c, Child &k) {
    const float4 xy = nodes[(int64_t)node * 4 + c];
    const float4 z = nodes[(int64_t)node * 4 + 2];
    k.lo[0] = xy.x;
    k.hi[0] = xy.y;
    k.lo[1] = xy.z;
    k.hi[1] = xy.w;
    k.lo[2] = c ? z.z : z.x;
    k.hi[2] = c ? z.w : z.y;
}

__device__ float half_area(const Child &k) {
    const float x = k.hi[0] - k.lo[0], y = k.hi[1] - k.lo[1], z = k.hi[2] - k.lo[2];
    return x * y + y * z + z * x;
}

// Appends the children of a two-child node to out; a leaf without triangles (one record
// with zero edges) is left out. False where a box is not finite, is inverted, or leaves
// the node's own (in): such trees keep the two-child walk alone.
__device__ bool add_children(const WideBuild &b, int32_t node, const Child *in, Child *out, int &n) {
    const int4 ch = reinterpret_cast<const int4 *>(b.nodes)[(int64_t)node * 4 + 3];
    for (int c = 0; c < 2; ++c) {
        Child k{};
        k.ref = c ? ch.y : ch.x;
        k.place = node * 2 + c;
        if (k.ref < 0) {
            const float4 *t = b.tris + (int64_t)~k.ref * 3;
            while (__float_as_int(t[3 * k.count + 2].w) == 0) ++k.count;
            ++k.count;
            if (k.count == 1 && t[1].x == 0.0f && t[1].y == 0.0f && t[1].z == 0.0f && t[2].x == 0.0f && t[2].y == 0.0f &&
                t[2].z == 0.0f)
                continue;
        }
        box_of(b.nodes, node, c, k);
        for (int q = 0; q < 3; ++q) {
            if (!(fabsf(k.lo[q]) < 0x1p60f && fabsf(k.hi[q]) < 0x1p60f && k.lo[q] <= k.hi[q])) return false;
            if (in && !(in->lo[q] <= k.lo[q] && k.hi[q] <= in->hi[q])) return false;
        }
        out[n++] = k;
    }
    return true;
}

// Whether the leaves among c[0, n) can be addressed: the inner children and all leaves but
// the largest lie before it.
__device__ bool leaves_fit(const Child *c, int n, int32_t step) {
    int64_t before = 0, most = 0;
    for (int k = 0; k < n; ++k) {
        before += c[k].count ? c[k].count : 1;
        most = max(most, (int64_t)c[k].count);
    }
    return (before - most) * step <= kMaxOffset;
}

__device__ int wave_scan(int v, int *total) {   // exclusive sum over the wave's lanes
    int s = v;
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(s, o);
        if ((int)__lane_id() >= o) s += y;
    }
    *total = __shfl(s, 63);
    return s - v;
}

// Equal to the rounding of its terms.
__device__ bool near(float x, float y, float v, float a, float b) {
    return fabsf(x - y) <= 0x1p-20f * (fabsf(v) + fabsf(a) + fabsf(b));
}

// (returns the largest size)
__device__ float copy_leaf(const WideBuild &b, int32_t ref, int32_t count, int32_t place, int32_t at, bool last) {
    float size = 0.0f;
    float3 centre[3];   // of the last three, the latest first
    int32_t ids[3] = {-1, -1, -1};
    const float4 *t = b.tris + (int64_t)~ref * 3;
    for (int i = 0; i < count; ++i) {
        const int32_t unit = b.step * (at + i);
        float4 *to = reinterpret_cast<float4 *>(b.wide) + unit;
        float4 e1 = t[3 * i + 1], e2 = t[3 * i + 2];
        // (edges too short for their squares count as 1e-18 long)
        const float n1 = sqrtf(fmaxf(e1.x * e1.x + e1.y * e1.y + e1.z * e1.z, 1e-36f));
        const float n2 = sqrtf(fmaxf(e2.x * e2.x + e2.y * e2.y + e2.z * e2.z, 1e-36f));
        const float far = 1.0f - kNoise * kUnitLength * n1 * n2;
        size = fmaxf(size, far >= 0.7f ? n1 * n2 * fmaxf(1.0f, fmaxf(n1, n2) * b.per_grain) / far * 1.00001f : INFINITY);
        const int32_t id = __float_as_int(t[3 * i].w);
        // the record before this one in the ring; the first closes it (k_wide_rings)
        int32_t link = id >= 0 && id < b.ids ? atomicExch(&b.last_of[id], unit) : unit;
        if (link < 0) link = kRingEnd;
        // (three times the centre; v0 + v0 + v0 + e1 + e2 whichever vertex comes first)
        const float4 v0 = t[3 * i];
        const float3 c = make_float3(3.0f * v0.x + (e1.x + e2.x), 3.0f * v0.y + (e1.y + e2.y), 3.0f * v0.z + (e1.z + e2.z));
        uint32_t back = 0;
        int32_t twin = kNone;
#pragma unroll
        for (int k = 2; k >= 0; --k)
            if (ids[k] >= 0 && near(c.x, centre[k].x, v0.x, e1.x, e2.x) && near(c.y, centre[k].y, v0.y, e1.y, e2.y) &&
                near(c.z, centre[k].z, v0.z, e1.z, e2.z)) {
                back = k + 1;
                twin = ids[k];
            }
        if (id >= 0 && id < b.ids) {
            const int32_t was = atomicCAS(&b.twin[id], -1, twin);
            if (was != -1 && was != twin) atomicExch(&b.twin[id], kNone);
        } else {
            back = 0;
        }
        for (int k = 2; k > 0; --k) {
            centre[k] = centre[k - 1];
            ids[k] = ids[k - 1];
        }
        centre[0] = c;
        ids[0] = id;
        e1.w = __int_as_float(place | (int32_t)(back << 30));
        e2.w = __int_as_float(link | (last && i + 1 == count ? (int32_t)0x80000000 : 0));
        to[0] = t[3 * i];
        to[1] = e1;
        to[2] = e2;
    }
    return size;
}

// Closes the rings: the record linked first (it holds kRingEnd) points to the one linked
// last. One thread per triangle id, which follows its ring to that record, and clears the twin
// bits of a triangle that has not the same one in all its leaves.
__global__ __launch_bounds__(256) void k_wide_rings(WideBuild b) {
    const int32_t id = blockIdx.x * 256 + threadIdx.x;
    if (id >= b.ids || b.last_of[id] < 0) return;
    const int32_t last = b.last_of[id];
    const bool twin = b.twin[id] >= 0;
    for (int32_t at = last;;) {
        int32_t *link = reinterpret_cast<int32_t *>(b.wide + at + 2) + 3;
        const int32_t v = *link;
        if (!twin) *(link - 4) &= 0x3FFFFFFF;
        if ((v & 0x7FFFFFFF) == kRingEnd) {
            *link = last | (v & (int32_t)0x80000000);
            return;
        }
        at = v & 0x7FFFFFFF;
    }
}

__global__ __launch_bounds__(256) void k_wide_clear(int32_t *p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = -1;
}

// Node i of the list, by one thread of a whole wave (live: there is such a node). A wave's
// child blocks come from one atomic add on the records, its inner children are listed (the
// next level) from another.
__device__ __forceinline__ void build_node(const WideBuild &b, const int32_t i, const bool live) {
    int32_t self_rec = 0;
    Child c[4];
    int n = 0;
    bool bad = false;
    if (live) {
        if (i < b.nroots) {
            self_rec = i;
            bad = !add_children(b, b.roots[i], nullptr, c, n);
        } else {
            self_rec = b.list[i].x;
            const int32_t p = b.list[i].y;
            Child self{};
            box_of(b.nodes, p >> 1, p & 1, self);
            const int4 ch = reinterpret_cast<const int4 *>(b.nodes)[(int64_t)(p >> 1) * 4 + 3];
            bad = !add_children(b, (p & 1) ? ch.y : ch.x, &self, c, n);
        }
        if (!bad && n == 2 && !leaves_fit(c, n, b.step)) {
            // two large leaves: one slot for both
            c[0].ref2 = c[1].ref;
            c[0].count2 = c[1].count;
            c[0].place2 = c[1].place;
            for (int q = 0; q < 3; ++q) {
                c[0].lo[q] = fminf(c[0].lo[q], c[1].lo[q]);
                c[0].hi[q] = fmaxf(c[0].hi[q], c[1].hi[q]);
            }
            n = 1;
        }
        bool shut[4] = {false, false, false, false};   // opening it would not fit
        while (!bad && n < 4) {
            int best = -1;
            float area = -1.0f;
            for (int k = 0; k < n; ++k)
                if (c[k].count == 0 && !shut[k] && half_area(c[k]) > area) {
                    area = half_area(c[k]);
                    best = k;
                }
            if (best < 0) break;
            Child two[2], trial[4];
            int m = 0, t = 0;
            bad = !add_children(b, c[best].ref, &c[best], two, m);
            for (int k = 0; k < n; ++k)
                if (k != best) trial[t++] = c[k];
            for (int k = 0; k < m; ++k) trial[t++] = two[k];
            if (bad) break;
            if (!leaves_fit(trial, t, b.step)) {
                shut[best] = true;
                continue;
            }
            // the slots moved: whatever was shut is tried again (it still does not fit)
            n = t;
            for (int k = 0; k < n; ++k) {
                c[k] = trial[k];
                shut[k] = false;
            }
        }
        // inner children, then leaves by rising count (insertion sort)
        for (int k = 1; k < n; ++k)
            for (int j = k; j > 0 && c[j].count < c[j - 1].count; --j) {
                const Child x = c[j];
                c[j] = c[j - 1];
                c[j - 1] = x;
            }
    }
    int inner = 0;
    int64_t records = 0;
    if (live && !bad)
        for (int k = 0; k < n; ++k) {
            inner += c[k].count == 0;
            records += c[k].count ? (int64_t)c[k].count + c[k].count2 : 1;
        }
    // the empty slots' leaf: the node's first, or a record of its own
    const bool no_leaf = live && !bad && n < 4 && inner == n;
    if (no_leaf) ++records;
    if (records > b.rec_cap) bad = true;
    int nodes_all = 0, recs_all = 0;
    int node0 = wave_scan(bad ? 0 : inner, &nodes_all);
    int rec0 = wave_scan(bad ? 0 : (int)records, &recs_all);
    int at[2] = {0, 0};
    if (__lane_id() == 63) {
        at[0] = atomicAdd(&b.state->nodes, nodes_all);
        at[1] = atomicAdd(&b.state->records, recs_all);
    }
    node0 += __shfl(at[0], 63);
    rec0 += __shfl(at[1], 63);
    if (!live) return;
    if (node0 < 0 || rec0 < 0 || (int64_t)node0 + inner > b.node_cap || (int64_t)rec0 + records > b.rec_cap) bad = true;
    if (bad) {
        b.state->unfit = 1;
        return;
    }
    // the box of all children, the scales and the planes
    float lo[3] = {0.0f, 0.0f, 0.0f}, hi[3] = {0.0f, 0.0f, 0.0f};
    for (int k = 0; k < n; ++k)
        for (int q = 0; q < 3; ++q) {
            lo[q] = k ? fminf(lo[q], c[k].lo[q]) : c[k].lo[q];
            hi[q] = k ? fmaxf(hi[q], c[k].hi[q]) : c[k].hi[q];
        }
    uint32_t code[3], planes[3][2] = {{0xFFFFFFFFu, 0u}, {0xFFFFFFFFu, 0u}, {0xFFFFFFFFu, 0u}};
    for (int q = 0; q < 3; ++q) {
        // the smallest power of two with 255 steps over the extent
        int e = -126;
        const double step = ((double)hi[q] - (double)lo[q]) / 255.0;
        if (step > 0.0) {
            const double m = frexp(step, &e);
            if (m == 0.5) --e;
            e = max(e, -126);
        }
        code[q] = (uint32_t)e & 255u;
        const double inv = ldexp(1.0, -e);
        for (int k = 0; k < n; ++k) {
            const uint32_t l = (uint32_t)floor(((double)c[k].lo[q] - (double)lo[q]) * inv);
            const uint32_t h = (uint32_t)ceil(((double)c[k].hi[q] - (double)lo[q]) * inv);
            if (l > 255u || h > 255u) {
                b.state->unfit = 1;
                return;
            }
            planes[q][0] = (planes[q][0] & ~(255u << (8 * k))) | l << (8 * k);
            planes[q][1] |= h << (8 * k);
        }
    }
    uint32_t offsets = 0;
    int32_t off = 0;
    float size = 0.0f;
    for (int k = 0; k < n; ++k) {
        if (c[k].count == 0) {
            b.list[node0 + k] = make_int2(rec0 + k, c[k].place);
            b.parent[node0 + k] = i;
            offsets |= (uint32_t)(b.step * off) << (8 * k);
            ++off;
            continue;
        }
        offsets |= (uint32_t)(128 | b.step * off) << (8 * k);
        size = fmaxf(size, copy_leaf(b, c[k].ref, c[k].count, c[k].place, rec0 + off, c[k].count2 == 0));
        if (c[k].count2)
            size = fmaxf(size, copy_leaf(b, c[k].ref2, c[k].count2, c[k].place2, rec0 + off + c[k].count, true));
        off += c[k].count + c[k].count2;
    }
    // up to the first ancestor that has as large a one from another child
    const int32_t bits = __float_as_int(size);
    for (int32_t j = i; j >= 0 && atomicMax(&b.size[j], bits) < bits;) j = b.parent[j];
    if (no_leaf) {
        // no edges (never accepted), no triangle, its own ring, the end of its leaf
        const int32_t unit = b.step * (rec0 + off);
        float4 *to = reinterpret_cast<float4 *>(b.wide) + unit;
        to[0] = make_float4(0.0f, 0.0f, 0.0f, __int_as_float(-1));
        to[1] = make_float4(0.0f, 0.0f, 0.0f, __int_as_float(0));
        to[2] = make_float4(0.0f, 0.0f, 0.0f, __int_as_float(unit | (int32_t)0x80000000));
    }
    for (int k = n; k < 4; ++k) offsets |= (uint32_t)(128 | b.step * inner) << (8 * k);
    uint4 *w = b.wide + b.step * self_rec;
    w[0] = make_uint4(__float_as_uint(lo[0]), __float_as_uint(lo[1]), __float_as_uint(lo[2]),
                      (uint32_t)(b.step * rec0));
    w[1] = make_uint4(offsets, code[0] | code[1] << 8 | code[2] << 16, planes[0][0], planes[0][1]);
    w[2] = make_uint4(planes[1][0], planes[1][1], planes[2][0], planes[2][1]);
}

// One level of the tree: nodes [first, first + count) of the list, one thread each.
__global__ __launch_bounds__(64) void k_wide_level(WideBuild b, int32_t first, int32_t count) {
    const int32_t i = first + (int32_t)(blockIdx.x * 64 + threadIdx.x);
    build_node(b, i, i < first + count);
}

// The levels from the roots down to the first with more nodes than one block has threads. A
// launch for each level, with its count read back, takes about 20 us more: creating a scene of
// 300 triangles 395 us, with this 321 (104 without the tree), of 2000 718 and 617, of 250k
// 12511 and 12337 (12078 with the sums of k_wide_sizes added by block).
constexpr int kTopThreads = 1024;
__global__ __launch_bounds__(kTopThreads) void k_wide_top(WideBuild b) {
    int32_t first = 0, count = b.nroots;
    while (count > 0 && count <= kTopThreads) {
        build_node(b, first + (int32_t)threadIdx.x, (int32_t)threadIdx.x < count);
        __syncthreads();
        first += count;
        const bool unfit = __hip_atomic_load(&b.state->unfit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
        count = unfit ? 0 : __hip_atomic_load(&b.state->nodes, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) - first;
        __syncthreads();
    }
    if (threadIdx.x == 0) b.state->built = first;
}

// Every node's size code into its record, and the cost of boxes widened by it. Bound by the
// atomic adds to the sums (13 ns each), so at most 256 blocks walk the nodes and add once each
// (200,000 nodes, a wave's sums added on their own: 305 us, with this 26).
constexpr int kSizeBlocks = 256;
__global__ __launch_bounds__(256) void k_wide_sizes(WideBuild b, int32_t count) {
    __shared__ unsigned long long sum[2 + kReaches];
    if (threadIdx.x < 2 + kReaches) sum[threadIdx.x] = 0;
    __syncthreads();
    float most = 0.0f;
    for (int32_t k = 0; k < b.nroots; ++k) most = fmaxf(most, __int_as_float(max(b.size[k], 0)));
    if (blockIdx.x == 0 && threadIdx.x == 0) b.state->most = most;
    unsigned long long cost[2 + kReaches] = {};
    for (int32_t i = blockIdx.x * 256 + threadIdx.x; i < count; i += gridDim.x * 256) {
        uint4 *w = b.wide + b.step * (i < b.nroots ? i : b.list[i].x);
        const uint4 q = w[1], r = w[2];
        const float share = __int_as_float(max(b.size[i], 0)) / most;
        const float code = most > 0.0f && most <= kMaxSize ? fminf(ceilf(sqrtf(share) * 255.01f), 255.0f) : 255.0f;
        w[1].y = (q.y & 0xFFFFFFu) | (uint32_t)code << 24;
        const float unit = 2.0f * kNoise * b.diagonal * most * (code * code / 65025.0f);
        const uint32_t lo[3] = {q.z, r.x, r.z}, hi[3] = {q.w, r.y, r.w};
        for (int k = 0; k < 4; ++k) {
            float size[3];
            for (int c = 0; c < 3; ++c)
                size[c] = ldexpf((float)((int)(hi[c] >> 8 * k & 255) - (int)(lo[c] >> 8 * k & 255)),
                                 (int)(int8_t)(q.y >> 8 * c & 255));
            if (size[0] < 0.0f) continue;   // an empty slot
#pragma unroll
            for (int f = 0; f < 2 + kReaches; ++f) {
                // (exact hits' allowance is four times that of others: kSlack)
                const float pad = f == 0 ? 0.0f : f == 1 ? b.slack : 4.0f * b.slack + unit * reach_of(f - 2);
                const float x = size[0] + pad, y = size[1] + pad, z = size[2] + pad;
                cost[f] += (unsigned long long)(fminf((x * y + y * z + z * x) / b.area, 1.0f) * 0x1p32f);
            }
        }
    }
#pragma unroll
    for (int f = 0; f < 2 + kReaches; ++f) {
        for (int o = 32; o > 0; o >>= 1) cost[f] += __shfl_down(cost[f], o);
        if (__lane_id() == 0) atomicAdd(&sum[f], cost[f]);
    }
    __syncthreads();
    if (threadIdx.x < 2 + kReaches) atomicAdd(&b.state->cost[threadIdx.x], sum[threadIdx.x]);
}

// Whether a random line through the tree's root box is expected to cost more than `limit`
// box pairs and triangle tests (the surface-area sum of BVHNode::computeSubtreeProbabilities:
// 2 per inner node, 1 per triangle, each weighted by its box's share of the root's area).
// Boxes below 1/256 of the root's area are left out, so the walk ends within 256 x limit nodes.
bool costs_more_than(const std::vector<int32_t> &nodes, int32_t root, double limit) {
    double sum = 2.0, root_area = -1.0;
    std::vector<int32_t> stack{root};
    while (!stack.empty() && sum <= limit) {
        const int32_t *w = &nodes[(size_t)stack.back() * 16];
        stack.pop_back();
        float f[12];
        std::memcpy(f, w, sizeof(f));
        double area[2];
        for (int c = 0; c < 2; ++c) {
            const double x = (double)f[4 * c + 1] - f[4 * c], y = (double)f[4 * c + 3] - f[4 * c + 2],
                         z = (double)f[9 + 2 * c] - f[8 + 2 * c];
            area[c] = x >= 0.0 && y >= 0.0 && z >= 0.0 ? x * y + y * z + z * x : 0.0;
        }
        if (root_area < 0.0) {
            const double x = std::max(f[1], f[5]) - (double)std::min(f[0], f[4]),
                         y = std::max(f[3], f[7]) - (double)std::min(f[2], f[6]),
                         z = std::max(f[9], f[11]) - (double)std::min(f[8], f[10]);
            root_area = x * y + y * z + z * x;
            if (!(root_area > 0.0 && root_area < INFINITY)) return false;
        }
        for (int c = 0; c < 2; ++c) {
            const double p = area[c] / root_area;
            sum += p * (w[12 + c] < 0 ? w[14 + c] : 2);
            if (w[12 + c] >= 0 && p >= 1.0 / 256) stack.push_back(w[12 + c]);
        }
    }
    return sum > limit;
}

}  // namespace

// Builds s->wide for the scene's uploaded two-child tree; roots: the scenes' root nodes
// (node 0 alone for a single scene). Leaves it null where the tree does not fit the format,
// memory is short, or rays are expected to be short: every ray then walks the two-child
// tree. The four-child walk has more to do per ray (setting up, checking its winner's leaf)
// and holds 6 waves per SIMD instead of 8; per node and triangle it is faster. Measured, by
// expected cost (closest hit, us, two-child / four-child): Cornell box with a 5120-triangle
// sphere 4.0, 64-spp reference render 2573 / 2703; closed room of 20 triangles 15, 64-spp
// render 2166 / 2341; soups of 524288 rays: 30 triangles 11, 38 / 38; 100 triangles 24,
// 79 / 68; 300 triangles 37, 130 / 97; 10000 triangles 155, 341 / 242.
tt_status build_wide(tt_scene *s, const std::vector<int32_t> &dev_nodes, const std::vector<int32_t> &roots) {
    // nodes at most as many as the two-child tree has; units below 2^30
    const int64_t recs = s->num_nodes + s->num_tris;
    if (s->num_nodes == 0 || recs >= (1 << 30) / 3) return TT_OK;
    // A tree past the L2s (8 of 4 MB) takes 64 bytes per record: a record then lies in one
    // 64-byte piece of memory instead of 1.5, which is what a miss fetches; a smaller one
    // stays packed. Measured with 48 / 64 bytes: any hit on soup, 1M rays, 223k records 378 /
    // 373 us, 448k 460 / 455, 909k 525 / 490, 1.6M 580 / 544; 1080p, 64 spp path tracing over
    // 1.76M records 96.2 / 91.9 ms; 540p guided render over 110k records 12.67 / 12.92 ms; 360p,
    // 4 spp over 110k records 2.60 / 2.69 ms, over 439k 3.60 / 3.68.
    constexpr int64_t kPacked = (32 << 20) / 48;
    const int32_t step = recs > kPacked && recs < (1 << 30) / 4 ? 4 : 3;
    constexpr double kShort = 20.0;
    if (std::none_of(roots.begin(), roots.end(), [&](int32_t r) { return costs_more_than(dev_nodes, r, kShort); }))
        return TT_OK;
    // the scenes' box, and its largest coordinate (a plane can lie one step past its box)
    double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY}, bound = 0.0;
    for (const int32_t r : roots) {
        float w[12];
        std::memcpy(w, &dev_nodes[(size_t)r * 16], sizeof(w));
        const int lo_at[3] = {0, 2, 8};
        for (int q = 0; q < 3; ++q) {
            const float *a = w + lo_at[q], *c = w + lo_at[q] + (q == 2 ? 2 : 4);
            for (const float *p : {a, c})
                if (p[0] <= p[1]) {   // a leaf without triangles has an inverted box
                    lo[q] = std::min(lo[q], (double)p[0]);
                    hi[q] = std::max(hi[q], (double)p[1]);
                    bound = std::max(bound, std::max(std::fabs((double)p[0]), std::fabs((double)p[1])));
                }
        }
    }
    if (!(bound < 0x1p60)) return TT_OK;
    void *mem = nullptr, *tmp = nullptr;
    const size_t bytes = (size_t)recs * step * 16;
    // triangle ids (0 .. max(id)): those of the scene's mesh, or of as many records as there are
    const int32_t ids = (int32_t)std::max<int64_t>(s->num_orig_tris, s->num_tris);
    const size_t nodes = (size_t)s->num_nodes, root_bytes = roots.size() * 4;
    if (hipMalloc(&mem, bytes) != hipSuccess ||
        hipMalloc(&tmp, sizeof(WideState) + nodes * 16 + (size_t)ids * 8 + root_bytes) != hipSuccess) {
        (void)hipGetLastError();
        if (mem) hipFree(mem);
        return TT_OK;
    }
    WideBuild b{};
    b.nodes = reinterpret_cast<const float4 *>(s->nodes);
    b.tris = reinterpret_cast<const float4 *>(s->tris);
    b.wide = static_cast<uint4 *>(mem);
    b.state = static_cast<WideState *>(tmp);
    b.list = reinterpret_cast<int2 *>(b.state + 1);
    b.parent = reinterpret_cast<int32_t *>(b.list + nodes);
    b.size = b.parent + nodes;
    b.last_of = b.size + nodes;
    b.twin = b.last_of + ids;
    int32_t *d_roots = b.twin + ids;
    b.roots = d_roots;
    b.step = step;
    b.nroots = (int32_t)roots.size();
    b.ids = ids;
    double x[3], half[3];
    for (int q = 0; q < 3; ++q) {
        x[q] = std::max(hi[q] - lo[q], 0.0);
        s->wide_mid[q] = x[q] > 0.0 ? (float)(0.5 * (lo[q] + hi[q])) : (float)lo[q];
        half[q] = std::max(hi[q] - s->wide_mid[q], s->wide_mid[q] - lo[q]);
        s->wide_half[q] = (float)(half[q] * 1.0001);
    }
    b.diagonal = (float)std::sqrt(x[0] * x[0] + x[1] * x[1] + x[2] * x[2]);
    b.per_grain = 1.0f / (b.diagonal * kGrain);
    b.slack = (float)bound * 0x1p-19f;   // two sides of 2^-21 (|o| + B), origins as far out as the scene
    b.area = (float)(x[0] * x[1] + x[1] * x[2] + x[2] * x[0]);
    b.node_cap = (int32_t)s->num_nodes;
    b.rec_cap = (int32_t)recs;
    WideState state{b.nroots, b.nroots, 0, 0, 0.0f, 0, {}};
    hipStream_t hs = s->ctx->stream;
    hipError_t err = hipMemcpyAsync(b.state, &state, sizeof(state), hipMemcpyHostToDevice, hs);
    if (err == hipSuccess) err = hipMemcpyAsync(d_roots, roots.data(), root_bytes, hipMemcpyHostToDevice, hs);
    if (err == hipSuccess) {
        const int64_t words = 2 * ((int64_t)nodes + ids);   // parent, size, last_of, twin
        hipLaunchKernelGGL(k_wide_clear, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, hs, b.parent, words);
        err = hipGetLastError();
    }
    if (err == hipSuccess) {
        hipLaunchKernelGGL(k_wide_top, dim3(1), dim3(kTopThreads), 0, hs, b);
        err = hipGetLastError();
    }
    if (err == hipSuccess) err = hipMemcpyAsync(&state, b.state, 16, hipMemcpyDeviceToHost, hs);
    if (err == hipSuccess) err = hipStreamSynchronize(hs);
    for (int32_t first = state.built; err == hipSuccess && first < state.nodes && state.unfit == 0;) {
        const int32_t count = state.nodes - first;
        hipLaunchKernelGGL(k_wide_level, dim3((unsigned)((count + 63) / 64)), dim3(64), 0, hs, b, first, count);
        err = hipGetLastError();
        first += count;
        if (err == hipSuccess) err = hipMemcpyAsync(&state, b.state, 16, hipMemcpyDeviceToHost, hs);
        if (err == hipSuccess) err = hipStreamSynchronize(hs);
    }
    if (err == hipSuccess && state.unfit == 0) {
        hipLaunchKernelGGL(k_wide_sizes, dim3((unsigned)std::min((state.nodes + 255) / 256, kSizeBlocks)), dim3(256), 0, hs, b,
                           state.nodes);
        if (ids > 0) hipLaunchKernelGGL(k_wide_rings, dim3((unsigned)((ids + 255) / 256)), dim3(256), 0, hs, b);
        err = hipGetLastError();
        if (err == hipSuccess) err = hipMemcpyAsync(&state, b.state, sizeof(state), hipMemcpyDeviceToHost, hs);
    }
    const hipError_t end = hipStreamSynchronize(hs);
    if (err == hipSuccess) err = end;
    hipFree(tmp);
    if (err != hipSuccess || state.unfit) {
        hipFree(mem);
        return err == hipSuccess ? TT_OK : fail(TT_ERR_DEVICE, std::string("scene tree: ") + hipGetErrorString(err));
    }
    // Far from the coordinates' origin the rounding allowance widens the boxes, which the two-child
    // walk has none of. Measured (400k rays, us, two-child loop / four-child walk): the unit cube of
    // 50k triangles at 0 365 / 302, offset by 1000 359 / 336, by 10000 366 / 567, by 100000 433 / 7679.
    const auto grown = [&](int k) { return (double)state.cost[k] / (double)state.cost[0]; };
    if (!(grown(1) <= 1.3)) {
        hipFree(mem);
        return TT_OK;
    }
    // Exact closest hits take the four-child walk where widening its boxes for rays from within
    // the scene adds less than 0.3 of them, and there for rays from as far away, or with
    // as long directions, as at most double them; the lanes of others walk the two-child tree.
    // Measured (1.2M rays, default configuration, us, two-child loop / widened walk, by cost): soup
    // of 250k triangles 1.02 1015 / 678, twice as large in all 1.27 1015 / 790, 2.8 times 1.57
    // 1015 / 958, 4 times 2.4 1015 / 1723; soup of 2000 1.22 466 / 376, 1.5 times 1.55 466 / 458;
    // 180k triangles of terrain 1.08 269 / 218, 1.24 269 / 259, 1.36 269 / 284; soup of 100k and a
    // floor quad 1.11 910 / 701, a larger one 1.47 910 / 1238. All rays too far: 1015 / 1637, 466 / 516.
    s->wide_grain = b.diagonal * kGrain;
    s->wide_noise = kNoise * state.most / (255.0f * 255.0f);
    s->wide_reach = 0.0f;
    if (state.most <= kMaxSize && grown(2) <= 1.3)
        for (int k = 0; k < kReaches && grown(2 + k) <= 2.0; ++k) s->wide_reach = b.diagonal * reach_of(k);
    s->wide = mem;
    s->wide_step = step;
    s->wide_bound = (float)(bound * (1.0 + 4.0 / 255.0)) * 1.0001f;
    s->bytes += bytes;
    return TT_OK;
}

}  // namespace tt
