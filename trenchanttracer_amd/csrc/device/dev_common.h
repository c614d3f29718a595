// Device-side shared definitions (gfx950, wave64).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../../include/tt.h"

namespace tt {

constexpr int kSentinel = 0x76543210;  // IntersectKernel.cuh:9
constexpr int kStackCap = 72;          // >= 64 outstanding pushes (tree depth <= 64)
constexpr int kWideCap = 48;           // entries of the wide walk's stack

// A queue filled by the blocks of one kernel and read by the next, in kSegs segments with a
// counter each: block b appends to segment b % kSegs. Atomic adds from all XCDs to one address
// take about 13 ns each, which bounded the shade kernels behind one counter (16384 blocks of
// a 256 x 256 render: 231 us, in 4 segments 159; 8 segments are no faster, and cost their
// readers more). The counters lie in lines of their own (side by side the kernels take four
// times as long). Readers go through the segments in turn, 64 entries each, which keeps the
// order the blocks wrote in as far as the counts agree; position r of that sequence holds no
// entry where its segment has ended. One counter / 4 segments / 8, us: 256 x 256 room 2093 /
// 1744 / 1780, reference mode 256 x 256 1104 / 981 / 984, its 640 x 360 frames 4110 / 3985 /
// 3995; under a sky 1080p 91.5 / 91.8 / 92.9 ms, a batch 12.19 / 12.20 / 12.35, guided 12.49 /
// 12.53 / 12.87 (their traversals follow the order a little less closely).
constexpr int kSegs = 4;
constexpr int kSegStride = 64;   // counter of segment s: counts[s * kSegStride]
struct Queue {
    const int32_t *counts;
    int32_t seg;                 // entries a segment can hold (0: one run of counts[0] entries)
};
// positions of the sequence
__device__ __forceinline__ int32_t queue_span(const Queue &q) {
    if (!q.seg) return q.counts[0];
    int32_t most = 0;
    for (int s = 0; s < kSegs; ++s) most = max(most, q.counts[s * kSegStride]);
    return (most + 63) / 64 * (64 * kSegs);
}
__device__ __forceinline__ int32_t queue_total(const Queue &q) {
    int32_t n = q.counts[0];
    for (int s = 1; q.seg && s < kSegs; ++s) n += q.counts[s * kSegStride];
    return n;
}
__device__ __forceinline__ int segment_of(int32_t r) { return (r >> 6) % kSegs; }
__device__ __forceinline__ int32_t entry_of(int32_t r) { return (r / (64 * kSegs) << 6) | (r & 63); }
__device__ __forceinline__ int32_t position_of(int s, int32_t entry) {
    return ((entry >> 6) * kSegs + s) * 64 + (entry & 63);
}
// slot of position r in the queue's arrays, -1 where there is no entry
__device__ __forceinline__ int32_t queue_slot(const Queue &q, int32_t r) {
    if (!q.seg) return r;
    const int s = segment_of(r);
    const int32_t i = entry_of(r);
    return i < q.counts[s * kSegStride] ? s * q.seg + i : -1;
}

// How far from its triangle a hit accepted by the reference's test can lie. With n = 2^-24 and
// w = o - v0, the test computes pv = d x e2 and qv = w x e1 to 2.42 n of the product of the
// factors' lengths (1.42 from the products, 1 from the differences), and from them det = e1 pv,
// Nu = w pv, Nv = d qv and Nt = e2 qv, each sum of three products to 2 n of its factors' lengths
// and its last rounding. Exactly, det w + Nt d = Nu e1 + Nv e2. An error e of pv enters that as
// (e1 e) w - (w e) e1 = e x (w x e1), one of qv in the same way, so together 4.84 n |e1||e2||d||w|,
// and the four sums 8 n of it. Hence, but for the unamplified roundings (of w, the last ones of
// the sums, the divide: 9 n of the coordinates),
//   |o + t d - (v0 + u e1 + v e2)| <= 12.9 n |e1||e2||d||w| / det,   det > 1e-5.
// (The largest found over 20M accepted rays nearly in their triangles' planes, edges of 1e-3 to
// 50, from 0.01 to 1000 away: 5.0 n.) The factor holds 1% for its own rounding.
constexpr float kNoise = 12.9f * 0x1p-24f / 1e-5f * 1.01f;

constexpr float kUnitLength = 1.02f;   // directions up to this length count as unit ones

struct TraceArgs {
    const float4 *nodes;   // 4 float4 per node
    const float4 *tris;    // 3 float4 per triangle record
    const tt_ray *rays;
    tt_hit *hits;          // closest-hit output (or nullptr)
    int32_t *flags;        // any-hit output (or nullptr)
    int64_t n;
    int32_t num_nodes;
    const uint4 *wide;        // four-child tree and its triangle records (nullptr: walk the two-child one)
    int32_t wide_step;        // 16-byte units from one record of it to the next
    float wide_bound;         // largest coordinate of a plane
    float wide_mid[3], wide_half[3];   // the scenes' box: centre and half extent (rounded up)
    float wide_noise;         // kNoise times the unit of the nodes' size codes (wide.hip)
    float wide_grain;         // length the sizes are taken against
    float wide_reach;         // exact closest hit: largest |d| times distance across the scenes
    const int32_t *ray_root;  // if set: scene of each ray (its root is that record of the wide tree)
    const int32_t *roots;     // if set: the scenes' roots in the two-child tree
    const int32_t *n_dev;  // if set: ray count read on the device (capped at n), or with seg set ...
    int32_t seg;           // ... the counts of a queue in segments of this capacity (Queue)
    int32_t *reset0;       // if set: the counts of a queue, zeroed by block 0
    int32_t *reset1;
    int32_t xcd_order;     // 1: each XCD (blocks b = x mod 8) holds one contiguous range of waves
    int32_t refill;        // a wave takes new rays once this many of its lanes are idle (1..64)
    int32_t sweep;         // if set: the range is traced in parts of this many groups per wave ...
    int32_t sweep_waves;   // ... and this many waves
    int32_t spread;        // if set: groups shrink to 2^k < 64 rays while there are at most 2^spread of them
    const uint32_t *order; // if set: the r-th ray traced is ray order[r] (a permutation of 0..n-1)
    // node-fetch probe (closest-hit loop): per ray the counts of node visits,
    // triangle tests and leaf visits, and from rec_off[ray] (32-bit words) the 4-bit
    // slab-test outcome of every node visit, 8 per word
    int32_t *rec_nodes;
    int32_t *rec_tris;
    int32_t *rec_leaves;
    int32_t *rec_log;
    const int64_t *rec_off;
};

// Triangle acceptance: the reference's test (front faces only, det > 1e-5) or
// a two-sided test with no epsilon (accept any det != 0) for the path tracer.
enum TriMode { kTriReference = 0, kTriTwoSided = 1 };

// Ray reordering (reorder.hip): workspace size for n rays (sort_bytes: the part the
// radix sort uses), and the permutation that sorts the rays by a Morton code of
// their origins within the box lo..hi.
hipError_t reorder_workspace_bytes(int64_t n, size_t *bytes, size_t *sort_bytes);
hipError_t reorder_rays(const tt_ray *rays, int64_t n, const float lo[3], const float hi[3], void *ws,
                        size_t sort_bytes, hipStream_t s, const uint32_t **order);
// The same for a queue whose length is read on the device (n_dev, capped at cap); the
// workspace is reorder_workspace_bytes(cap); launches sized for cap, blocks past the
// count leave at once.
hipError_t reorder_rays_dev(const tt_ray *rays, int64_t cap, const int32_t *n_dev, const float lo[3],
                            const float hi[3], void *ws, hipStream_t s, const uint32_t **order);

// Inversion of a float CDF (cdf[0] = 0, nondecreasing): the largest k in [lo, hi]
// with cdf[k] < u, or lo when there is none. Over [0, n - 1] this is the sampled
// entry: cdf[k] < u <= cdf[k + 1].
__device__ __forceinline__ int cdf_search_range(const float *cdf, int lo, int hi, float u) {
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (cdf[mid] < u) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// Guide-table cell of u in [0, 1) for a table of m cells; the build and the
// lookup use these same float operations.
__device__ __forceinline__ int guide_cell(float u, int m) { return min(m - 1, max(0, (int)(u * (float)m))); }

// CDF inversion through a guide table of n cells (Chen & Asau's index table):
// guide[c] holds the smallest and largest index the full search returns for any
// float u of cell c, so the search runs inside that range (usually 0-2 steps
// instead of log2 n) and returns the full search's index for every u.
__device__ __forceinline__ int cdf_search_guided(const float *cdf, const int2 *guide, int n, float u) {
    const int2 r = guide[guide_cell(u, n)];
    return cdf_search_range(cdf, r.x, r.y, u);
}

// One cell of a row's conditional guide table together with everything a sample drawn
// in it reads: the index range [lo, hi] the CDF search can return for a u of the cell,
// the CDF entries lo + 1 and lo + 2, and the texels (rgb, sampling weight) of columns
// lo, lo + 1 and lo + 2 (zero past the row's end). 64 bytes, so a next-event sample of
// the environment reads one record; ranges of more than three entries fall back to the
// CDF and texel arrays.
struct alignas(64) EnvCell {
    int32_t lo, hi;
    float c1, c2;
    float4 t[3];
};
static_assert(sizeof(EnvCell) == 64, "EnvCell is one 64-byte record");

// One cell of the marginal CDF's guide table: its search range and the CDF entries
// lo + 1, lo + 2 (16 bytes; ranges of more than three entries read the CDF).
struct alignas(16) MargCell {
    int32_t lo, hi;
    float c1, c2;
};

// Launchers (trace.hip).
hipError_t launch_trace(const TraceArgs &a, int variant, bool any, int lds_stack, int block, int xcd_order,
                        int refill, int num_cus, hipStream_t s, int tri_mode = kTriReference);
// The closest-hit loop (variant 0 or 1, LDS stack 16, reference triangle test) for
// the node-fetch probe: pass 1 counts (rec_nodes / rec_tris / rec_leaves), pass 2
// records the node visits' outcomes (rec_off, rec_log), pass 3 replays them,
// writing one 16-byte record per ray to hits.
hipError_t launch_trace_record(const TraceArgs &a, int variant, int pass, int block, int refill, int num_cus,
                               hipStream_t s);

}  // namespace tt
