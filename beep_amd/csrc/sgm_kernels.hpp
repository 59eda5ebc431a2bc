// sgm_kernels.hpp -- kernel-side data layout shared by the HIP kernels and the
// host engine.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace beep {

constexpr int kBlock = 256;     // threads per workgroup (4 wave64s)
constexpr int kMaxLevels = 10;  // query positions (DEPTH)

// Device-wide atomics on one address serialise across the whole GPU, so
// result accumulators and work cursors are spread over kStripes counters,
// one per 128-byte line of kLine u64 words.
constexpr int kLine = 16, kStripes = 16;

constexpr uint32_t kNoSplit = 1u << 20;  // KPlan::chunk: an item is a whole x_1

// Query plan as the kernels consume it (by value).  Level l in [2, L) is
// the candidate set C_l:
//   C_l = {i in [0,d) \ {x_1..x_{l-1}} : E[x_q][i] = 1 for q in qmask[l],
//          i > x_s for s in smask[l]}
// which is count_tri for l = 2 and compute_intersection for l >= 3
// (device_utils.cuh:179-209, 426-456).
struct KPlan {
    int32_t k;
    int32_t L;           // k - LUNMAT
    int32_t skip_split;  // skip x_1 < split(u) (sgm_kernelsLD.cuh:60)
    int32_t emit;        // BEEP_EMIT_*
    // LDS bitmap build: a row vertex whose larger-key range is longer than
    // bin_ratio x the row's partners (pair_partners) looks those up in the
    // range's lookup table instead of streaming the range (0: always, ~0u:
    // never)
    uint32_t bin_ratio;
    // Count-only plans whose last level L-1 does not intersect with the row
    // of x_{L-2}: C_{L-1} depends on x_{L-2} only through the exclusion of
    // x_{L-2} and, when L-2 is in smask[L-1], the bound x_{L-1} > x_{L-2}.
    // The kernels then sum |C_{L-1}| over all x_{L-2} in C_{L-2} in one pass
    // (prefix popcounts) instead of walking x_{L-2}.
    int32_t tail;
    // Count-only plans whose last three levels a = L-3, b = L-2, c = L-1 have
    //   qmask[c] = qmask[a] + {b},  smask[c] = smask[a] + {a},
    //   a in qmask[b], and qmask[b] - {a}, smask[b] below a:
    // x_c ranges over the same set S = C_a as x_a, restricted to the row of
    // x_b and above x_a, and x_b does not depend on x_a otherwise.  For fixed
    // x_1..x_{a-1}, the levels a..c then add up to
    //   sum over x_b in B of C(|S n E[x_b]|, 2),
    // B = the candidates of b without the a constraints (hub + 4-cycle, W5).
    int32_t pair;
    // Every row a level intersects with is used above its own index only
    // (through the symmetry bounds): the bitmap builds set, of each adjacent
    // pair, only the bit in the row of the smaller index.
    int32_t upper;
    uint32_t qmask[kMaxLevels];
    uint32_t smask[kMaxLevels];
    // What is left to do for level l when the walk starts from an earlier
    // level's set: C_l = C_base with the rows rq, the bounds rs and the
    // exclusions rx applied (base 0: from all of [0, d)).  lev[l] holds
    // rq | rs << 16, lev[kMaxLevels + l] holds rx | base << 16.  For the last
    // level (L >= 4) they leave x_{L-2}'s constraints out: the rest, F, is the
    // same for every x_{L-2}, and leaf_row, leaf_gt and leaf_x say whether
    // x_{L-2} adds its row, the bound and its exclusion.
    uint32_t lev[2 * kMaxLevels];
    int32_t leaf_row, leaf_gt, leaf_x;
    // Every level is C_l = C_{l-1} n E[x_{l-1}] over bitmaps without mirrored
    // bits (cliques): one row per step, no bounds, no exclusions.
    int32_t nested;
    // x_2 candidates of one DFS item of the LDS batches (see lds_items).
    uint32_t chunk;
    int32_t deep;        // two or more levels are walked below x_2
    int32_t reads_rows;  // some level intersects with a bitmap row
    // Count-only plans whose count below x_1 is a function of |C_2| = c and
    // the root's row length d alone (diamond: c (c - 1) / 2); see closed_count.
    int32_t closed;
    int32_t kept;  // only bitmap rows from the split on are read
    int32_t hits;  // the LDS build counts the pairs it finds, no bitmap is needed
};

// KPlan::closed: triangle-like plans (L = 3), or a summed level 3 whose set is
// C_2 again (with or without x_3 > x_2), or all of the row but x_1 (and x_2).
enum { kOpen = 0, kClosedC = 1, kClosedPairs = 2, kClosedOrdered = 3, kClosedRow = 4 };
__host__ __device__ __forceinline__ uint64_t closed_count(int closed, uint64_t c, uint32_t d)
{
    return closed == kClosedC ? c
           : closed == kClosedPairs ? c * (c - 1u) / 2u
           : closed == kClosedOrdered ? c * (c - 1u)
                                      : c * (d - 2u);
}

// Whether the LDS batches of lane class lg walk this plan one item per lane
// (clique_walk), and the u64 words of LDS stack a thread then needs: the sets
// of levels 3..L-2 of 1 << lg words each, against one word per level for the
// lane groups (group_walk).  16 words (32 KB a workgroup) leave the widest
// class one workgroup per CU fewer; plans deeper than that keep the groups.
__host__ __device__ inline bool lds_lane_walk(const KPlan &pl, int lg)
{
    return pl.nested && lg <= 3 && ((pl.L - 4) << lg) <= 16;
}
__host__ __device__ inline uint32_t lds_stack_words(const KPlan &pl, int lg)
{
    const int group = pl.L > 3 ? pl.L - 3 : 1, lane = lds_lane_walk(pl, lg) ? (pl.L - 4) << lg : 0;
    return (uint32_t)(group > lane ? group : lane);
}

// What a launch needs of the LDS layout (see make_lds_layout).
struct LdsNeeds {
    uint32_t stack_words = 1;
    int levels = 3;
    bool rows = false, bitmap = false, walk = false;
    void add(const KPlan &pl, int lg)
    {
        const uint32_t w = lds_stack_words(pl, lg);
        if (w > stack_words) stack_words = w;
        if (pl.L > levels) levels = pl.L;
        rows |= pl.reads_rows != 0;
        bitmap |= pl.reads_rows && !pl.hits;
        walk |= !pl.closed;
    }
};

// Per-vertex record read when the vertex appears in a root's row: where its
// bitmap-build scan range starts in ocol and how long it is (one 16-byte
// gather instead of three scattered ones).
struct VInfo {
    uint64_t hbeg;  // rowptr[v] (+ nlow[v] for ascending rows)
    uint32_t hlen;  // neighbours with a larger key in the orientation's order
    uint32_t deg;
};

struct KGraph {
    const uint32_t *ocol;    // degree-oriented rows
    const VInfo *vinfo;      // n records
    // Lookup table of every vertex's larger-key range: the range [hbeg, hbeg +
    // hlen) hashed into the 2 hlen slots at 2 hbeg (key w + 1, 0 empty,
    // linear probing from lookup_slot(w, 2 hlen)).
    const uint32_t *htab;
    int32_t asc;             // rows ascend by (degree, id); else degree descends, ids ascend
};

// First slot of w in a lookup table of `size` slots (host and device).
__host__ __device__ __forceinline__ uint32_t lookup_slot(uint32_t w, uint32_t size)
{
    uint32_t h = w * 0x9E3779B1u;
    h ^= h >> 15;
    return (uint32_t)(((uint64_t)h * size) >> 32);
}

// Staged range of a row vertex: start (40 bits) and length (24 bits).
constexpr int kRangeShift = 40;

// Per-root record of an LDS batch, offsets relative to the batch.
struct RootRec {
    uint64_t rbeg;   // rowptr[u]
    uint32_t u;      // root vertex
    uint32_t d;      // degree
    uint32_t split;  // nlow[u]
    uint32_t doff;   // offset of the root's row in the batch's concatenated rows
    uint32_t eoff;   // offset of the root's bitmap (u64 words)
    uint32_t hoff;   // offset of the root's hash table (slots)
};

// Per-hub record (bitmap and hash table in HBM).
struct HubRec {
    uint64_t rbeg;   // rowptr[u]
    uint64_t eoff;   // bitmap offset in the arena (u64 words)
    uint64_t hoff;   // hash offset in the arena (slots)
    uint32_t u, d, split, hslots;
    uint64_t joff;   // first global row index of this hub (bitmap build)
    uint64_t ioff;   // first global DFS item of this hub
    uint32_t jbeg;   // first x_1 of the hub's items
    uint32_t rlo;    // first bitmap row kept (rows below are never read)
};

// Rows [row0, row0 + rows) of a hub's bitmap build, for hubs with at most
// kSliceKept kept rows (of those that keep rows from the split on only, with
// both bits of every pair): their vertices fit an LDS table. A limit of 512 or
// 2,048 rows measures the same (diamond on 1.1M vertices 359 us, a served mix
// of ten queries 4.35 ms).
struct SliceRec {
    uint32_t hub, row0, rows;
};
constexpr uint32_t kSliceKept = 1024, kSliceRows = 512;
constexpr uint64_t kSliceUnits = 3072;

// Donated level-2 subtree of a hub item: x_2 in C_2 n [lo, hi), with C_2
// published at slots[slot, slot + W).
struct HubChunk {
    uint32_t hub;
    uint32_t x1;
    uint64_t slot;
    uint32_t lo, hi;
};

// Every field defaults to null / 0, i.e. donation off, unless set on purpose.
struct HubQueue {
    HubChunk *q = nullptr;                    // null: donation off
    unsigned long long *tail = nullptr;       // records reserved
    unsigned long long *head = nullptr;       // striped cursor of the draining pass
    uint64_t cap = 0;
    uint64_t *slots = nullptr;                // published C_2 bitmaps
    unsigned long long *slot_tail = nullptr;  // words reserved
    uint64_t slot_cap = 0;
    unsigned long long *donated = nullptr;    // records published over the whole call
    uint32_t split_min = 0;                   // donate when |C_2| > split_min
    uint32_t chunk = 0;                       // candidates per record
};

// Hub items of 5-vertex plans with paired levels have a kernel of their own,
// for hubs of up to 2^20 - 1 neighbours (its counters' range).
__host__ __device__ inline bool hub_pair5(int L, bool pair, uint32_t wmax) { return pair && L == 5 && wmax < (1u << 14); }

// Words (u64) of one hub-DFS wave's buffer: nlev candidate-stack rows, the
// bitmap row of x_1 and, for paired levels over rows shorter than it, a list
// of kPairListWords words of S's members.
constexpr uint32_t kPairListWords = 256;
__host__ __device__ inline uint64_t hub_wave_words(int nlev, uint32_t wmax, bool pair)
{
    return (uint64_t)(nlev + 1) * wmax + (pair && wmax < kPairListWords ? kPairListWords : 0);
}

struct KOut {
    // kStripes lines: stripe s holds [0] count [1] hash_sum [2] hash_xor of
    // the waves that flush to it; word 3 of stripe 0 counts tuples written
    unsigned long long *acc = nullptr;
    uint32_t *buf = nullptr;  // device tuple buffer (cap * L words) or null
    uint64_t cap = 0;
    // Deadlines in wall_clock64() ticks, written on the device by the launch
    // sequence's first kernel (all ones: none): dl[0] for the hub kernels,
    // dl[1] for the LDS kernels.  Kernels stop claiming work and leave their
    // DFS once theirs has passed, and set *stop.
    const unsigned long long *dl = nullptr;
    unsigned long long *stop = nullptr;
    // kStripes lines of wall_clock64() stamps, cleared before: latest end of a hub
    // kernel (kStampHub), of lane class lg's launch (kStampEnd + lg), and in
    // stripe 0 the class's start (kStampStart + lg); or null.
    unsigned long long *stamp = nullptr;
    // Optional busy-time accumulators (wall_clock64 ticks), kProfPhases x
    // kProfSlots: phase 0 LDS workgroups, 1 hub waves on their own items, 2 hub
    // waves on donated subtrees, 3 the LDS workgroups' staging and bitmap
    // build; slot = workgroup (LDS) or wave (hub) index.  Phase 4 sums
    // phases 0-2 by compute unit (slot = XCC, shader engine, array, CU).
    unsigned long long *prof = nullptr;
};

// Words of a stamp stripe (KOut::stamp).
constexpr int kStampHub = 0, kStampEnd = 1, kStampStart = 8, kStampWords = 15;

constexpr int kProfSlots = 4096, kProfPhases = 5, kProfCuPhase = 4;

// One prepared query of a multi-query launch.
struct MultiQuery {
    KGraph g;
    KPlan pl;
    const RootRec *recs;
    const uint32_t *batch_first;
    const uint32_t *batch_count;
    KOut out;
};

// One LDS batch of one query.
struct MultiWork {
    uint32_t query;
    uint32_t batch;
    uint32_t lanes_log2;
    uint32_t pad;
};

}  // namespace beep
