// sgm_kernels.hip -- CDNA4 (gfx950) kernels of the enumeration path.
//
// The reference runs one persistent CUDA kernel in which a 320-thread block
// claims a root, builds the root's d x ceil(d/32) neighbourhood bitmap in
// global memory by binary search, and 16-lane partitions walk the DFS over
// 32-bit words (sgm_kernelsLD.cuh:7-273, device_utils.cuh:60-456).
//
// Here the same enumeration is organised for wave64:
//  * bitmap words are 64 bits; a DFS group is P lanes of one wave (P = 1..64,
//    lane i of a group owns word i), the next candidate is found with one wave
//    ballot over the group's words; cliques are walked one lane an item;
//  * roots whose bitmap fits are packed into LDS batches: a workgroup stages
//    the rows, an LDS hash (vertex -> row index) and the bitmaps, then its
//    lanes or groups claim items -- an x_1 with some of its x_2 -- from an LDS
//    counter; counts that follow from |C_2| need no walk;
//  * a root's adjacent pairs are found once each, from the endpoint with the
//    smaller (degree, id) key: by streaming the part of its oriented row that
//    holds larger keys, or, when that part is long next to what it can pair
//    with, by looking those vertices up in a hash table of it (one load each)
//    -- instead of d^2/2 binary searches;
//  * roots too large for LDS ("hubs") keep their bitmap in an HBM arena, built
//    by workgroups that each own a slice of a hub where few rows are kept, else
//    by grid-wide kernels, and every wave of the grid takes (hub, x_1) items,
//    so one hub is shared by the whole GPU.
//
// Candidate sets follow count_tri (device_utils.cuh:179-209) for level 2 and
// compute_intersection (:426-456) for deeper levels; counting stops at level
// L-1 = k-1-LUNMAT as backtrack does (:294-326).

#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>

#include "internal.hpp"
#include "sgm_kernels.hpp"

namespace beep {

// ------------------------------------------------------------------ helpers

// bits [0, d) of word w
__device__ __forceinline__ uint64_t valid_mask(uint32_t w, uint32_t d)
{
    const uint32_t lo = w << 6;
    if (lo + 64 <= d) return ~0ull;
    if (lo >= d) return 0ull;
    return (1ull << (d - lo)) - 1ull;
}

// bits > x of word w (explicit branches: shifts by 64 are never issued)
__device__ __forceinline__ uint64_t gt_mask(uint32_t x, uint32_t w)
{
    const uint32_t xw = x >> 6;
    if (xw > w) return 0ull;
    if (xw < w) return ~0ull;
    const uint32_t b = x & 63u;
    return b == 63u ? 0ull : (~0ull << (b + 1u));
}

__device__ __forceinline__ uint64_t bit_at(uint32_t x, uint32_t w)
{
    return (x >> 6) == w ? (1ull << (x & 63u)) : 0ull;
}

// bits < x of word w
__device__ __forceinline__ uint64_t lt_mask(uint32_t x, uint32_t w)
{
    const uint32_t xw = x >> 6;
    if (xw > w) return ~0ull;
    if (xw < w) return 0ull;
    return (1ull << (x & 63u)) - 1ull;
}

// Pairs (x, y) with x in S, y in F and y > x, inside one word: C(|S|, 2) when
// S = F, else a loop over the sparser operand.
__device__ __forceinline__ uint32_t pairs_in_word(uint64_t S, uint64_t F)
{
    if (S == F) {
        const uint32_t k = (uint32_t)__popcll(S);
        return k * (k - 1) / 2;
    }
    uint32_t n = 0;
    if (__popcll(S) <= __popcll(F)) {
        while (S) {
            const uint32_t b = (uint32_t)__builtin_ctzll(S);
            S &= S - 1;
            n += (uint32_t)__popcll((F >> b) >> 1);
        }
    } else {
        while (F) {
            const uint32_t b = (uint32_t)__builtin_ctzll(F);
            F &= F - 1;
            n += (uint32_t)__popcll(S & ((1ull << b) - 1ull));
        }
    }
    return n;
}

__device__ __forceinline__ uint32_t hash_slot(uint32_t v, uint32_t H)
{
    uint32_t h = v * 0x9E3779B1u;
    h ^= h >> 15;
    return h & (H - 1u);
}

// An adjacent pair (j, i) of an LDS neighbourhood bitmap (W words per row):
// both bits, or with `upper` only the one in the row of the smaller index
// (the symmetry bounds never read a row below its own index then).
__device__ __forceinline__ void set_pair(uint64_t *E, uint32_t W, uint32_t j, uint32_t i, int upper)
{
    if (!upper || i > j) atomicOr((unsigned long long *)&E[j * W + (i >> 6)], 1ull << (i & 63));
    if (!upper || j > i) atomicOr((unsigned long long *)&E[i * W + (j >> 6)], 1ull << (j & 63));
}

__device__ __forceinline__ uint64_t mix64(uint64_t z)
{
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}

__device__ __forceinline__ uint64_t hash_step(uint64_t h, int pos, uint32_t v)
{
    return mix64(h + 0x9e3779b97f4a7c15ull * (uint64_t)(pos + 1) + v);
}

__device__ __forceinline__ uint64_t wave_sum_u64(uint64_t v)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

__device__ __forceinline__ uint64_t wave_xor_u64(uint64_t v)
{
    for (int o = 32; o > 0; o >>= 1) v ^= __shfl_xor(v, o, 64);
    return v;
}

// Wave inclusive scan.
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v)
{
    const int lane = threadIdx.x & 63;
    for (int o = 1; o < 64; o <<= 1) {
        uint32_t y = __shfl_up(v, o, 64);
        if (lane >= o) v += y;
    }
    return v;
}

// Set bits of m below the lane.
__device__ __forceinline__ uint32_t bits_below(uint64_t m)
{
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

__device__ __forceinline__ uint32_t lane_u32(uint32_t v, uint32_t l)
{
    return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)l);
}

// Orders a wave's own LDS writes before its following reads by other lanes.
__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Deadline check: wall_clock64() is a constant-rate device clock.
__device__ __forceinline__ bool past(uint64_t dl) { return (uint64_t)wall_clock64() > dl; }

__device__ __forceinline__ void mark_stop(const KOut &out) { atomicOr(out.stop, 1ull); }

// DFS steps between two deadline checks.
constexpr uint32_t kClockEvery = 1024;

// Paired last levels of the hub DFS: bit-sliced counters of kPairSlices bits
// count up to kPairMembers members of S (more than any hub row holds below the
// root window's 100 x cutoff on graphs of up to 2^26 vertices).  The
// instantiation with them is held to 3 waves per SIMD (168 VGPRs, a few spilled).
constexpr int kPairSlices = 20;
constexpr uint32_t kPairMembers = (1u << kPairSlices) - 1u;
// A 5-vertex pair plan's hub item of more than kPairSplitWork member-rounds
// (|C_2| x rounds of 64 words of B) is donated in parts of about
// kPairChunkWork member-rounds, whole rounds each.
constexpr uint64_t kPairSplitWork = 1u << 11;
constexpr uint32_t kPairChunkWork = 1u << 10;

// Compute unit the wave runs on, as a slot below 2048: the XCC (HW_REG_XCC_ID
// bits 2:0) and, within it, shader engine, shader array and CU (HW_REG_HW_ID
// bits 15:8).  The reference reads %smid for its per-SM times (utils.cuh:66-99).
__device__ __forceinline__ uint32_t cu_slot()
{
    const uint32_t hw = __builtin_amdgcn_s_getreg((31 << 11) | (0 << 6) | 4);    // HW_ID, 32 bits
    const uint32_t xcc = __builtin_amdgcn_s_getreg((15 << 11) | (0 << 6) | 20);  // XCC_ID, 16 bits
    return ((xcc & 7u) << 8) | ((hw >> 8) & 0xffu);
}

// Busy time since t0 into phase `phase`, slot `slot`; phases 0-2 (work, not
// the build share) also into the compute unit's slot of phase kProfCuPhase.
__device__ __forceinline__ void prof_add(const KOut &out, int phase, uint32_t slot, uint64_t t0)
{
    if (out.prof) {
        const unsigned long long dt = (unsigned long long)((uint64_t)wall_clock64() - t0);
        atomicAdd(&out.prof[phase * kProfSlots + (slot % kProfSlots)], dt);
        if (phase < 3) atomicAdd(&out.prof[kProfCuPhase * kProfSlots + cu_slot()], dt);
    }
}

// Stamps the end of a workgroup (one thread calls it).
__device__ __forceinline__ void stamp_end(const KOut &out, int word)
{
    if (out.stamp)
        atomicMax(&out.stamp[(blockIdx.x % kStripes) * kLine + word], (unsigned long long)wall_clock64());
}

// Flushes per-lane accumulators: one atomic per wave and counter, into the
// wave's stripe.
__device__ __forceinline__ void flush_acc(const KOut &out, uint64_t cnt, uint64_t hs, uint64_t hx)
{
    cnt = wave_sum_u64(cnt);
    hs = wave_sum_u64(hs);
    hx = wave_xor_u64(hx);
    if ((threadIdx.x & 63) == 0) {
        const uint32_t wave = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
        unsigned long long *a = out.acc + (uint64_t)(wave % kStripes) * kLine;
        if (cnt) atomicAdd(&a[0], (unsigned long long)cnt);
        if (hs) atomicAdd(&a[1], (unsigned long long)hs);
        if (hx) atomicXor(&a[2], (unsigned long long)hx);
    }
}

// Claims up to `step` indices of [0, n) from a striped cursor (kStripes
// counters kLine words apart).  Part t of [0, n) holds the indices t,
// t + kStripes, t + 2 kStripes, ..., so every part walks the work in its
// order (heaviest first where the work is sorted so).  A claimant starts at
// part `home` and moves on once a part is exhausted; on entering a part, a
// plain load usually tells an exhausted one without an atomic.  k (start at
// 0) holds the parts left behind and whether the current part has been
// claimed from.  On success the claimed indices are first + q kStripes for
// q < count; returns false when every part is exhausted.
constexpr uint32_t kPartEntered = 1u << 16;
__device__ __forceinline__ bool claim_striped(unsigned long long *cur, uint64_t n, uint32_t home, uint32_t &k,
                                              uint64_t step, uint64_t &first, uint64_t &count)
{
    while ((k & 0xffffu) < (uint32_t)kStripes) {
        const uint32_t t = (home + (k & 0xffffu)) % kStripes;
        const uint64_t len = t < n ? (n - t + kStripes - 1) / kStripes : 0;
        unsigned long long *p = cur + (uint64_t)t * kLine;
        if (!(k & kPartEntered) && __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= len) {
            k = (k & 0xffffu) + 1;
            continue;
        }
        k |= kPartEntered;
        const uint64_t o = atomicAdd(p, (unsigned long long)step);
        if (o < len) {
            first = t + o * kStripes;
            count = o + step < len ? step : len - o;
            return true;
        }
        k = (k & 0xffffu) + 1;
    }
    return false;
}

// Hash of an empty prefix of a tuple of `len` vertices.
__device__ __forceinline__ uint64_t hash_seed(int len) { return 0x6a09e667f3bcc909ull ^ (uint64_t)len; }

// Emits the tuples (u, A[x_1], ..., A[x_{l-1}], A[i]) for every bit i of word
// w of the last level: hash accumulation and optional buffer append.  h is the
// hash of the first l entries.
template <class XGet>
__device__ __forceinline__ void emit_bits(const KOut &out, int l, uint32_t u, const uint32_t *A, uint64_t h,
                                          uint64_t t, uint32_t w, XGet xget, uint64_t &hs, uint64_t &hx)
{
    const int len = l + 1;
    uint64_t base = 0;
    if (out.buf) base = atomicAdd(&out.acc[3], (unsigned long long)__popcll(t));
    uint64_t idx = 0;
    while (t) {
        const uint32_t b = (uint32_t)__builtin_ctzll(t);
        t &= t - 1;
        const uint32_t vi = A[(w << 6) + b];
        const uint64_t hv = hash_step(h, l, vi);
        hs += hv;
        hx ^= hv;
        if (out.buf && base + idx < out.cap) {
            uint32_t *dst = out.buf + (base + idx) * (uint64_t)len;
            dst[0] = u;
            for (int q = 1; q < l; q++) dst[q] = A[xget(q)];
            dst[l] = vi;
        }
        idx++;
    }
}

template <class XGet>
__device__ __forceinline__ void emit_word(const KOut &out, const KPlan &pl, int l, uint32_t u,
                                          const uint32_t *A, uint64_t t, uint32_t w, XGet xget,
                                          uint64_t &hs, uint64_t &hx)
{
    uint64_t h = hash_step(hash_seed(l + 1), 0, u);
    for (int q = 1; q < l; q++) h = hash_step(h, q, A[xget(q)]);
    emit_bits(out, l, u, A, h, t, w, xget, hs, hx);
}

// ------------------------------------------------------------ LDS batches

// Context of a row of an LDS batch that has build units (see find_pairs):
// streamed rows: unit e is ocol[base + e]; looked-up rows: unit e looks the row
// entry aoff + e up in the range whose hbeg | hlen << kRangeShift is `base`.
struct alignas(16) RowCtx {
    uint64_t base;
    uint32_t aoff;
    uint32_t info;  // row (9 bits) | looked up << 9 | filter word << 10 (10) | filter bits' log2 << 20
};

// Units of the tile of build work whose row starts are marked at once, and the
// entries of a wave's queue of probable pairs.
constexpr uint32_t kTile = 4096, kQueue = 128;

// What the build needs (hash, filter, row contexts, marks, queues) and what the
// walk needs (items, stack, x) share the space after `shared`.
struct LdsLayout {
    uint32_t oE, oRoot, oA, oMisc, oJRoot;
    uint32_t oCtx, oQ, oMark, oHKey, oFlt, oHVal;  // build
    uint32_t oStk, oPre, oX;                       // walk
    uint32_t bytes;
};

__host__ __device__ inline uint32_t align_up(uint32_t x, uint32_t a) { return (x + a - 1) / a * a; }

// Layout of lane class lg's batches; stack_words words of DFS stack and
// `levels` positions of x are kept per thread.
__host__ inline LdsLayout make_lds_layout(int lg, const LdsNeeds &need)
{
    const uint32_t sd = LdsBudget::sumdeg(lg), hs = LdsBudget::hash(lg);
    LdsLayout L{};
    uint32_t o = 0;
    // past the last row's words, clique_walk reads up to 7 more
    L.oE = o;       o += need.bitmap ? (LdsBudget::ewords(lg) + 8) * 8 : 0;
    L.oRoot = o;    o += LdsBudget::kMaxRoots * (uint32_t)sizeof(RootRec);
    L.oA = o;       o += sd * 4;
    L.oMisc = o;    o += 32 * 4;
    L.oMark = o;    o += kTile / 8;
    L.oJRoot = o;   o += sd;
    const uint32_t shared = align_up(o, 16);
    o = shared;
    if (need.rows) {
        L.oCtx = o;     o += sd * (uint32_t)sizeof(RowCtx);
        L.oQ = o;       o += (kBlock / 64) * kQueue * 8;
        L.oHKey = o;    o += hs * 4;
        L.oFlt = o;     o += hs / 2 * 4;
        L.oHVal = o;    o += hs * 2;
    }
    const uint32_t build = o;
    o = shared;
    if (need.walk) {
        L.oStk = o;     o += need.stack_words * kBlock * 8;
        L.oPre = o;     o += align_up((sd + 1) * 4, 8);
        L.oX = o;       o += (uint32_t)need.levels * kBlock * 2;
    }
    L.bytes = align_up(o > build ? o : build, 16);
    return L;
}

// Misc slots
enum { M_BATCH = 0, M_NEXT = 1, M_LEV = 4 };  // M_LEV: 2 kMaxLevels words (KPlan::lev); 24..31: scans

// Block-wide exclusive scan of a[0..n) in place (n <= 4 * kBlock); a[n] = total.
__device__ void block_excl_scan(uint32_t *a, uint32_t n, uint32_t *tmp4)
{
    const int tid = threadIdx.x;
    const int per = (int)((n + kBlock - 1) / kBlock);
    const uint32_t b = (uint32_t)(tid * per);
    uint32_t loc = 0;
    for (int i = 0; i < per; i++)
        if (b + i < n) loc += a[b + i];
    uint32_t inc = wave_incl_scan(loc);
    const int wv = tid >> 6;
    if ((tid & 63) == 63) tmp4[wv] = inc;
    __syncthreads();
    uint32_t wofs = 0;
    for (int i = 0; i < wv; i++) wofs += tmp4[i];
    uint32_t run = wofs + inc - loc;
    for (int i = 0; i < per; i++)
        if (b + i < n) {
            uint32_t x = a[b + i];
            a[b + i] = run;
            run += x;
        }
    if (tid == kBlock - 1) a[n] = run;
    __syncthreads();
}

// LDS carve-up of one workgroup.
struct LdsView {
    uint64_t *sE, *sStk, *sMark, *sQ;
    RootRec *sRoot;
    RowCtx *sCtx;
    uint32_t *sA, *sPre, *sHKey, *sFlt, *sMisc;
    uint16_t *sHVal, *sX;
    uint8_t *sJRoot;
};

__device__ __forceinline__ LdsView lds_view(unsigned char *smem, const LdsLayout &lay)
{
    LdsView v;
    v.sE = (uint64_t *)(smem + lay.oE);
    v.sStk = (uint64_t *)(smem + lay.oStk);
    v.sMark = (uint64_t *)(smem + lay.oMark);
    v.sQ = (uint64_t *)(smem + lay.oQ);
    v.sRoot = (RootRec *)(smem + lay.oRoot);
    v.sCtx = (RowCtx *)(smem + lay.oCtx);
    v.sA = (uint32_t *)(smem + lay.oA);
    v.sPre = (uint32_t *)(smem + lay.oPre);
    v.sHKey = (uint32_t *)(smem + lay.oHKey);
    v.sFlt = (uint32_t *)(smem + lay.oFlt);
    v.sMisc = (uint32_t *)(smem + lay.oMisc);
    v.sHVal = (uint16_t *)(smem + lay.oHVal);
    v.sX = (uint16_t *)(smem + lay.oX);
    v.sJRoot = (uint8_t *)(smem + lay.oJRoot);
    return v;
}

// The items a workgroup takes of a batch: those congruent to part modulo parts
// (see lds_batch_kernel).
struct Share {
    uint32_t part, parts;
};

// Rows whose index range holds item e: the largest j with pre[j] <= e (pre
// ascends, pre[n] > e).
__device__ __forceinline__ uint32_t find_row(const uint32_t *pre, uint32_t n, uint32_t e)
{
    uint32_t lo = 0, hi = n;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (pre[mid] <= e) lo = mid; else hi = mid;
    }
    return lo;
}

// The n lowest set bits of v (n <= popcount).
__device__ __forceinline__ uint64_t low_bits(uint64_t v, uint32_t n)
{
    uint64_t r = v;
    for (uint32_t i = 0; i < n; i++) r &= r - 1;
    return v ^ r;
}

__device__ __forceinline__ bool whole_rows(const KPlan &pl)
{
    return pl.chunk == kNoSplit && !pl.closed && !pl.nested;
}

// DFS items of a batch, once its bitmaps are there: row j (x_1 = j of its root)
// gives ceil(|C_2| / chunk) items, each the x_2 of `chunk` consecutive
// candidates, so a row with many candidates under a deep plan is walked by
// many lanes and an x_1 without candidates by none.  Leaves the rows' item
// offsets in sPre (sPre[sumd] = the number of items, also returned).  Plans whose
// count follows from |C_2| (KPlan::closed) are counted right here (no items),
// and where an item is a whole x_1 the rows themselves are the items.
//
// Why: with one item per x_1, a lane's serial chain under a 6-clique's x_1 ran
// 40 ms (R-MAT scale 17) while the GPU idled: mean/max workgroup time 0.07.
__device__ uint32_t lds_items(const KPlan &pl, const LdsView &v, uint32_t sumd, uint64_t &cnt)
{
    const int L = pl.L;
    if (whole_rows(pl)) return sumd;
    const bool row1 = (pl.qmask[2] & 2u) != 0, above = (pl.smask[2] & 2u) != 0;
    const uint32_t need = pl.nested ? (uint32_t)L - 2u : 1u;  // a clique's x_2..x_{L-1} all lie in C_2
    for (uint32_t j = threadIdx.x; j < sumd; j += kBlock) {
        const RootRec rr = v.sRoot[v.sJRoot[j]];
        const uint32_t jl = j - rr.doff, d = rr.d, W = (d + 63) >> 6;
        uint32_t c2 = 0;
        // x_1..x_{L-1} are distinct row entries
        if (!(pl.skip_split && jl < rr.split) && d + 1u >= (uint32_t)L) {
            if (row1) {
                const uint64_t *E = v.sE + rr.eoff + jl * W;
                for (uint32_t w = above ? jl >> 6 : 0u; w < W; w++)
                    c2 += (uint32_t)__popcll(above ? E[w] & gt_mask(jl, w) : E[w]);
            } else {
                c2 = above ? d - 1u - jl : d - 1u;
            }
        }
        if (pl.closed) cnt += c2 ? closed_count(pl.closed, c2, d) : 0ull;
        else v.sPre[j] = c2 < need ? 0u : pl.chunk == kNoSplit ? 1u : (c2 + pl.chunk - 1u) / pl.chunk;
    }
    if (pl.closed) return 0;
    __syncthreads();
    block_excl_scan(v.sPre, sumd, v.sMisc + 28);
    return v.sPre[sumd];
}

// Plans whose levels nest (KPlan::nested, cliques): every lane walks items of
// its own and holds all WT words of the current level's set in registers, so a
// step is one row read, WT ANDs and popcounts and no cross-lane traffic.
// E[x] holds bits above x only, so the candidates not yet taken are the whole
// set as far as the next level is concerned: one set per level is kept, in
// registers for the current level and in the LDS stack above it.
//
// Lanes of a wave are at different depths.  Each round first brings every lane
// that ran out of candidates to its next last-level set (climb, claim,
// descend), then steps all lanes through their sets until half of the lanes
// that still have work are out of candidates: the two phases' instructions are
// then paid by at least half of the lanes they serve.
template <int WT, bool EMIT>
__device__ void clique_walk(const KPlan &pl, const LdsView &v, uint32_t sumd, uint32_t items, Share sh,
                            const KOut &out, uint64_t dl, uint64_t &cnt, uint64_t &hs, uint64_t &hx)
{
    const int tid = threadIdx.x;
    const int L = pl.L;
    uint64_t *stk = v.sStk + tid;  // word k of level l's set: stk[((l - 3) * WT + k) * kBlock]
    uint16_t *sX = v.sX;
    auto xget = [&](int q) -> uint32_t { return sX[q * kBlock + tid]; };
    uint64_t S[WT];
#pragma unroll
    for (int k = 0; k < WT; k++) S[k] = 0ull;
    int l = 3;             // S = what is left of C_{l-1}; x_{l-1} is taken next
    uint32_t left = 0;     // x_2's of the item not yet taken
    bool live = true;
    const uint64_t *E = v.sE;
    const uint32_t *A = v.sA;
    uint32_t W = 1, u = 0;
    uint32_t rounds = 0;
    uint64_t hpre = 0;  // EMIT: hash of u, x_1..x_{L-3}
    auto any = [&]() -> bool {
        uint64_t o = S[0];
#pragma unroll
        for (int k = 1; k < WT; k++) o |= S[k];
        return o != 0ull;
    };
    // takes the smallest candidate out of S (not empty)
    auto take = [&]() -> uint32_t {
        uint32_t k0 = 0;
        uint64_t c = S[0];
#pragma unroll
        for (int k = 1; k < WT; k++)
            if (c == 0ull) {
                c = S[k];
                k0 = k;
            }
#pragma unroll
        for (int k = 0; k < WT; k++)
            if ((uint32_t)k == k0) S[k] = c & (c - 1ull);
        return (k0 << 6) + (uint32_t)__builtin_ctzll(c);
    };
    for (;;) {
        // ---- bring every lane to a last-level set
        while (live && !(l == L - 1 && any())) {
            if (l > 3 && !any()) {  // climb
                --l;
#pragma unroll
                for (int k = 0; k < WT; k++) S[k] = stk[((l - 3) * WT + k) * kBlock];
            } else if (l == 3 && (left == 0 || !any())) {  // claim
                // one LDS atomic for the lanes that claim together
                const uint64_t m = __ballot(1);
                const uint32_t rank = bits_below(m);
                uint32_t first = 0;
                if (rank == 0) first = atomicAdd(&v.sMisc[M_NEXT], (uint32_t)__popcll(m));
                const uint32_t item = ((uint32_t)__builtin_amdgcn_readfirstlane((int)first) + rank) * sh.parts + sh.part;
                if (item >= items) {
                    live = false;
#pragma unroll
                    for (int k = 0; k < WT; k++) S[k] = 0ull;
                } else {
                    const uint32_t row = find_row(v.sPre, sumd, item);
                    const RootRec rr = v.sRoot[v.sJRoot[row]];
                    const uint32_t jl = row - rr.doff;
                    W = (rr.d + 63) >> 6;
                    E = v.sE + rr.eoff;
                    uint32_t skip = 0;
                    left = 0xffffffffu;
                    if (pl.chunk != kNoSplit) {
                        skip = (item - v.sPre[row]) * pl.chunk;
                        left = pl.chunk;
                    }
#pragma unroll
                    for (int k = 0; k < WT; k++) {
                        uint64_t c = (uint32_t)k < W ? E[jl * W + k] : 0ull;
                        if (skip) {
                            const uint32_t pc = (uint32_t)__popcll(c);
                            const uint32_t drop = skip < pc ? skip : pc;
                            c ^= low_bits(c, drop);
                            skip -= drop;
                        }
                        S[k] = c;
                    }
                    if (EMIT) {
                        A = v.sA + rr.doff;
                        u = rr.u;
                        sX[1 * kBlock + tid] = (uint16_t)jl;
                        if (L == 4) hpre = hash_step(hash_step(hash_seed(L), 0, u), 1, A[jl]);
                    }
                }
            } else {  // descend: l < L - 1 and a candidate is left
                const uint32_t x = take();
                if (l == 3) left--;
                uint64_t t[WT];
                uint32_t pc = 0;
#pragma unroll
                for (int k = 0; k < WT; k++) {
                    t[k] = S[k] & E[x * W + k];  // past the row's words S is 0
                    pc += (uint32_t)__popcll(t[k]);
                }
                if (pc >= (uint32_t)(L - l)) {  // enough for x_l..x_{L-1}
#pragma unroll
                    for (int k = 0; k < WT; k++) {
                        stk[((l - 3) * WT + k) * kBlock] = S[k];
                        S[k] = t[k];
                    }
                    ++l;
                    if (EMIT) {
                        sX[(l - 2) * kBlock + tid] = (uint16_t)x;
                        if (l == L - 1) {
                            hpre = hash_step(hash_seed(L), 0, u);
                            for (int q = 1; q < L - 2; q++) hpre = hash_step(hpre, q, A[xget(q)]);
                        }
                    }
                }
            }
        }
        const uint32_t alive = (uint32_t)__popcll(__ballot(live));
        if (alive == 0) break;
        if ((++rounds & 255u) == 0u && past(dl)) {
            mark_stop(out);
            break;
        }
        // ---- last level: add |S n E[x]| for every x in S
        for (;;) {
            const bool on = any();
            if (2u * (uint32_t)__popcll(__ballot(on)) < alive + 1u) break;
            if (on) {
                const uint32_t x = take();
                const uint64_t *Ex = E + x * W;
                const bool end = L == 4 && --left == 0;  // the item's last x_2
                uint32_t pc = 0;
#pragma unroll
                for (int k = 0; k < WT; k++) {
                    const uint64_t t = S[k] & Ex[k];
                    pc += (uint32_t)__popcll(t);
                    if (EMIT && t) {
                        if (out.buf) sX[(L - 2) * kBlock + tid] = (uint16_t)x;
                        emit_bits(out, L - 1, u, A, hash_step(hpre, L - 2, A[x]), t, (uint32_t)k, xget, hs, hx);
                    }
                }
                cnt += pc;
                if (end) {
#pragma unroll
                    for (int k = 0; k < WT; k++) S[k] = 0ull;
                }
            }
        }
    }
}

// DFS over the items of a batch, P lanes an item: lane i of the group owns word
// i of every set, the next candidate is one ballot over the group's words, and
// the sets of the levels above are kept in the thread's LDS stack.
template <int P>
__device__ void group_walk(const KPlan &pl, const LdsView &v, uint32_t sumd, uint32_t items, Share sh,
                           const KOut &out, uint64_t dl, uint64_t &cnt, uint64_t &hs, uint64_t &hx)
{
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int lx = lane & (P - 1);
    const int pbase = lane & ~(P - 1);
    const int L = pl.L;
    uint64_t *sStk = v.sStk;
    uint32_t *sMisc = v.sMisc;
    uint16_t *sX = v.sX;
    auto xget = [&](int q) -> uint32_t { return sX[q * kBlock + tid]; };
    uint32_t spins = 0;
    for (;;) {
        uint32_t item = 0;
        if (lx == 0) {
            if (past(dl)) {
                item = 0xffffffffu;
                mark_stop(out);
            } else {
                item = atomicAdd(&sMisc[M_NEXT], 1u) * sh.parts + sh.part;
            }
        }
        item = __shfl(item, 0, P);
        if (item >= items) break;
        const bool whole = whole_rows(pl);
        const uint32_t row = whole ? item : find_row(v.sPre, sumd, item);
        const RootRec rr = v.sRoot[v.sJRoot[row]];
        const uint32_t jl = row - rr.doff;
        if (whole && ((pl.skip_split && jl < rr.split) || rr.d + 1u < (uint32_t)L)) continue;
        const uint32_t skip = whole ? 0u : (item - v.sPre[row]) * pl.chunk;
        const uint32_t d = rr.d, W = (d + 63) >> 6;
        const uint64_t *E = v.sE + rr.eoff;
        const uint32_t *A = v.sA + rr.doff;
        const uint32_t w = (uint32_t)lx;
        const bool own = w < W;
        sX[1 * kBlock + tid] = (uint16_t)jl;

        // C_l from the set of its base level (KPlan::lev)
        auto level_word = [&](int l) -> uint64_t {
            const uint32_t a = sMisc[M_LEV + l], b = sMisc[M_LEV + kMaxLevels + l];
            uint64_t t = b >> 16 ? sStk[((b >> 16) - 2) * kBlock + tid] : valid_mask(w, d);
            uint32_t m = b & 0xffffu;
            while (m) {
                const int s = __builtin_ctz(m);
                m &= m - 1;
                t &= ~bit_at(xget(s), w);
            }
            m = a >> 16;
            while (m) {
                const int s = __builtin_ctz(m);
                m &= m - 1;
                t &= gt_mask(xget(s), w);
            }
            m = a & 0xffffu;
            while (m && t) {  // no row reads once the word is empty
                const int q = __builtin_ctz(m);
                m &= m - 1;
                t &= E[xget(q) * W + w];
            }
            return t;
        };

        // Summed last level (pl.tail): F = the part of C_{L-1} fixed by
        // x_1..x_{L-3}; for x_{L-2} = x, |C_{L-1}| = |F n (x, inf)| when
        // L-2 is in smask[L-1], else |F \ {x}|.  Summed over x in S = C_{L-2}:
        //   sum_w [ |S_w| (|F| - |F_{<=w}|) + pairs_w(S, F) ]  or  |S||F| - |S n F|
        // with one group prefix sum of |F_w|.
        auto tail_sum = [&](int l) -> uint64_t {
            const uint64_t S = own ? sStk[(l - 3) * kBlock + tid] : 0ull;
            const uint64_t F = own ? level_word(l) : 0ull;
            const uint32_t sc = (uint32_t)__popcll(S);
            uint32_t fin = (uint32_t)__popcll(F);
            for (int o = 1; o < P; o <<= 1) {
                const uint32_t y = __shfl_up(fin, o, P);
                if (lx >= o) fin += y;
            }
            const uint32_t ftot = __shfl(fin, P - 1, P);
            if (pl.leaf_gt) return (uint64_t)sc * (ftot - fin) + pairs_in_word(S, F);
            return (uint64_t)sc * ftot - (uint64_t)__popcll(S & F);
        };

        // Paired last levels (pl.pair), l = L-2 = b: S = C_{l-1} = C_a with
        // x_1..x_{a-1} fixed; adds C(|S n E[x_b]|, 2) over x_b in B, the
        // candidates of level b without its constraints on x_a.  Only an x_b
        // adjacent to some member of S can add anything, so B is first cut to
        // the union of their rows.
        auto pair_sum = [&](int l) -> uint64_t {
            const uint64_t S = own ? sStk[(l - 3) * kBlock + tid] : 0ull;
            uint64_t U = 0;
            for (uint64_t rem = S;;) {
                const uint64_t bal = __ballot(rem != 0ull);
                const uint64_t mine = (P == 64) ? bal : ((bal >> pbase) & ((1ull << P) - 1ull));
                if (mine == 0ull) break;
                const int f = __builtin_ctzll(mine);
                const uint64_t vf = __shfl(rem, f, P);
                const uint32_t xs = ((uint32_t)f << 6) + (uint32_t)__builtin_ctzll(vf);
                if (lx == f) rem &= rem - 1ull;
                if (own) U |= E[xs * W + w];
            }
            uint64_t B = 0;
            if (own) {
                B = valid_mask(w, d) & U;
                uint32_t qm = pl.qmask[l] & ~(1u << (l - 1));
                while (qm) {
                    const int q = __builtin_ctz(qm);
                    qm &= qm - 1;
                    B &= E[xget(q) * W + w];
                }
                for (int s = 1; s < l - 1; s++) B &= ~bit_at(xget(s), w);
                uint32_t sm = pl.smask[l];
                while (sm) {
                    const int s = __builtin_ctz(sm);
                    sm &= sm - 1;
                    B &= gt_mask(xget(s), w);
                }
            }
            uint64_t sum = 0;
            for (;;) {
                const uint64_t bal = __ballot(B != 0ull);
                const uint64_t mine = (P == 64) ? bal : ((bal >> pbase) & ((1ull << P) - 1ull));
                if (mine == 0ull) break;
                const int f = __builtin_ctzll(mine);
                const uint64_t vf = __shfl(B, f, P);
                const uint32_t xb = ((uint32_t)f << 6) + (uint32_t)__builtin_ctzll(vf);
                if (lx == f) B &= B - 1ull;  // lane f's lowest bit is x_b
                uint32_t pc = own ? (uint32_t)__popcll(S & E[xb * W + w]) : 0u;
                for (int o = 1; o < P; o <<= 1) pc += __shfl_xor(pc, o, P);
                if (lx == 0) sum += (uint64_t)pc * (pc - 1u) / 2u;
            }
            return sum;
        };

        const uint64_t t2 = own ? level_word(2) : 0ull;
        if (L == 3) {
            cnt += (uint64_t)__popcll(t2);
            if (pl.emit && t2) emit_word(out, pl, 2, rr.u, A, t2, w, xget, hs, hx);
            continue;
        }
        sStk[tid] = t2;
        // the item's x_2: the candidates of rank [skip, skip + chunk) in C_2
        uint64_t x2s = t2;
        if (pl.chunk != kNoSplit) {
            const uint32_t pc = (uint32_t)__popcll(t2);
            uint32_t before = pc;
            for (int o = 1; o < P; o <<= 1) {
                const uint32_t y = __shfl_up(before, o, P);
                if (lx >= o) before += y;
            }
            before -= pc;
            uint32_t drop = skip > before ? skip - before : 0u;
            uint32_t end = skip + pl.chunk > before ? skip + pl.chunk - before : 0u;
            if (drop > pc) drop = pc;
            if (end > pc) end = pc;
            x2s = end > drop ? low_bits(t2, end) & ~low_bits(t2, drop) : 0ull;
        }
        int l = 3;
        uint32_t pos = 0;
        uint64_t F = 0, hpre = 0;  // last level: what x_{L-2} does not change
        for (;;) {
            if (++spins == kClockEvery) {
                spins = 0;
                if (past(dl)) break;  // the next claim records the stop
            }
            if (pl.tail && l == L - 1) {  // every x_{L-2} of C_{L-2} at once
                cnt += tail_sum(l);
                if (l == 3) break;
                --l;
                pos = (uint32_t)xget(l - 1) + 1u;
                continue;
            }
            if (pl.pair && l == L - 2) {  // levels L-3..L-1 at once
                cnt += pair_sum(l);
                if (l == 3) break;
                --l;
                pos = (uint32_t)xget(l - 1) + 1u;
                continue;
            }
            if (l == L - 1 && pos == 0u) {
                F = own ? level_word(l) : 0ull;
                if (pl.emit) {
                    hpre = hash_step(hash_seed(L), 0, rr.u);
                    for (int q = 1; q < l - 1; q++) hpre = hash_step(hpre, q, A[xget(q)]);
                }
            }
            uint64_t vv = l == 3 ? x2s : own ? sStk[(l - 3) * kBlock + tid] : 0ull;
            const uint32_t pw = pos >> 6;
            if (w < pw) vv = 0ull;
            else if (w == pw) vv &= (~0ull << (pos & 63u));
            const uint64_t bal = __ballot(vv != 0ull);
            const uint64_t mine = (P == 64) ? bal : ((bal >> pbase) & ((1ull << P) - 1ull));
            if (mine == 0ull) {
                if (l == 3) break;
                --l;
                pos = (uint32_t)xget(l - 1) + 1u;
                continue;
            }
            const int f = __builtin_ctzll(mine);
            const uint64_t vf = __shfl(vv, f, P);
            const uint32_t xi = ((uint32_t)f << 6) + (uint32_t)__builtin_ctzll(vf);
            sX[(l - 1) * kBlock + tid] = (uint16_t)xi;
            if (l == L - 1) {
                uint64_t t = F;
                if (pl.leaf_row && t) t &= E[xi * W + w];
                if (pl.leaf_gt) t &= gt_mask(xi, w);
                if (pl.leaf_x) t &= ~bit_at(xi, w);
                cnt += (uint64_t)__popcll(t);
                if (pl.emit && t)
                    emit_bits(out, l, rr.u, A, hash_step(hpre, l - 1, A[xi]), t, w, xget, hs, hx);
                pos = xi + 1u;
            } else {
                const uint64_t t = own ? level_word(l) : 0ull;
                sStk[(l - 2) * kBlock + tid] = t;
                ++l;
                pos = 0;
            }
        }
    }
}

// Hash of a vertex for the LDS tables: the top bits of a 24-bit product (a
// full-rate multiply; the 32-bit one runs at a quarter of the rate).
__device__ __forceinline__ uint32_t lds_hash(uint32_t v) { return __umul24(v, 0x9E3779u); }

// Table of 2^lh slots (key + 1, value) with a filter of 16 bits per slot.  Linear
// probing from an even slot, so that a probe reads two slots at once: at most
// half of the slots are taken, and 64 lanes' longest chain is then about two
// reads instead of seven.
__device__ __forceinline__ void table_add(uint32_t *key, uint16_t *val, uint32_t *flt, uint32_t lh, uint32_t vx,
                                          uint32_t value)
{
    const uint32_t h = lds_hash(vx), mask = (1u << lh) - 1u;
    uint32_t s = (h >> (32u - lh)) & ~1u;
    while (atomicCAS(&key[s], 0u, vx + 1u) != 0u) s = (s + 1) & mask;
    val[s] = (uint16_t)value;
    const uint32_t fb = h >> (28u - lh);
    atomicOr(&flt[fb >> 5], 1u << (fb & 31u));
}

__device__ __forceinline__ bool table_find(const uint32_t *key, const uint16_t *val, uint32_t lh, uint32_t vx,
                                           uint32_t &value)
{
    const uint32_t mask = (1u << lh) - 1u, want = vx + 1u;
    uint32_t s = (lds_hash(vx) >> (32u - lh)) & ~1u;
    uint32_t k0, k1;
    for (;;) {  // one exit: two of them cost the wave a third of the search's time
        const uint64_t kk = *(const uint64_t *)&key[s];
        k0 = (uint32_t)kk;
        k1 = (uint32_t)(kk >> 32);
        if (k0 == want || k1 == want || k0 == 0u || k1 == 0u) break;
        s = (s + 2u) & mask;
    }
    const bool hit = k0 == want || k1 == want;
    if (hit) value = val[s + (k0 == want ? 0u : 1u)];
    return hit;
}

// Whether w is in v's larger-key range, by the range's table past w's first slot.
__device__ __forceinline__ bool later_slot(const KGraph &g, uint32_t v, uint32_t w)
{
    const VInfo vi = g.vinfo[v];
    const uint32_t size = 2 * vi.hlen;
    const uint32_t *t = g.htab + 2 * vi.hbeg;
    uint32_t s = lookup_slot(w, size);
    bool hit;
    for (;;) {
        s = s + 1 == size ? 0 : s + 1;
        const uint32_t x = t[s];
        hit = x == w + 1u;
        if (hit || x == 0u) break;
    }
    return hit;
}

// LDS of the pair search: row contexts, row-start marks, the waves' queues, the
// filters and the vertices that looked-up units name.
struct UnitView {
    RowCtx *ctx;
    uint64_t *mark, *q;
    const uint32_t *flt, *A, *key;
};

// Finds adjacent pairs (v, w), key(v) < key(w), from v, for up to N * kBlock
// rows (thread t has rows t, t + kBlock, ...; un[q] units and context cx[q]
// each, base and aoff relative to the row's first unit).  A row's work units
// are the entries of v's larger-key range, each tested against a table of
// wanted vertices, or, where that range is longer than kLookupRatio times the
// vertices it can pair with, those vertices, each looked up in the range's
// table.  settle(lo, info) is called for units that are probably a pair, 64 a
// wave at a time: info is the row's, lo the entry, or for looked-up units the
// index of the wanted vertex with bit 31 set when its first slot held it.
//
// What bounds it is instruction issue (a wave64 VALU instruction takes a SIMD
// four cycles), so a unit costs as little as possible:
//  * all rows' units are numbered through and a wave takes 64 consecutive ones,
//    one a lane.  A unit's row is the number of row starts at or before it,
//    one 64-bit mark word and one count per 64 units and a mask-and-count per
//    lane; the row's context is one 16-byte LDS read;
//  * a streamed entry is first tested against a filter of 16 to 32 bits per
//    wanted vertex.  The few per cent that pass (and the looked-up slots that
//    are taken) go to a queue per wave, so the exact probe and what a pair does
//    run with full waves;
//  * four loads a lane are in flight.
// Before, each thread took 8 consecutive units and reloaded the row's context
// wherever one of 64 lanes crossed into another row, and every lane waited for
// the longest probe: 216 lane instructions per unit (4-clique on 1.1M vertices,
// 362 us; now 257 us).
//  * where a pair only counts (`count`), those that a first slot settles -- most
//    -- are counted on the spot and never queued.
template <int N, class Settle>
__device__ __forceinline__ void find_pairs(const KGraph &g, const UnitView &u, const uint32_t (&un)[N],
                                           RowCtx (&cx)[N], uint32_t rows, bool count, uint64_t &cnt, Settle &&settle)
{
    uint32_t counted = 0;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    uint32_t at[N];
    uint64_t act[N];
#pragma unroll
    for (int r = 0; r < N; r++) {
        at[r] = 0;
        act[r] = 0;
        if ((uint32_t)r * kBlock >= rows) continue;
        at[r] = wave_incl_scan(un[r]);
        act[r] = __ballot(un[r] != 0);
        if (lane == 63)
            u.mark[16 + r * (kBlock / 64) + wv] = (uint64_t)at[r] | (uint64_t)__popcll(act[r]) << 32;
    }
    __syncthreads();
    uint32_t total = 0, nrows = 0;  // units; rows that have any
#pragma unroll
    for (int r = 0; r < N; r++) {
        if ((uint32_t)r * kBlock >= rows) continue;
        uint32_t ub = total, rb = nrows;
        for (int w = 0; w < kBlock / 64; w++) {
            const uint64_t t = u.mark[16 + r * (kBlock / 64) + w];
            if (w < wv) {
                ub += (uint32_t)t;
                rb += (uint32_t)(t >> 32);
            }
            total += (uint32_t)t;
            nrows += (uint32_t)(t >> 32);
        }
        at[r] = ub + at[r] - un[r];  // the row's first unit
        if (un[r]) {
            cx[r].aoff -= at[r];
            if (!((cx[r].info >> 9) & 1u)) cx[r].base -= at[r];
            u.ctx[rb + bits_below(act[r])] = cx[r];
        }
    }
    uint64_t *q = u.q + wv * kQueue;
    auto flush = [&](uint32_t from, uint32_t n) {
        wave_lds_sync();
        if ((uint32_t)lane < n) settle((uint32_t)q[from + lane], (uint32_t)(q[from + lane] >> 32));
        wave_lds_sync();
    };
    constexpr int kUnroll = 4;
    uint32_t k_done = 0, qn = 0;  // rows started before the tile; queued units
    for (uint32_t t0 = 0; t0 < total; t0 += kTile) {
        __syncthreads();
        if (tid < (int)(kTile / 64)) u.mark[tid] = 0;
        __syncthreads();
#pragma unroll
        for (int r = 0; r < N; r++) {
            const uint32_t o = at[r] - t0;
            if (un[r] && o < kTile) atomicOr((unsigned long long *)&u.mark[o >> 6], 1ull << (o & 63u));
        }
        __syncthreads();
        const uint64_t mw = u.mark[lane];
        const uint32_t pc = (uint32_t)__popcll(mw), ic = wave_incl_scan(pc);
        const uint32_t k0 = k_done + ic - pc;
        k_done += lane_u32(ic, 63);
        const uint32_t nseg = total - t0 < kTile ? (total - t0 + 63u) >> 6 : kTile / 64;
        for (uint32_t s0 = wv; s0 < nseg; s0 += kUnroll * (kBlock / 64)) {
            uint32_t val[kUnroll], aux[kUnroll], info[kUnroll];
#pragma unroll
            for (int i = 0; i < kUnroll; i++) {
                const uint32_t s = s0 + i * (kBlock / 64);
                val[i] = aux[i] = info[i] = 0;
                if (s >= nseg) continue;
                const uint32_t m0 = lane_u32((uint32_t)mw, s), m1 = lane_u32((uint32_t)(mw >> 32), s);
                const uint64_t m = (uint64_t)m1 << 32 | m0;
                const uint32_t k = lane_u32(k0, s) + (m0 & 1u) - 1u + bits_below(m >> 1);
                const uint32_t e = t0 + s * 64 + lane;
                if (e >= total) continue;
                const RowCtx c = u.ctx[k];
                info[i] = c.info;
                if ((c.info >> 9) & 1u) {
                    const uint64_t hb = c.base & ((1ull << kRangeShift) - 1ull);
                    aux[i] = c.aoff + e;
                    val[i] = g.htab[2 * hb + lookup_slot(u.A[aux[i]], 2u * (uint32_t)(c.base >> kRangeShift))];
                } else {
                    val[i] = g.ocol[c.base + e];
                }
            }
#pragma unroll
            for (int i = 0; i < kUnroll; i++) {
                const uint32_t s = s0 + i * (kBlock / 64);
                if (s >= nseg) break;
                const uint32_t e = t0 + s * 64 + lane;
                bool on = false;
                uint32_t lo = val[i];
                if (e < total) {
                    if ((info[i] >> 9) & 1u) {
                        on = val[i] != 0u;
                        lo = aux[i] | (val[i] == u.A[aux[i]] + 1u ? 1u << 31 : 0u);
                    } else {
                        const uint32_t fb = lds_hash(val[i]) >> (32u - ((info[i] >> 20) & 31u));
                        on = (u.flt[((info[i] >> 10) & 1023u) + (fb >> 5)] >> (fb & 31u)) & 1u;
                    }
                }
                if (count && on) {
                    const uint32_t lh = ((info[i] >> 20) & 31u) - 4u;
                    const uint32_t slot = 2u * ((info[i] >> 10) & 1023u) + ((lds_hash(val[i]) >> (32u - lh)) & ~1u);
                    const uint64_t kk = *(const uint64_t *)&u.key[slot];
                    const bool sure = (info[i] >> 9) & 1u ? (lo >> 31) != 0u
                                                          : (uint32_t)kk == val[i] + 1u || (uint32_t)(kk >> 32) == val[i] + 1u;
                    counted += sure ? 1u : 0u;
                    on = !sure;
                }
                const uint64_t m = __ballot(on);
                if (on) q[qn + bits_below(m)] = (uint64_t)info[i] << 32 | lo;
                qn += (uint32_t)__popcll(m);
                if (qn >= 64u) {
                    qn -= 64u;
                    flush(qn, 64u);
                }
            }
        }
    }
    if (qn) flush(0, qn);
    cnt += counted;
    __syncthreads();
}

// Stages a batch -- its roots, row vertices and each row's root -- and builds
// the roots' bitmaps (or counts their pairs, KPlan::hits).  Returns the number
// of rows.
template <bool MAY_COUNT>
__device__ uint32_t build_batch(const KGraph &g, const KPlan &pl, const LdsView &v, const RootRec *__restrict__ recs,
                                uint32_t first, uint32_t nr, uint64_t &cnt)
{
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const bool rows = pl.reads_rows != 0;
    if (tid < (int)(LdsBudget::kMaxSumDeg / 64)) v.sMark[tid] = 0;
    if (tid == 0) v.sMisc[M_NEXT] = 0;
    RootRec mine{};
    if (tid < (int)nr) {
        mine = recs[first + tid];
        v.sRoot[tid] = mine;
    }
    __syncthreads();
    if (tid < (int)nr) atomicOr((unsigned long long *)&v.sMark[mine.doff >> 6], 1ull << (mine.doff & 63u));
    const RootRec last = v.sRoot[nr - 1];
    const uint32_t sumd = last.doff + last.d;
    if (rows) {
        const uint32_t ew = pl.hits ? 0u : last.eoff + last.d * ((last.d + 63) >> 6);
        const uint32_t hsl = last.hoff + lds_hash_slots(last.d);
        for (uint32_t i = tid; i < ew; i += kBlock) v.sE[i] = 0;
        for (uint32_t i = tid; i < hsl; i += kBlock) v.sHKey[i] = 0;
        for (uint32_t i = tid; i < hsl / 2; i += kBlock) v.sFlt[i] = 0;
    }
    __syncthreads();
    // A thread holds at most kRowsPer rows; their row entries, then their
    // vertex records, are loaded together.  A row's root is the number of
    // roots that start at or before it.
    constexpr int kRowsPer = (int)(LdsBudget::kMaxSumDeg / kBlock);
    static_assert(LdsBudget::kMaxSumDeg % kBlock == 0, "rows per thread");
    uint32_t rvx[kRowsPer], rro[kRowsPer];
#pragma unroll
    for (int q = 0; q < kRowsPer; q++) {
        const uint32_t j = (uint32_t)tid + (uint32_t)q * kBlock;
        rvx[q] = 0;
        rro[q] = 0;
        if ((uint32_t)q * kBlock >= sumd) continue;
        const int wj = q * (kBlock / 64) + wv;
        uint32_t before = 0;
        for (int w = 0; w < wj; w++) before += (uint32_t)__popcll(v.sMark[w]);
        const uint64_t m = v.sMark[wj];
        if (j < sumd) {
            const uint32_t r = before + bits_below(m) + (uint32_t)((m >> lane) & 1u) - 1u;
            rro[q] = r;
            rvx[q] = g.ocol[v.sRoot[r].rbeg + (j - v.sRoot[r].doff)];
            v.sA[j] = rvx[q];
            v.sJRoot[j] = (uint8_t)r;
        }
    }
    if (!rows) {
        __syncthreads();
        return sumd;
    }
    VInfo rvi[kRowsPer];
#pragma unroll
    for (int q = 0; q < kRowsPer; q++)
        if ((uint32_t)tid + (uint32_t)q * kBlock < sumd) rvi[q] = g.vinfo[rvx[q]];
    uint32_t un[kRowsPer];
    RowCtx cx[kRowsPer];
#pragma unroll
    for (int q = 0; q < kRowsPer; q++) {
        const uint32_t j = (uint32_t)tid + (uint32_t)q * kBlock;
        un[q] = 0;
        if (j < sumd) {
            const RootRec rr = v.sRoot[rro[q]];
            const uint32_t jl = j - rr.doff, vx = rvx[q], lh = lds_hash_log2(rr.d);
            // only kept entries are looked for
            if (!pl.kept || jl >= rr.split) table_add(v.sHKey + rr.hoff, v.sHVal + rr.hoff, v.sFlt + (rr.hoff >> 1), lh, vx, jl);
            // x_1..x_{L-1} are distinct row entries: shorter rows hold no tuple
            const uint32_t c = rr.d + 1u < (uint32_t)pl.L
                                   ? 0u : pair_partners(jl, rr.d, rr.split, g.asc, pl.kept, pl.upper);
            const VInfo vi = rvi[q];
            if (c) {
                const bool look = (uint64_t)vi.hlen > (uint64_t)c * pl.bin_ratio;
                un[q] = look ? c : vi.hlen;
                cx[q].base = look ? vi.hbeg | ((uint64_t)vi.hlen << kRangeShift) : vi.hbeg;
                cx[q].aoff = rr.doff + (g.asc ? rr.d - c : 0u);  // first partner
                cx[q].info = j | (look ? 1u << 9 : 0u) | (rr.hoff >> 1) << 10 | (lh + 4u) << 20;
            }
        }
    }
    const UnitView uv{v.sCtx, v.sMark, v.sQ, v.sFlt, v.sA, v.sHKey};
    find_pairs(g, uv, un, cx, sumd, MAY_COUNT && pl.hits && pl.closed == kClosedC, cnt, [&](uint32_t lo, uint32_t info) {
        const uint32_t j = info & 511u;
        const RootRec rr = v.sRoot[v.sJRoot[j]];
        const uint32_t jl = j - rr.doff;
        uint32_t i = 0;
        bool hit;
        if ((info >> 9) & 1u) {
            const uint32_t p = lo & 0x7fffffffu;
            i = p - rr.doff;
            hit = (lo >> 31) || later_slot(g, v.sA[j], v.sA[p]);
        } else {
            hit = table_find(v.sHKey + rr.hoff, v.sHVal + rr.hoff, ((info >> 20) & 31u) - 4u, lo, i);
        }
        if (hit) {
            if (MAY_COUNT && pl.hits) cnt += pl.closed == kClosedRow ? rr.d - 2u : 1u;
            else set_pair(v.sE + rr.eoff, (rr.d + 63) >> 6, jl, i, pl.upper);
        }
    });
    return sumd;
}

// Processes one LDS batch: build, then the DFS over its items (lds_items).  The
// plan's level records are in sMisc[M_LEV..].  WALK fixes the walk at compile
// time where the launch serves one plan (the walks need different registers);
// kWalkAny picks it per plan.
enum { kWalkAny = 0, kWalkGroup = 1, kWalkLane = 2, kWalkLaneEmit = 3, kWalkNone = 4 };
template <int PC, int WALK>
__device__ void process_batch(const KGraph &g, const KPlan &pl, const LdsView &v,
                              const RootRec *__restrict__ recs, uint32_t first, uint32_t nr, Share sh,
                              const KOut &out, uint64_t dl, uint64_t &cnt, uint64_t &hs, uint64_t &hx)
{
    const int tid = threadIdx.x;
    const uint64_t t_build = wall_clock64();
    constexpr bool kMayCount = WALK == kWalkAny || WALK == kWalkNone;
    const uint32_t sumd = build_batch<kMayCount>(g, pl, v, recs, first, nr, cnt);
    if (tid == 0) prof_add(out, 3, blockIdx.x, t_build);  // staging + bitmap build

    if (pl.hits) return;  // the pairs found are the count
    const uint32_t items = lds_items(pl, v, sumd, cnt);
    if (WALK == kWalkNone || items == 0) {
        __syncthreads();  // the next batch reuses the LDS arrays
        return;
    }
    constexpr int WT = PC <= 8 ? PC : 1, kLg = WT == 8 ? 3 : WT >> 1;
    const int walk = WALK != kWalkAny ? WALK
                     : PC <= 8 && lds_lane_walk(pl, kLg) ? (pl.emit ? kWalkLaneEmit : kWalkLane) : kWalkGroup;
    if (PC <= 8 && walk == kWalkLane) clique_walk<WT, false>(pl, v, sumd, items, sh, out, dl, cnt, hs, hx);
    else if (PC <= 8 && walk == kWalkLaneEmit) clique_walk<WT, true>(pl, v, sumd, items, sh, out, dl, cnt, hs, hx);
    else group_walk<PC>(pl, v, sumd, items, sh, out, dl, cnt, hs, hx);
    __syncthreads();
}

// A class of few batches leaves CUs idle while its workgroups walk deep plans
// (W5's hashed matches on 20,000 vertices: 16 batches of the widest class, 3.2
// of 3.4 ms).  Each of its batches is then taken by `parts` workgroups, which
// all build it and walk every parts-th item.
// MinWaves > 1: the compiler keeps the registers to that many waves per SIMD
// (7 workgroups per CU instead of 5 for the narrow classes, at the cost of a
// few bytes of spill); used when no hub kernels of the query share the CUs.
template <int P, int MinWaves, int WALK>
__global__ __launch_bounds__(kBlock, MinWaves) void lds_batch_kernel(KGraph g, KPlan pl,
                                                           const RootRec *__restrict__ recs,
                                                           const uint32_t *__restrict__ batch_first,
                                                           const uint32_t *__restrict__ batch_count,
                                                           uint32_t b0, uint32_t b1, uint32_t parts,
                                                           unsigned long long *cursor, LdsLayout lay,
                                                           KOut out)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const LdsView v = lds_view(smem, lay);
    const int tid = threadIdx.x;
    if (tid < 2 * kMaxLevels) v.sMisc[M_LEV + tid] = pl.lev[tid];
    uint64_t cnt = 0, hs = 0, hx = 0;
    const uint64_t dl = out.dl[1];
    const uint64_t t_start = wall_clock64();
    constexpr int kLg = P == 64 ? 6 : P == 32 ? 5 : P == 16 ? 4 : P == 8 ? 3 : P >> 1;
    if (out.stamp && blockIdx.x == 0 && tid == 0) out.stamp[kStampStart + kLg] = t_start;
    uint32_t seen = 0;  // thread 0's claim state
    for (;;) {
        if (tid == 0) {
            uint64_t bb = 0, be = 0;
            if (past(dl)) {
                v.sMisc[M_BATCH] = ~0u;
                mark_stop(out);
            } else if (claim_striped(cursor, (uint64_t)(b1 - b0) * parts, blockIdx.x % kStripes, seen, 1, bb, be)) {
                v.sMisc[M_BATCH] = (uint32_t)bb;
            } else {
                v.sMisc[M_BATCH] = ~0u;
            }
        }
        __syncthreads();
        const uint32_t t = v.sMisc[M_BATCH];
        if (t == ~0u) break;
        const uint32_t b = b0 + t / parts;
        process_batch<P, WALK>(g, pl, v, recs, batch_first[b], batch_count[b], Share{t % parts, parts}, out, dl, cnt, hs,
                               hx);
    }
    flush_acc(out, cnt, hs, hx);
    if (tid == 0) {
        prof_add(out, 0, blockIdx.x, t_start);
        stamp_end(out, kStampEnd + kLg);
    }
}

// One persistent launch over the LDS batches of several prepared queries.
// Work records are ordered heaviest first; a workgroup takes the next record,
// loads that query's plan and graph and runs the batch, then flushes its counts
// to that query's counters.  One launch per lane class (P lanes an item).
template <int P>
__global__ __launch_bounds__(kBlock) void lds_multi_kernel(const MultiQuery *__restrict__ qs,
                                                           const MultiWork *__restrict__ work,
                                                           uint32_t nwork, unsigned long long *cursor,
                                                           LdsLayout lay)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const LdsView v = lds_view(smem, lay);
    const int tid = threadIdx.x;
    uint32_t parts = 0;  // thread 0's claim state
    for (;;) {
        if (tid == 0) {
            uint64_t bb = 0, be = 0;
            v.sMisc[M_BATCH] = claim_striped(cursor, nwork, blockIdx.x % kStripes, parts, 1, bb, be)
                                   ? (uint32_t)bb : nwork;
        }
        __syncthreads();
        const uint32_t wi = (uint32_t)__builtin_amdgcn_readfirstlane((int)v.sMisc[M_BATCH]);
        if (wi >= nwork) break;
        const MultiWork w = work[wi];
        const MultiQuery &q = qs[w.query];
        const KPlan &pl = q.pl;
        if (tid < 2 * kMaxLevels) v.sMisc[M_LEV + tid] = pl.lev[tid];
        __syncthreads();
        uint64_t cnt = 0, hs = 0, hx = 0;
        const uint64_t dl = q.out.dl[1];
        const uint64_t t_start = wall_clock64();
        process_batch<P, kWalkAny>(q.g, pl, v, q.recs, q.batch_first[w.batch], q.batch_count[w.batch], Share{0, 1}, q.out,
                                   dl, cnt, hs, hx);
        flush_acc(q.out, cnt, hs, hx);
        if (tid == 0) prof_add(q.out, 0, blockIdx.x, t_start);
    }
}

// ------------------------------------------------------------------- hubs

// Hash of every hub row: vertex -> row index (linear probing, 0 = empty).
__global__ __launch_bounds__(kBlock) void hub_hash_kernel(KGraph g, const HubRec *__restrict__ hubs,
                                                          const uint32_t *__restrict__ hub_of_row,
                                                          uint64_t g0, uint64_t g1, uint64_t *kv,
                                                          const unsigned long long *dl)
{
    if (past(*dl)) return;  // the encode and the DFS that follow stop at once
    for (uint64_t r = g0 + blockIdx.x * (uint64_t)kBlock + threadIdx.x; r < g1;
         r += (uint64_t)gridDim.x * kBlock) {
        const HubRec h = hubs[hub_of_row[r]];
        const uint32_t jl = (uint32_t)(r - h.joff);
        if (jl < h.rlo) continue;  // rows below rlo are never found by a scan range
        const uint32_t v = g.ocol[h.rbeg + jl];
        uint32_t s = hash_slot(v, h.hslots);
        for (;;) {
            // slot = key (low word) | row index (high word): a hit costs one load
            uint32_t *slot = (uint32_t *)&kv[h.hoff + s];
            if (atomicCAS(&slot[0], 0u, v + 1u) == 0u) {
                slot[1] = jl;
                break;
            }
            s = (s + 1) & (h.hslots - 1);
        }
    }
}

// Hub bitmaps: waves take chunks of 64 rows (of the round's rows whose scan
// range is not empty, listed on the host), scan the lengths of their scan
// ranges (the larger-key range of the row vertex, cut on the host to the part
// that can hold kept columns) and stream the concatenation lane-parallel.  A
// chunk takes every nchunks-th row, so the long ranges of one hub's rows
// spread over many waves.
// Each lane loads its kChunk entries back to back before probing the hash.
__global__ __launch_bounds__(kBlock) void hub_encode_kernel(KGraph g, const HubRec *__restrict__ hubs,
                                                            const uint32_t *__restrict__ hub_of_row,
                                                            const uint64_t *__restrict__ hub_range,
                                                            const uint64_t *__restrict__ rows, uint64_t nrows,
                                                            const uint64_t *__restrict__ kv,
                                                            uint64_t *E, int upper, int count, KOut out)
{
    __shared__ uint64_t sBeg[kBlock];
    __shared__ uint32_t sPre[kBlock];
    __shared__ uint32_t sHub[kBlock];
    __shared__ uint32_t sJl[kBlock];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const uint64_t nchunks = (nrows + 63) / 64;
    const uint64_t wstride = (uint64_t)gridDim.x * (kBlock / 64);
    const uint64_t dl = *out.dl;
    const uint64_t t_start = wall_clock64();
    uint64_t cnt = 0;  // count: KPlan::closed of a plan whose pairs are counted, no bitmap (KPlan::hits)
    for (uint64_t c = blockIdx.x * (uint64_t)(kBlock / 64) + wv; c < nchunks; c += wstride) {
        if (past(dl)) {  // the bitmap stays incomplete; the DFS that follows stops at once
            if (lane == 0) mark_stop(out);
            break;
        }
        const uint64_t x = (uint64_t)lane * nchunks + c;  // rows strided over the chunks
        uint32_t len = 0;
        if (x < nrows) {
            const uint64_t r = rows[x];
            const uint32_t hi = hub_of_row[r];
            const uint64_t rg = hub_range[r];
            sBeg[tid] = rg & ((1ull << kRangeShift) - 1ull);
            len = (uint32_t)(rg >> kRangeShift);
            sHub[tid] = hi;
            sJl[tid] = (uint32_t)(r - hubs[hi].joff);
        }
        const uint32_t inc = wave_incl_scan(len);
        sPre[tid] = inc;
        const uint32_t total = __shfl(inc, 63, 64);
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const int wb = wv * 64;
        // every lane takes kChunk consecutive elements: one search for the row
        // of the first, then the rows advance with the elements
        constexpr uint32_t kChunk = 8;
        for (uint32_t e0 = lane * kChunk; e0 < total; e0 += 64 * kChunk) {
            int kfirst = 0;
            {
                int hi = 63;  // smallest k with pre[k] > e0
                while (kfirst < hi) {
                    const int mid = (kfirst + hi) >> 1;
                    if (sPre[wb + mid] > e0) hi = mid; else kfirst = mid + 1;
                }
            }
            int k = 0;
            uint32_t kbeg = 0, kend = 0;  // elements of row k: [kbeg, kend)
            HubRec h;
            uint32_t jl = 0;
            uint64_t W = 0, beg = 0;
            auto load_row = [&]() {
                h = hubs[sHub[wb + k]];
                jl = sJl[wb + k];
                W = (h.d + 63) >> 6;
                beg = sBeg[wb + k];
            };
            auto restart = [&]() {
                k = kfirst;
                kend = sPre[wb + k];
                kbeg = k ? sPre[wb + k - 1] : 0u;
                load_row();
            };
            auto seek = [&](uint32_t e) {
                if (e >= kend) {
                    do {
                        k++;
                        kbeg = kend;
                        kend = sPre[wb + k];
                    } while (e >= kend);
                    load_row();
                }
            };
            const uint32_t e1 = e0 + kChunk < total ? e0 + kChunk : total;
            uint32_t ent[kChunk];
            restart();
#pragma unroll
            for (uint32_t q = 0; q < kChunk; q++) {
                const uint32_t e = e0 + q;
                ent[q] = 0;
                if (e < e1) {
                    seek(e);
                    ent[q] = g.ocol[beg + (e - kbeg)];
                }
            }
            restart();
#pragma unroll
            for (uint32_t q = 0; q < kChunk; q++) {
                const uint32_t e = e0 + q;
                if (e >= e1) break;
                seek(e);
                const uint32_t wv2 = ent[q];
                uint32_t s = hash_slot(wv2, h.hslots);
                uint64_t slot = kv[h.hoff + s];
                for (;;) {
                    const uint32_t key = (uint32_t)slot;
                    if (key == 0u) break;
                    if (key == wv2 + 1u) {
                        const uint32_t i = (uint32_t)(slot >> 32);
                        if (count) {
                            cnt += count == kClosedRow ? h.d - 2u : 1u;
                            break;
                        }
                        // upper plans keep the bit in the row of the smaller index only
                        const bool fwd = !upper || i > jl, mir = !upper || jl > i;
                        if (fwd && jl >= h.rlo)
                            atomicOr((unsigned long long *)&E[h.eoff + (uint64_t)(jl - h.rlo) * W + (i >> 6)],
                                     1ull << (i & 63));
                        if (mir && i >= h.rlo)
                            atomicOr((unsigned long long *)&E[h.eoff + (uint64_t)(i - h.rlo) * W + (jl >> 6)],
                                     1ull << (jl & 63));
                        break;  // a hub row holds each vertex once
                    }
                    s = (s + 1) & (h.hslots - 1);
                    slot = kv[h.hoff + s];
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
    if (count) {
        flush_acc(out, cnt, 0, 0);
        if (lane == 0) prof_add(out, 1, blockIdx.x * (kBlock / 64) + wv, t_start);
    }
    if (tid == 0) stamp_end(out, kStampHub);
}

// Slices of hubs with few kept rows (K <= kSliceKept): a workgroup takes up to
// kSliceRows consecutive row vertices of a hub, holds the kept vertices' table
// in LDS and finds the slice's pairs as the LDS batches do (find_pairs).  Every
// pair has a kept endpoint.
//   CLOSED: the plan's count follows from |C_2| of each kept x_1 (KPlan::closed):
//     the pairs are counted per kept row, in LDS, and added to c2 (one counter
//     per hub item, cleared before) at the end.  No bitmap is built or read.
//   else the kept rows' words of the slice's columns are built in LDS, 256
//     columns at a time, and stored: the slice alone holds them, but for columns
//     of kept rows, whose words also take the bits set from the kept row's own
//     side (atomics, on zeroed words).
// The grid-wide hub_encode_kernel probed a table in HBM and set bits by HBM
// atomics, 64 bytes of write traffic each: diamond on 1.1M vertices 356 us alone
// for 8.5 M entries.  Slices come heaviest first (listed so at upload).
constexpr int kSliceWords = kBlock / 64;
struct SliceLayout {
    uint32_t oCtx, oQ, oMark, oKey, oFlt, oA, oE, oVal, bytes;
};
__host__ inline SliceLayout make_slice_layout(uint32_t kmax, bool closed)
{
    const uint32_t hs = lds_hash_slots(kmax);
    SliceLayout L{};
    uint32_t o = 0;
    L.oE = o;    o += closed ? align_up(kmax * 4, 16) : kmax * kSliceWords * 8;
    L.oCtx = o;  o += kBlock * (uint32_t)sizeof(RowCtx);
    L.oQ = o;    o += (kBlock / 64) * kQueue * 8;
    L.oMark = o; o += kTile / 8;
    L.oKey = o;  o += hs * 4;
    L.oFlt = o;  o += hs / 2 * 4;
    L.oA = o;    o += kmax * 4;
    L.oVal = o;  o += hs * 2;
    L.bytes = align_up(o, 16);
    return L;
}

template <bool CLOSED>
__global__ __launch_bounds__(kBlock) void hub_slice_kernel(KGraph g, const HubRec *__restrict__ hubs,
                                                           const SliceRec *__restrict__ slices,
                                                           const uint64_t *__restrict__ hub_range,
                                                           uint32_t bin_ratio, uint64_t *E, uint32_t *c2, uint64_t i0,
                                                           SliceLayout lay, KOut out)
{
    extern __shared__ __align__(16) unsigned char smem[];
    uint64_t *sE = (uint64_t *)(smem + lay.oE);
    uint32_t *sCnt = (uint32_t *)(smem + lay.oE);
    uint32_t *sKey = (uint32_t *)(smem + lay.oKey), *sFlt = (uint32_t *)(smem + lay.oFlt);
    uint32_t *sA = (uint32_t *)(smem + lay.oA);
    uint16_t *sVal = (uint16_t *)(smem + lay.oVal);
    const UnitView uv{(RowCtx *)(smem + lay.oCtx), (uint64_t *)(smem + lay.oMark), (uint64_t *)(smem + lay.oQ), sFlt,
                      sA, sKey};
    const int tid = threadIdx.x;
    if (past(*out.dl)) {  // what follows stops at once
        if (tid == 0) mark_stop(out);
        return;
    }
    const uint64_t t_start = wall_clock64();
    const SliceRec sl = slices[blockIdx.x];
    const HubRec h = hubs[sl.hub];
    const uint32_t d = h.d, rlo = h.rlo, K = d - rlo, W = (d + 63) >> 6, lh = lds_hash_log2(K);
    for (uint32_t i = tid; i < (1u << lh); i += kBlock) sKey[i] = 0;
    for (uint32_t i = tid; i < (1u << lh) / 2; i += kBlock) sFlt[i] = 0;
    if (CLOSED)
        for (uint32_t i = tid; i < K; i += kBlock) sCnt[i] = 0;
    __syncthreads();
    for (uint32_t i = tid; i < K; i += kBlock) {
        const uint32_t v = g.ocol[h.rbeg + rlo + i];
        sA[i] = v;
        table_add(sKey, sVal, sFlt, lh, v, i);
    }
    for (uint32_t r0 = sl.row0; r0 < sl.row0 + sl.rows; r0 += kBlock) {
        const uint32_t rows = sl.row0 + sl.rows - r0 < (uint32_t)kBlock ? sl.row0 + sl.rows - r0 : (uint32_t)kBlock;
        if (!CLOSED)
            for (uint32_t i = tid; i < K * kSliceWords; i += kBlock) sE[i] = 0;
        uint32_t un[1] = {0};
        RowCtx cx[1];
        if (tid < (int)rows) {
            const uint32_t j = r0 + tid;
            const uint64_t rg = hub_range[h.joff + j];
            const uint32_t len = (uint32_t)(rg >> kRangeShift);
            const uint32_t c = j < rlo ? K : d - 1u - j;  // kept rows it can pair with
            if (len && c) {
                const bool look = (uint64_t)len > (uint64_t)c * bin_ratio;
                un[0] = look ? c : len;
                cx[0].base = rg & ((1ull << kRangeShift) - 1ull);
                if (look) {
                    const VInfo vi = g.vinfo[g.ocol[h.rbeg + j]];
                    cx[0].base = vi.hbeg | ((uint64_t)vi.hlen << kRangeShift);
                }
                cx[0].aoff = K - c;
                cx[0].info = (uint32_t)tid | (look ? 1u << 9 : 0u) | (lh + 4u) << 20;
            }
        }
        __syncthreads();
        uint64_t none = 0;
        find_pairs(g, uv, un, cx, rows, false, none, [&](uint32_t lo, uint32_t info) {
            const uint32_t row = info & 511u, j = r0 + row;
            uint32_t i = 0;
            bool hit;
            if ((info >> 9) & 1u) {
                i = lo & 0x7fffffffu;
                hit = (lo >> 31) || later_slot(g, g.ocol[h.rbeg + j], sA[i]);
            } else {
                hit = table_find(sKey, sVal, lh, lo, i);
            }
            if (!hit) return;
            if (CLOSED) {
                atomicAdd(&sCnt[i], 1u);
                if (j >= rlo) atomicAdd(&sCnt[j - rlo], 1u);
            } else {
                atomicOr((unsigned long long *)&sE[i * kSliceWords + (row >> 6)], 1ull << (row & 63u));
                if (j >= rlo) {
                    const uint32_t ci = i + rlo;
                    atomicOr((unsigned long long *)&E[h.eoff + (uint64_t)(j - rlo) * W + (ci >> 6)], 1ull << (ci & 63u));
                }
            }
        });
        if (!CLOSED) {
            const uint32_t w0 = r0 >> 6, nw = (rows + 63u) >> 6;
            for (uint32_t x = tid; x < K * kSliceWords; x += kBlock) {
                const uint32_t w = x % kSliceWords;
                if (w >= nw) continue;
                uint64_t *to = &E[h.eoff + (uint64_t)(x / kSliceWords) * W + w0 + w];
                const uint64_t val = sE[x];
                if (w0 + w < (rlo >> 6)) *to = val;
                else if (val) atomicOr((unsigned long long *)to, val);
            }
            __syncthreads();
        }
    }
    if (CLOSED)
        for (uint32_t i = tid; i < K; i += kBlock)
            if (sCnt[i]) atomicAdd(&c2[h.ioff - i0 + i], sCnt[i]);
    if (tid == 0) {
        prof_add(out, 1, blockIdx.x, t_start);
        stamp_end(out, kStampHub);
    }
}

// Sums closed_count over the items' |C_2| counters.
__global__ __launch_bounds__(kBlock) void hub_closed_kernel(const HubRec *__restrict__ hubs,
                                                            const uint32_t *__restrict__ hub_of_item, uint64_t i0,
                                                            uint64_t i1, const uint32_t *__restrict__ c2, int closed,
                                                            KOut out)
{
    uint64_t cnt = 0;
    for (uint64_t i = i0 + blockIdx.x * (uint64_t)kBlock + threadIdx.x; i < i1; i += (uint64_t)gridDim.x * kBlock) {
        const uint32_t c = c2[i - i0];
        if (c) cnt += closed_count(closed, c, hubs[hub_of_item[i]].d);
    }
    flush_acc(out, cnt, 0, 0);
    if (threadIdx.x == 0) stamp_end(out, kStampHub);
}

// Copies a W-word row (HBM) into a wave's buffer, lane i taking words i,
// i + 64, ...; four loads per lane are in flight at a time.
__device__ __forceinline__ void copy_row(uint64_t *dst, const uint64_t *__restrict__ src, uint32_t W, int lane)
{
    for (uint32_t w0 = 0; w0 < W; w0 += 4 * 64) {
        uint64_t v[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const uint32_t w = w0 + k * 64 + lane;
            v[k] = w < W ? src[w] : 0ull;
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const uint32_t w = w0 + k * 64 + lane;
            if (w < W) dst[w] = v[k];
        }
    }
}

// k-th (0-based) set bit of w
__device__ __forceinline__ uint32_t select_bit(uint64_t w, uint32_t k)
{
    for (uint32_t i = 0; i < k; i++) w &= w - 1;
    return (uint32_t)__builtin_ctzll(w);
}

// Bit-sliced counters of the paired levels: adds a word of weight 2^J.
template <int J>
__device__ __forceinline__ void ripple_add(uint64_t *sl, uint64_t c)
{
#pragma unroll
    for (int j = J; j < kPairSlices; j++) {
        if (c) {
            const uint64_t t = sl[j] & c;
            sl[j] ^= c;
            c = t;
        }
    }
}

// a + b + c = 2 h + l, bit by bit
__device__ __forceinline__ uint64_t full_add(uint64_t &l, uint64_t b, uint64_t c)
{
    const uint64_t u = l ^ b, h = (l & b) | (u & c);
    l = u ^ c;
    return h;
}

// Adds eight words to the slices 0..2; returns the word of weight 8 left over.
__device__ __forceinline__ uint64_t add8(uint64_t *sl, const uint64_t *c)
{
    const uint64_t f0 = full_add(sl[1], full_add(sl[0], c[0], c[1]), full_add(sl[0], c[2], c[3]));
    const uint64_t f1 = full_add(sl[1], full_add(sl[0], c[4], c[5]), full_add(sl[0], c[6], c[7]));
    return full_add(sl[2], f0, f1);
}

// Hub DFS: one wave per (hub, x_1) item; lane i owns words i, i+64, ...
// The candidate stack (nlev x wmax words per wave) and, when the plan reads
// it, the bitmap row of x_1 live in LDS (LDSBUF) or, for very wide hubs, in a
// per-wave HBM slot.  Words below the largest symmetry lower bound of a level
// are neither computed nor scanned.
//
// mode 0 walks the items.  An item whose level-2 candidate set holds more
// than hq.split_min candidates is donated instead of walked: C_2 is copied to
// a donation slot and cut into chunks of hq.chunk consecutive candidates,
// each a (hub, x_1, slot, [lo, hi)) record appended to the queue with one
// atomic.  mode 1 (the next launch on the stream) drains the queue: every
// wave of the grid takes chunks and walks the x_2 in [lo, hi) of its chunk.
// PAIR compiles in the paired last levels (5-vertex pair plans: hub_pair5_kernel).
template <bool LDSBUF, bool PAIR>
__global__ __launch_bounds__(kBlock, PAIR ? 3 : 1) void hub_dfs_kernel(KGraph g, KPlan pl,
                                                         const HubRec *__restrict__ hubs,
                                                         const uint32_t *__restrict__ hub_of_item,
                                                         uint64_t i0, uint64_t i1,
                                                         unsigned long long *cursor,
                                                         const uint64_t *__restrict__ E,
                                                         uint64_t *stk, uint32_t wmax, KOut out,
                                                         HubQueue hq, int mode)
{
    extern __shared__ __align__(16) uint64_t hsm[];
    __shared__ uint32_t sX[kBlock / 64][kMaxLevels];
    __shared__ uint32_t sWlo[kBlock / 64][kMaxLevels];
    __shared__ uint32_t sQM[kMaxLevels], sSM[kMaxLevels], sLev[2 * kMaxLevels];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    if (tid < kMaxLevels) {
        sQM[tid] = pl.qmask[tid];
        sSM[tid] = pl.smask[tid];
    }
    if (tid < 2 * kMaxLevels) sLev[tid] = pl.lev[tid];
    __syncthreads();
    const int L = pl.L;
    const int nlev = L > 3 ? L - 3 : 1;
    // x_1's bitmap row is cached when some level intersects with it
    bool row1 = false;
    for (int l = 2; l < L; l++) row1 |= (sQM[l] & 2u) != 0;
    uint64_t *my;
    const uint64_t wave_words = hub_wave_words(nlev, wmax, PAIR);
    if (LDSBUF) my = hsm + (uint64_t)wv * wave_words;
    else my = stk + ((uint64_t)blockIdx.x * (kBlock / 64) + wv) * wave_words;
    uint64_t *e1 = my + (uint64_t)nlev * wmax;
    uint64_t cnt = 0, hs = 0, hx = 0;
    const uint64_t dl = *out.dl;
    const uint64_t t_start = wall_clock64();
    const uint32_t wslot = blockIdx.x * (kBlock / 64) + wv;
    uint32_t spins = 0;
    auto xget = [&](int q) -> uint32_t { return sX[wv][q]; };

    // per-item context
    const uint64_t *Eh = nullptr;
    const uint32_t *A = nullptr;
    uint32_t d = 0, W = 0, R = 0, u = 0, rlo = 0;

    // first word of level l that can hold a candidate
    auto word_lo = [&](int l) -> uint32_t {
        uint32_t lo = 0;
        uint32_t sm = sSM[l];
        while (sm) {
            const int s = __builtin_ctz(sm);
            sm &= sm - 1;
            const uint32_t v = xget(s) >> 6;
            lo = v > lo ? v : lo;
        }
        return lo;
    };
    // C_l (for l = L-1 >= 3: without x_{l-1}'s constraints, KPlan::lev) from its
    // base level's set.  The masks go first, then the rows (x_1's from LDS
    // first), and a lane whose word is already empty loads no further row word.
    auto level_word = [&](int l, uint32_t w) -> uint64_t {
        const uint32_t a = sLev[l], b = sLev[kMaxLevels + l], base = b >> 16;
        uint64_t t = !base ? valid_mask(w, d) : w >= sWlo[wv][base] ? my[(uint64_t)(base - 2) * wmax + w] : 0ull;
        uint32_t m = b & 0xffffu;
        while (m) {
            const int s = __builtin_ctz(m);
            m &= m - 1;
            t &= ~bit_at(xget(s), w);
        }
        m = a >> 16;
        while (m) {
            const int s = __builtin_ctz(m);
            m &= m - 1;
            t &= gt_mask(xget(s), w);
        }
        m = a & 0xffffu;
        if (row1 && (m & 2u)) {
            t &= e1[w];
            m &= ~2u;
        }
        while (m && t) {
            const int q = __builtin_ctz(m);
            m &= m - 1;
            t &= Eh[(uint64_t)(xget(q) - rlo) * W + w];
        }
        return t;
    };
    // x_{L-2} = x's part of the last level
    auto leaf_word = [&](uint64_t t, uint32_t x, uint32_t w) -> uint64_t {
        if (pl.leaf_gt) t &= gt_mask(x, w);
        if (pl.leaf_x) t &= ~bit_at(x, w);
        if (pl.leaf_row && t) t &= Eh[(uint64_t)(x - rlo) * W + w];
        return t;
    };

    // Summed last level (pl.tail), l = L-1: adds |C_l| over every x_{l-1} in
    // S = C_{l-1} n [pos0, hi2).  F = the part of C_l fixed by x_1..x_{l-2};
    // with carry-chained wave prefix sums of |F_w| over the rounds,
    //   sum_x |F n (x, inf)| = |S||F| - sum_w (|S_w| |F_{<=w}| - pairs_w(S, F))
    //   sum_x |F \ {x}|      = |S||F| - |S n F|
    // (words below both S's and F's first word add nothing to either).
    const bool tail_gt = pl.tail && pl.leaf_gt;
    auto tail_count = [&](int l, uint32_t pos0, uint32_t hi2) {
        const int lv = l - 1;
        const uint32_t wl = sWlo[wv][l - 1];
        const uint32_t ws = (pos0 >> 6) > wl ? (pos0 >> 6) : wl;  // first word of S
        uint32_t fl = 0;  // first word where F can be non-zero
        uint32_t fsm = sSM[l] & ~(1u << lv);
        while (fsm) {
            const int s = __builtin_ctz(fsm);
            fsm &= fsm - 1;
            const uint32_t v = xget(s) >> 6;
            fl = v > fl ? v : fl;
        }
        const uint32_t w0 = tail_gt ? ws : (ws < fl ? ws : fl);
        uint64_t acc = 0, sl = 0;
        uint32_t carry = 0;
        for (uint32_t rr = w0 >> 6; rr < R; rr++) {
            const uint32_t w = rr * 64 + lane;
            uint64_t S = 0, F = 0;
            if (w < W && w >= w0) {
                if (w >= ws) S = my[(uint64_t)(l - 3) * wmax + w] & ~lt_mask(pos0, w) & lt_mask(hi2, w);
                if (w >= fl) F = level_word(l, w);
            }
            const uint32_t sc = (uint32_t)__popcll(S);
            const uint32_t fin = wave_incl_scan((uint32_t)__popcll(F)) + carry;
            acc += tail_gt ? (uint64_t)sc * fin - pairs_in_word(S, F) : (uint64_t)__popcll(S & F);
            sl += sc;
            carry = __shfl(fin, 63, 64);
        }
        const uint64_t stot = wave_sum_u64(sl);
        if (lane == 0) cnt += stot * (uint64_t)carry;
        cnt -= acc;  // the wave's sum is exact modulo 2^64
    };

    // Paired last levels (pl.pair), l = L-2 = b: S = C_{l-1} in the stack with
    // x_1..x_{l-2} fixed, B = level b without its constraints on x_a = x_{l-1}.
    // The three levels add sum over x_b in B of
    // C(|S n E[x_b]|, 2).  Returns true when the deadline passed before it was
    // done (a hub of hundreds of thousands of neighbours makes one call long):
    // the item is left with part of its count.
    //
    // Pair plans keep both bits of every adjacent pair (a paired level c
    // intersects with the row of x_b and is bound only above x_a < x_b), so
    // |S n E[p]| = c_p = |{s in S : E[s][p]}|, and the sum is
    //   sum over p in B of C(c_p, 2)
    // over the rows of S alone.  In each round of 64 words a lane keeps the
    // c_p of its word's 64 positions as bit-sliced counters (slice j = bit j
    // of every c_p), adds the members' words eight at a time through full
    // adders, and at the round's end takes
    //   sum_p C(c_p, 2) = sum_j 2^(j-1) (2^j - 1) |sl_j|
    //                     + sum_{i<j} 2^(i+j) |sl_i & sl_j|.
    // Every member row is read once per round where B can hold candidates.
    // The members come from a list in the next stack row (u32, eight rows in
    // flight) when it holds them, else straight from S's words.  An S with more
    // members than the counters hold takes the walk at the end: B restricted
    // to the union of the members' rows, then C(|S n E[x_b]|, 2) for every x_b
    // in it.
    auto pair_count = [&](int l) -> bool {
        uint32_t steps = 0;
        const uint64_t *S = my + (uint64_t)(l - 3) * wmax;
        uint64_t *Bv = my + (uint64_t)(l - 2) * wmax;
        const uint32_t blo = word_lo(l), bhi = W;  // B's words: [blo, bhi)
        const uint32_t slo = sWlo[wv][l - 1];
        if (blo >= bhi) return false;
        // B's mask on word w (x_a's constraints left out)
        auto b_word = [&](uint32_t w) -> uint64_t {
            uint64_t t = valid_mask(w, d);
            uint32_t qm = sQM[l] & ~(1u << (l - 1));
            while (qm && t) {
                const int q = __builtin_ctz(qm);
                qm &= qm - 1;
                if (q == 1 && row1) t &= e1[w];
                else t &= Eh[(uint64_t)(xget(q) - rlo) * W + w];
            }
            for (int s = 1; s < l - 1; s++) t &= ~bit_at(xget(s), w);
            uint32_t sm = sSM[l];
            while (sm) {
                const int s = __builtin_ctz(sm);
                sm &= sm - 1;
                t &= gt_mask(xget(s), w);
            }
            return t;
        };
        {
            // members: in the next stack row, or, where rows are short, after the rows
            uint32_t *list = (uint32_t *)(wmax >= kPairListWords ? Bv : my + (uint64_t)(nlev + 1) * wmax);
            uint32_t cap = 2u * (wmax >= kPairListWords ? wmax : kPairListWords);
            if (cap > kPairMembers) cap = kPairMembers;
            uint32_t ns = 0;
            for (uint32_t rr = slo >> 6; rr < R; rr++) {
                const uint32_t w = rr * 64 + lane;
                uint64_t v = (w < W && w >= slo) ? S[w] : 0ull;
                const uint32_t pc = (uint32_t)__popcll(v);
                const uint32_t incl = wave_incl_scan(pc);
                uint32_t at = ns + incl - pc;
                if (ns + incl <= cap) {
                    while (v) {
                        list[at++] = (w << 6) + (uint32_t)__builtin_ctzll(v);
                        v &= v - 1;
                    }
                }
                ns += __shfl(incl, 63, 64);
            }
            if (ns == 0u) return false;
            if (ns <= kPairMembers) {
                const bool listed = ns <= cap;
                if (listed) {
                    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
                }
                const int nb = 32 - __builtin_clz(ns);  // bits of the largest c_p
                // A row of at most 32 words leaves lanes idle: the wave splits
                // into G groups of P lanes, each with every G-th member.
                const uint32_t P = W <= 16u ? 16u : W <= 32u ? 32u : 64u, G = 64u / P;
                const uint32_t grp = (uint32_t)lane / P;
                auto member = [&](uint32_t x, uint32_t w) -> uint64_t {
                    if (G > 1u) return Eh[__umul24(x - rlo, W) + w];
                    x = (uint32_t)__builtin_amdgcn_readfirstlane((int)x);
                    return Eh[(uint64_t)(x - rlo) * W + w];
                };
                for (uint32_t rr = blo >> 6; rr * 64 < bhi; rr++) {
                    if ((++steps & 15u) == 0u && past(dl)) return true;
                    const uint32_t w = rr * 64 + ((uint32_t)lane & (P - 1u));
                    const uint64_t bc = (w < bhi && w >= blo) ? b_word(w) : 0ull;
                    if (__ballot(bc != 0ull) == 0ull) continue;
                    uint64_t sl[kPairSlices];
#pragma unroll
                    for (int j = 0; j < kPairSlices; j++) sl[j] = 0ull;
                    if (!listed) {
                        for (uint32_t sr = slo >> 6; sr < R; sr++) {  // S's words, 64 at a time
                            const uint32_t sw = sr * 64 + lane;
                            uint64_t v = (sw < W && sw >= slo) ? S[sw] : 0ull;
                            for (;;) {
                                const uint64_t bal = __ballot(v != 0ull);
                                if (bal == 0ull) break;
                                const int f = __builtin_ctzll(bal);
                                const uint64_t vf = __shfl(v, f, 64);
                                if (lane == f) v &= v - 1ull;
                                const uint32_t x = ((sr * 64 + (uint32_t)f) << 6) + (uint32_t)__builtin_ctzll(vf);
                                ripple_add<0>(sl, bc && grp == 0 ? Eh[(uint64_t)(x - rlo) * W + w] : 0ull);
                            }
                        }
                    } else if (bc) {
                        // eight members' words at a time through full adders; what
                        // overflows the three low slices ripples on
                        uint32_t m0 = (uint32_t)grp;
                        for (; m0 + 7u * G < ns; m0 += 8u * G) {
                            uint64_t c[8];
#pragma unroll
                            for (int i = 0; i < 8; i++) c[i] = member(list[m0 + i * G], w);
                            ripple_add<3>(sl, add8(sl, c));
                        }
                        for (; m0 < ns; m0 += G) ripple_add<0>(sl, member(list[m0], w));
                    }
                    // groups hold the counters of different members: add them up
                    for (uint32_t o = P; o < 64u; o <<= 1) {
                        uint64_t carry = 0;
#pragma unroll
                        for (int j = 0; j < kPairSlices; j++)
                            if (j < nb) {
                                const uint64_t y = __shfl_xor(sl[j], o, 64), x = sl[j];
                                sl[j] = x ^ y ^ carry;
                                carry = (x & y) | (carry & (x ^ y));
                            }
                    }
                    uint64_t acc = 0;
                    if (grp == 0) {
#pragma unroll
                        for (int j = 0; j < kPairSlices; j++) {
                            if (j < nb) {
                                sl[j] &= bc;
                                if (j == 0) continue;
                                // sum over i < j of 2^i |sl_i & sl_j|, highest i first
                                uint32_t t = 0;
#pragma unroll
                                for (int i = j - 1; i >= 0; i--) t = (t << 1) + (uint32_t)__popcll(sl[i] & sl[j]);
                                acc += (uint64_t)t << j;
                                acc += ((1ull << (j - 1)) * ((1ull << j) - 1ull)) * (uint64_t)__popcll(sl[j]);
                            }
                        }
                    }
                    cnt += acc;
                }
                return false;
            }
        }
        // only an x_b adjacent to some member of S adds anything: B starts as
        // the union of their rows (words [blo, bhi))
        for (uint32_t rr = blo >> 6; rr < R; rr++) {
            const uint32_t w = rr * 64 + lane;
            if (w < bhi && w >= blo) Bv[w] = 0ull;
        }
        for (uint32_t pos = slo << 6;;) {
            uint32_t xs = 0xffffffffu;
            const uint32_t pw = pos >> 6;
            for (uint32_t rr = pw >> 6; rr < R; rr++) {
                const uint32_t w = rr * 64 + lane;
                uint64_t v = (w < W && w >= pw) ? S[w] : 0ull;
                if (w == pw) v &= (~0ull << (pos & 63u));
                const uint64_t bal = __ballot(v != 0ull);
                if (bal) {
                    const int f = __builtin_ctzll(bal);
                    const uint64_t vf = __shfl(v, f, 64);
                    xs = ((rr * 64 + (uint32_t)f) << 6) + (uint32_t)__builtin_ctzll(vf);
                    break;
                }
            }
            if (xs == 0xffffffffu) break;
            if ((++steps & 63u) == 0u && past(dl)) return true;
            const uint64_t *Es = Eh + (uint64_t)(xs - rlo) * W;  // x_a's row: kept, as the walk reads it
            for (uint32_t rr = blo >> 6; rr < R; rr++) {
                const uint32_t w = rr * 64 + lane;
                if (w < bhi && w >= blo) Bv[w] |= Es[w];
            }
            pos = xs + 1u;
        }
        __builtin_amdgcn_wave_barrier();
        for (uint32_t rr = 0; rr < R; rr++) {
            const uint32_t w = rr * 64 + lane;
            if (w >= W) break;
            Bv[w] = (w >= blo && w < bhi && Bv[w]) ? Bv[w] & b_word(w) : 0ull;
        }
        __builtin_amdgcn_wave_barrier();
        uint32_t pos = blo << 6;
        for (;;) {
            uint32_t xb = 0xffffffffu;
            const uint32_t pw = pos >> 6;
            for (uint32_t rr = pw >> 6; rr < R; rr++) {
                const uint32_t w = rr * 64 + lane;
                uint64_t v = (w < W && w >= pw) ? Bv[w] : 0ull;
                if (w == pw) v &= (~0ull << (pos & 63u));
                const uint64_t bal = __ballot(v != 0ull);
                if (bal) {
                    const int f = __builtin_ctzll(bal);
                    const uint64_t vf = __shfl(v, f, 64);
                    xb = ((rr * 64 + (uint32_t)f) << 6) + (uint32_t)__builtin_ctzll(vf);
                    break;
                }
            }
            if (xb == 0xffffffffu) break;
            if ((++steps & 63u) == 0u && past(dl)) return true;
            const uint64_t *Eb = Eh + (uint64_t)(xb - rlo) * W;
            uint32_t pc = 0;
            for (uint32_t rr = slo >> 6; rr < R; rr++) {
                const uint32_t w = rr * 64 + lane;
                if (w < W && w >= slo) {
                    const uint64_t sw = S[w];
                    if (sw) pc += (uint32_t)__popcll(sw & Eb[w]);  // x_b's row only where S has members
                }
            }
            pc = (uint32_t)wave_sum_u64(pc);
            if (lane == 0) cnt += (uint64_t)pc * (pc - 1u) / 2u;
            pos = xb + 1u;
        }
        return false;
    };

    // DFS below level 2 with C_2 in my[0, W): x_2 runs over C_2 n [pos0, hi2).
    auto dfs3 = [&](uint32_t pos0, uint32_t hi2) {
        int l = 3;
        uint32_t pos = pos0;
        for (;;) {
            if (++spins >= kClockEvery) {
                spins = 0;
                if (past(dl)) break;  // the next claim records the stop
            }
            if (pl.tail && l == L - 1) {  // every x_{L-2} of the level at once
                tail_count(l, pos, l == 3 ? hi2 : 0xffffffffu);
                if (l == 3) break;
                --l;
                pos = xget(l - 1) + 1u;
                continue;
            }
            if (PAIR && l == L - 2) {  // levels L-3..L-1 at once
                if (pair_count(l)) break;  // the next claim records the stop
                if (l == 3) break;
                --l;
                pos = xget(l - 1) + 1u;
                continue;
            }
            if (l == L - 1 && R == 1u) {
                // Rows of at most 64 words: the whole last level here, F once, four
                // x_{L-2}'s rows in flight (each is a dependent load from L2 or
                // beyond: W5's hashed matches on hubs of 865 waited 1.5 us a row)
                const uint32_t w = lane, lo = sWlo[wv][l - 1];
                uint64_t v = (w < W && w >= lo) ? my[(uint64_t)(l - 3) * wmax + w] & ~lt_mask(pos, w) : 0ull;
                if (l == 3) v &= lt_mask(hi2, w);
                const uint64_t F = w < W ? level_word(l, w) : 0ull;
                uint64_t hpre = 0;
                if (pl.emit) {
                    hpre = hash_step(hash_seed(L), 0, u);
                    for (int q = 1; q < l - 1; q++) hpre = hash_step(hpre, q, A[xget(q)]);
                }
                for (;;) {
                    uint32_t x[4];
                    uint64_t t[4];
                    int n = 0;
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        const uint64_t bal = __ballot(v != 0ull);
                        x[k] = 0;
                        if (bal) {
                            const int f = __builtin_ctzll(bal);
                            const uint64_t vf = (uint64_t)lane_u32((uint32_t)(v >> 32), f) << 32 | lane_u32((uint32_t)v, f);
                            x[k] = ((uint32_t)f << 6) + (uint32_t)__builtin_ctzll(vf);
                            if (lane == f) v &= v - 1ull;
                            n++;
                        }
                    }
                    if (n == 0) break;
#pragma unroll
                    for (int k = 0; k < 4; k++) t[k] = k < n ? leaf_word(F, x[k], w) : 0ull;
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        if (k >= n) break;
                        cnt += (uint64_t)__popcll(t[k]);
                        if (pl.emit) {
                            if (out.buf) {
                                if (lane == 0) sX[wv][l - 1] = x[k];
                                wave_lds_sync();
                            }
                            if (t[k])
                                emit_bits(out, l, u, A, hash_step(hpre, l - 1, A[x[k]]), t[k], w, xget, hs, hx);
                        }
                    }
                    spins += 4;
                    if (spins >= kClockEvery) {
                        spins = 0;
                        if (past(dl)) break;  // the next claim records the stop
                    }
                }
                if (l == 3) break;
                --l;
                pos = xget(l - 1) + 1u;
                continue;
            }
            uint32_t xi = 0xffffffffu;
            uint32_t pw = pos >> 6;
            const uint32_t wl = sWlo[wv][l - 1];
            const uint32_t start = pw > wl ? pw : wl;
            for (uint32_t rr = start >> 6; rr < R; rr++) {
                const uint32_t w = rr * 64 + lane;
                uint64_t v = (w < W && w >= start) ? my[(uint64_t)(l - 3) * wmax + w] : 0ull;
                if (w == pw) v &= (~0ull << (pos & 63u));
                const uint64_t bal = __ballot(v != 0ull);
                if (bal) {
                    const int f = __builtin_ctzll(bal);
                    const uint64_t vf = __shfl(v, f, 64);
                    xi = ((rr * 64 + (uint32_t)f) << 6) + (uint32_t)__builtin_ctzll(vf);
                    break;
                }
            }
            if (l == 3 && xi != 0xffffffffu && xi >= hi2) xi = 0xffffffffu;
            if (xi == 0xffffffffu) {
                if (l == 3) break;
                --l;
                pos = xget(l - 1) + 1u;
                continue;
            }
            if (lane == 0) sX[wv][l - 1] = xi;
            __builtin_amdgcn_wave_barrier();
            const uint32_t lo = word_lo(l);
            if (l == L - 1) {
                for (uint32_t rr = lo >> 6; rr < R; rr++) {
                    const uint32_t w = rr * 64 + lane;
                    if (w >= W) break;
                    if (w < lo) continue;
                    const uint64_t t = leaf_word(level_word(l, w), xi, w);
                    cnt += (uint64_t)__popcll(t);
                    if (pl.emit && t) emit_word(out, pl, l, u, A, t, w, xget, hs, hx);
                }
                pos = xi + 1u;
            } else {
                for (uint32_t rr = lo >> 6; rr < R; rr++) {
                    const uint32_t w = rr * 64 + lane;
                    if (w < W && w >= lo) my[(uint64_t)(l - 2) * wmax + w] = level_word(l, w);
                }
                if (lane == 0) sWlo[wv][l] = lo;
                __builtin_amdgcn_wave_barrier();
                ++l;
                pos = 0;
            }
        }
    };

    auto bind = [&](const HubRec &h, uint32_t x1) {
        d = h.d;
        W = (d + 63) >> 6;
        R = (W + 63) >> 6;
        u = h.u;
        rlo = h.rlo;
        Eh = E + h.eoff;
        A = g.ocol + h.rbeg;
        if (lane == 0) {
            sX[wv][1] = x1;
            sWlo[wv][2] = 0;
        }
        __builtin_amdgcn_wave_barrier();
        if (row1) copy_row(e1, Eh + (uint64_t)(x1 - rlo) * W, W, lane);
    };

    if (mode == 1) {
        const uint64_t ntail = *hq.tail;
        const uint64_t nq = ntail < hq.cap ? ntail : hq.cap;
        uint32_t parts = 0;  // lane 0's claim state
        for (;;) {
            unsigned long long c = ~0ull;
            if (lane == 0) {
                uint64_t cb = 0, ce = 0;
                if (past(dl)) mark_stop(out);
                else if (claim_striped(hq.head, nq, wslot % kStripes, parts, 1, cb, ce)) c = cb;
            }
            c = __shfl(c, 0, 64);
            if (c >= nq) break;
            const HubChunk ch = hq.q[c];
            if (ch.lo >= ch.hi) continue;
            bind(hubs[ch.hub], ch.x1);
            copy_row(my, hq.slots + ch.slot, W, lane);
            dfs3(ch.lo, ch.hi);
        }
        flush_acc(out, cnt, hs, hx);
        if (lane == 0) prof_add(out, 2, wslot, t_start);
        if (threadIdx.x == 0) stamp_end(out, kStampHub);
        return;
    }

    constexpr uint32_t kClaim = 4;  // items per cursor claim
    uint64_t nxt = 0, left = 0;
    uint32_t parts = 0;  // lane 0's claim state
    for (;;) {
        if (left == 0) {
            unsigned long long cb = ~0ull, cc = 0;
            if (lane == 0) {
                uint64_t b = 0, n = 0;
                if (past(dl)) mark_stop(out);
                else if (claim_striped(cursor, i1 - i0, wslot % kStripes, parts, kClaim, b, n)) {
                    cb = b;
                    cc = n;
                }
            }
            cb = __shfl(cb, 0, 64);
            cc = __shfl(cc, 0, 64);
            if (cb == ~0ull) break;
            nxt = i0 + cb;
            left = cc;
        }
        const uint64_t item = nxt;
        nxt += kStripes;
        left--;
        const uint32_t hidx = hub_of_item[item];
        const HubRec h = hubs[hidx];
        const uint32_t jl = h.jbeg + (uint32_t)(item - h.ioff);
        if (L < 3) continue;
        if (pl.closed) {  // the count follows from |C_2|: one pass over x_1's row, nothing staged
            const uint32_t hw = (h.d + 63) >> 6;
            const uint64_t *row = E + h.eoff + (uint64_t)(jl - h.rlo) * hw;
            const bool rd = (sQM[2] & 2u) != 0, gt = (sSM[2] & 2u) != 0;
            uint32_t c = 0;
            for (uint32_t w = (gt ? jl >> 6 : 0u) + lane; w < hw; w += 64) {
                uint64_t t = (rd ? row[w] : valid_mask(w, h.d)) & ~bit_at(jl, w);
                if (gt) t &= gt_mask(jl, w);
                c += (uint32_t)__popcll(t);
            }
            c = (uint32_t)wave_sum_u64(c);
            if (lane == 0 && c) cnt += closed_count(pl.closed, c, h.d);
            continue;
        }
        bind(h, jl);
        const uint32_t lo2 = word_lo(2);
        if (L == 3) {
            for (uint32_t rr = lo2 >> 6; rr < R; rr++) {
                const uint32_t w = rr * 64 + lane;
                if (w >= W) break;
                if (w < lo2) continue;
                const uint64_t t = level_word(2, w);
                cnt += (uint64_t)__popcll(t);
                if (pl.emit && t) emit_word(out, pl, 2, u, A, t, w, xget, hs, hx);
            }
            continue;
        }
        uint32_t c2 = 0;
        for (uint32_t rr = 0; rr < R; rr++) {
            const uint32_t w = rr * 64 + lane;
            if (w < W) {
                const uint64_t t = w >= lo2 ? level_word(2, w) : 0ull;
                my[w] = t;
                c2 += (uint32_t)__popcll(t);
            }
        }
        c2 = (uint32_t)wave_sum_u64(c2);
        if (hq.q && c2 > hq.split_min && !(PAIR && L == 5)) {  // L = 5: one paired pass, no x_2 to donate
            // donate: publish C_2, then cut it into chunks of hq.chunk candidates
            unsigned long long sb = 0;
            if (lane == 0) sb = atomicAdd(hq.slot_tail, (unsigned long long)W);
            sb = __shfl(sb, 0, 64);
            if (sb + W <= hq.slot_cap) {
                const uint32_t nc = (c2 + hq.chunk - 1) / hq.chunk;
                unsigned long long qb = 0;
                if (lane == 0) qb = atomicAdd(hq.tail, (unsigned long long)nc);
                qb = __shfl(qb, 0, 64);
                if (qb + nc <= hq.cap) {
                    if (lane == 0) atomicAdd(hq.donated, (unsigned long long)nc);
                    uint32_t carry = 0;
                    for (uint32_t rr = 0; rr < R; rr++) {
                        const uint32_t w = rr * 64 + lane;
                        const uint64_t t = (w < W) ? my[w] : 0ull;
                        if (w < W) hq.slots[sb + w] = t;
                        const uint32_t pc = (uint32_t)__popcll(t);
                        const uint32_t incl = wave_incl_scan(pc) + carry;
                        const uint32_t excl = incl - pc;
                        for (uint32_t c = (excl + hq.chunk - 1) / hq.chunk; c * hq.chunk < incl; c++) {
                            const uint32_t idx = (w << 6) + select_bit(t, c * hq.chunk - excl);
                            HubChunk *rec = hq.q + qb + c;
                            rec->hub = hidx;
                            rec->x1 = jl;
                            rec->slot = sb;
                            rec->lo = idx;
                            if (c > 0) hq.q[qb + c - 1].hi = idx;
                        }
                        carry = __shfl(incl, 63, 64);
                    }
                    if (lane == 0) hq.q[qb + nc - 1].hi = W << 6;
                    continue;
                }
                // queue full: neutralise the reserved records that exist, walk inline
                for (uint64_t c = qb + lane; c < qb + nc && c < hq.cap; c += 64) {
                    hq.q[c].lo = 0;
                    hq.q[c].hi = 0;
                }
            }
        }
        dfs3(0, 0xffffffffu);
    }
    flush_acc(out, cnt, hs, hx);
    if (lane == 0) prof_add(out, 1, wslot, t_start);
    if (threadIdx.x == 0) stamp_end(out, kStampHub);
}

// Hub items of 5-vertex plans with paired levels (KPlan::pair, L = 5; W5): with
// x_1 fixed, S = C_2 and B (the candidates of x_3 without x_2's constraints)
// follow from x_1 alone, and the item adds sum over p in B of C(c_p, 2),
// c_p = |{s in S : E[s][p]}| (see hub_dfs_kernel's pair_count, which deeper
// pair plans use).  No DFS, so a kernel of its own: S goes from the bitmap row
// straight into a list in LDS, nothing else is staged.
//
// The lanes take B's words from the first that can hold a candidate on; when
// fewer than 64 words are left the wave splits into groups of P lanes, each
// adding every G-th member, and the groups' counters are added at the end.
// Eight member words are in flight a lane and go through full adders together.
//
// An item is short (35 member reads on average on R-MAT scale 20), so what
// bounds it is the per-item instructions (2,500 VALU in the DFS kernel before)
// and the latency of its few dependent loads: the registers are kept to 4 waves
// per SIMD.  R-MAT scale 20, W5: 20.9 ms in the DFS kernel (items and records),
// 7.0 ms here.
//
// mode 0 walks items and cuts long ones into records of whole rounds (P = 64
// words each); mode 1 drains the records.
constexpr uint32_t kPairList = 1024;  // members listed at once, per wave
__global__ __launch_bounds__(kBlock, 4) void hub_pair5_kernel(KPlan pl, const HubRec *__restrict__ hubs,
                                                              const uint32_t *__restrict__ hub_of_item, uint64_t i0,
                                                              uint64_t i1, unsigned long long *cursor,
                                                              const uint64_t *__restrict__ E, KOut out, HubQueue hq,
                                                              int mode)
{
    __shared__ uint32_t sList[kBlock / 64][kPairList];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    uint32_t *list = sList[wv];
    const uint32_t wslot = blockIdx.x * (kBlock / 64) + wv;
    const uint64_t dl = *out.dl, t_start = wall_clock64();
    // level a = 2 is S, level b = 3 is B without x_2; both see x_1 only
    const bool s_row = (pl.qmask[2] & 2u) != 0, s_gt = (pl.smask[2] & 2u) != 0;
    const bool b_row = (pl.qmask[3] & 2u) != 0, b_gt = (pl.smask[3] & 2u) != 0;
    uint64_t cnt = 0;

    // adds the rounds [r0, r1) of item (h, x1); false: the deadline passed
    auto item_sum = [&](const HubRec &h, uint32_t x1, uint32_t ns, uint32_t r0, uint32_t r1) -> bool {
        const uint32_t d = h.d, W = (d + 63) >> 6;
        const uint64_t *Eh = E + h.eoff;
        const uint64_t *row1 = Eh + (uint64_t)(x1 - h.rlo) * W;
        const uint32_t slo = s_gt ? x1 >> 6 : 0u, blo = b_gt ? x1 >> 6 : 0u;
        const uint32_t left = W - blo;
        const uint32_t P = left <= 8u ? 8u : left <= 16u ? 16u : left <= 32u ? 32u : 64u, G = 64u / P;
        const uint32_t grp = (uint32_t)lane / P;
        const int nb = 32 - __builtin_clz(ns);
        const bool once = ns <= kPairList;
        // lists the members of rank [from, from + kPairList)
        auto fill = [&](uint32_t from) {
            wave_lds_sync();
            uint32_t base = 0;
            for (uint32_t w0 = slo; w0 < W; w0 += 64) {
                const uint32_t w = w0 + lane;
                uint64_t v = 0;
                if (w < W) {
                    v = (s_row ? row1[w] : valid_mask(w, d)) & ~bit_at(x1, w);
                    if (s_gt) v &= gt_mask(x1, w);
                }
                const uint32_t pc = (uint32_t)__popcll(v), inc = wave_incl_scan(pc);
                uint32_t at = base + inc - pc - from;  // list slot of the word's first member
                // words of a few members: a lane lists its own; fuller ones: a
                // word at a time, one lane per bit
                uint64_t dense = __ballot(pc > 4u);
                if (pc <= 4u)
                    while (v) {
                        if (at < kPairList) list[at] = (w << 6) + (uint32_t)__builtin_ctzll(v);
                        at++;
                        v &= v - 1;
                    }
                while (dense) {
                    const int f = __builtin_ctzll(dense);
                    dense &= dense - 1;
                    const uint64_t m = (uint64_t)lane_u32((uint32_t)(v >> 32), f) << 32 | lane_u32((uint32_t)v, f);
                    const uint32_t slot = lane_u32(at, f) + bits_below(m);
                    if (((m >> lane) & 1u) && slot < kPairList) list[slot] = ((w0 + (uint32_t)f) << 6) + (uint32_t)lane;
                }
                base += lane_u32(inc, 63);
                if (base >= from + kPairList) break;
            }
            wave_lds_sync();
        };
        if (once) fill(0);
        uint32_t steps = 0;
        for (uint32_t r = r0; r < r1; r++) {
            if ((++steps & 15u) == 0u && past(dl)) return false;
            const uint32_t w = blo + r * P + ((uint32_t)lane & (P - 1u));
            uint64_t bc = 0;
            if (w < W) {
                bc = (b_row ? row1[w] : valid_mask(w, d)) & ~bit_at(x1, w);
                if (b_gt) bc &= gt_mask(x1, w);
            }
            if (__ballot(bc != 0ull) == 0ull) continue;
            uint64_t sl[kPairSlices];
#pragma unroll
            for (int j = 0; j < kPairSlices; j++) sl[j] = 0ull;
            for (uint32_t from = 0; from < ns; from += kPairList) {
                if (!once) fill(from);
                const uint32_t n = ns - from < kPairList ? ns - from : kPairList;
                for (uint32_t m0 = 0; m0 < n; m0 += 8u * G) {
                    uint64_t c[8];
#pragma unroll
                    for (int i = 0; i < 8; i++) {
                        const uint32_t m = m0 + i * G + grp;
                        c[i] = 0;
                        if (G == 1u) {
                            if (m < n) {
                                const uint32_t x = (uint32_t)__builtin_amdgcn_readfirstlane((int)list[m]);
                                const uint64_t *Ex = Eh + (uint64_t)(x - h.rlo) * W;
                                if (bc) c[i] = Ex[w];
                            }
                        } else if (m < n && bc) {
                            c[i] = Eh[(uint64_t)(list[m] - h.rlo) * W + w];
                        }
                    }
                    uint64_t over = add8(sl, c);
#pragma unroll
                    for (int j = 3; j < kPairSlices; j++)
                        if (__ballot(over != 0ull) != 0ull) {
                            const uint64_t t = sl[j] & over;
                            sl[j] ^= over;
                            over = t;
                        }
                }
                if (!once && past(dl)) return false;
            }
            for (uint32_t o = P; o < 64u; o <<= 1) {
                uint64_t carry = 0;
#pragma unroll
                for (int j = 0; j < kPairSlices; j++)
                    if (j < nb) {
                        const uint64_t y = __shfl_xor(sl[j], o, 64), x = sl[j];
                        sl[j] = x ^ y ^ carry;
                        carry = (x & y) | (carry & (x ^ y));
                    }
            }
            if (grp != 0u) bc = 0;
            uint64_t acc = 0;
            sl[0] &= bc;
#pragma unroll
            for (int j = 1; j < kPairSlices; j++)
                if (j < nb) {
                    sl[j] &= bc;
                    uint32_t t = 0;  // sum over i < j of 2^i |sl_i & sl_j|, highest i first
#pragma unroll
                    for (int i = j - 1; i >= 0; i--) t = (t << 1) + (uint32_t)__popcll(sl[i] & sl[j]);
                    acc += (uint64_t)t << j;
                    acc += ((1ull << (j - 1)) * ((1ull << j) - 1ull)) * (uint64_t)__popcll(sl[j]);
                }
            cnt += acc;
        }
        return true;
    };
    // |S| of item (h, x1)
    auto members = [&](const HubRec &h, uint32_t x1) -> uint32_t {
        const uint32_t W = (h.d + 63) >> 6;
        const uint64_t *row1 = E + h.eoff + (uint64_t)(x1 - h.rlo) * W;
        uint32_t c = 0;
        for (uint32_t w = (s_gt ? x1 >> 6 : 0u) + lane; w < W; w += 64) {
            uint64_t v = (s_row ? row1[w] : valid_mask(w, h.d)) & ~bit_at(x1, w);
            if (s_gt) v &= gt_mask(x1, w);
            c += (uint32_t)__popcll(v);
        }
        return lane_u32(wave_incl_scan(c), 63);
    };
    auto hub = [&](uint32_t i) -> HubRec { return hubs[(uint32_t)__builtin_amdgcn_readfirstlane((int)i)]; };
    auto first_lane64 = [&](uint64_t v) -> uint64_t {
        return (uint64_t)lane_u32((uint32_t)(v >> 32), 0) << 32 | lane_u32((uint32_t)v, 0);
    };

    uint32_t parts = 0;  // lane 0's claim state
    if (mode == 1) {
        const uint64_t ntail = *hq.tail, nq = ntail < hq.cap ? ntail : hq.cap;
        for (;;) {
            uint64_t c = ~0ull;
            if (lane == 0) {
                uint64_t cb = 0, ce = 0;
                if (past(dl)) mark_stop(out);
                else if (claim_striped(hq.head, nq, wslot % kStripes, parts, 1, cb, ce)) c = cb;
            }
            c = first_lane64(c);
            if (c >= nq) break;
            const HubChunk ch = hq.q[c];
            if (ch.lo >= ch.hi) continue;
            const HubRec h = hub(ch.hub);
            const uint32_t x1 = (uint32_t)__builtin_amdgcn_readfirstlane((int)ch.x1);
            const uint32_t ns = members(h, x1);
            if (ns >= 2u) (void)item_sum(h, x1, ns, ch.lo, ch.hi);
        }
        flush_acc(out, cnt, 0, 0);
        if (lane == 0) prof_add(out, 2, wslot, t_start);
        if (threadIdx.x == 0) stamp_end(out, kStampHub);
        return;
    }
    constexpr uint32_t kClaim = 4;  // items per cursor claim
    uint64_t nxt = 0, left = 0;
    for (;;) {
        if (left == 0) {
            uint64_t cb = ~0ull, cc = 0;
            if (lane == 0) {
                uint64_t b = 0, n = 0;
                if (past(dl)) mark_stop(out);
                else if (claim_striped(cursor, i1 - i0, wslot % kStripes, parts, kClaim, b, n)) {
                    cb = b;
                    cc = n;
                }
            }
            cb = first_lane64(cb);
            cc = first_lane64(cc);
            if (cb == ~0ull) break;
            nxt = i0 + cb;
            left = cc;
        }
        const uint64_t item = nxt;
        nxt += kStripes;
        left--;
        const uint32_t hidx = hub_of_item[item];
        const HubRec h = hub(hidx);
        const uint32_t x1 = h.jbeg + (uint32_t)(item - h.ioff);
        const uint32_t ns = members(h, x1);
        if (ns < 2u) continue;  // no pair
        const uint32_t words = ((h.d + 63) >> 6) - (b_gt ? x1 >> 6 : 0u);
        const uint32_t rounds = (words + 63u) >> 6;  // more than one: P = 64
        uint32_t rpc = kPairChunkWork / ns;
        if (rpc < 1u) rpc = 1u;
        const uint32_t nc = (rounds + rpc - 1u) / rpc;
        if (hq.q && nc >= 2u && (uint64_t)ns * rounds > kPairSplitWork) {
            uint64_t qb = 0;
            if (lane == 0) qb = atomicAdd(hq.tail, (unsigned long long)nc);
            qb = first_lane64(qb);
            if (qb + nc <= hq.cap) {
                if (lane == 0) atomicAdd(hq.donated, (unsigned long long)nc);
                for (uint32_t c = lane; c < nc; c += 64) {
                    HubChunk *rec = hq.q + qb + c;
                    rec->hub = hidx;
                    rec->x1 = x1;
                    rec->slot = 0;
                    rec->lo = c * rpc;
                    rec->hi = c + 1u == nc ? rounds : (c + 1u) * rpc;
                }
                continue;
            }
            // queue full: neutralise the reserved records that exist, walk inline
            for (uint64_t c = qb + lane; c < qb + nc && c < hq.cap; c += 64) {
                hq.q[c].lo = 0;
                hq.q[c].hi = 0;
            }
        }
        if (!item_sum(h, x1, ns, 0, rounds)) continue;  // the next claim records the stop
    }
    flush_acc(out, cnt, 0, 0);
    if (lane == 0) prof_add(out, 1, wslot, t_start);
    if (threadIdx.x == 0) stamp_end(out, kStampHub);
}

// ------------------------------------------------------------ launchers

// Workgroups of a kernel per CU with `lds` bytes of dynamic LDS, and its
// dynamic-LDS attribute raised to at least `lds`.  Both are host calls of
// several microseconds on the launch path of every query, so they are made
// once per (kernel, LDS size); the attribute only ever grows.
struct LdsLaunchCache {
    std::mutex mu;
    size_t attr = 0;
    size_t lds[16] = {};
    int occ[16] = {};
    int n = 0;
    int get(const void *fn, size_t bytes)
    {
        std::lock_guard<std::mutex> lk(mu);
        for (int i = 0; i < n; i++)
            if (lds[i] == bytes) return occ[i];
        if (bytes > attr) {
            (void)hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
            attr = bytes;
        }
        int nb = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, fn, kBlock, bytes) != hipSuccess || nb < 1) nb = 1;
        if (n < 16) {
            lds[n] = bytes;
            occ[n++] = nb;
        }
        return nb;
    }
};

constexpr int kBesideHubs = 3;
constexpr uint32_t kMaxParts = 16;

template <int P, int MinWaves, int WALK>
static hipError_t launch_lds_p(int cus, size_t lds, hipStream_t st, const KGraph &g, const KPlan &pl,
                               const RootRec *recs, const uint32_t *bf, const uint32_t *bc,
                               uint32_t b0, uint32_t b1, unsigned long long *cursor, const LdsLayout &lay,
                               const KOut &out)
{
    static LdsLaunchCache cache;
    int occ = cache.get((const void *)lds_batch_kernel<P, MinWaves, WALK>, lds);
    // Beside hub kernels a class leaves them wave slots: with seven workgroups
    // per CU the hub chain's second kernel started 245 us late (diamond, 1.1M
    // vertices); the query takes 749 us with 3 per CU, 784 with 4, 809 with 5,
    // 826 with 6.
    if (MinWaves == 1 && occ > kBesideHubs) occ = kBesideHubs;
    int grid = occ * cus;
    uint32_t parts = 1;
    if (pl.deep && WALK != kWalkNone) parts = std::min(kMaxParts, std::max(1u, (uint32_t)grid / (b1 - b0)));
    if ((uint64_t)grid > (uint64_t)(b1 - b0) * parts) grid = (int)((b1 - b0) * parts);
    if (grid < 1) grid = 1;
    hipLaunchKernelGGL((lds_batch_kernel<P, MinWaves, WALK>), dim3(grid), dim3(kBlock), lds, st, g, pl, recs, bf,
                       bc, b0, b1, parts, cursor, lay, out);
    return hipGetLastError();
}

// Dispatch on the DFS group width and the plan's walk.
template <int LG>
static hipError_t launch_lds_lg(int cus, hipStream_t st, const KGraph &g, const KPlan &pl, const RootRec *recs,
                                const uint32_t *bf, const uint32_t *bc, uint32_t b0, uint32_t b1,
                                unsigned long long *cursor, const KOut &out, bool dense)
{
    constexpr int P = 1 << LG;
    LdsNeeds need;
    need.add(pl, LG);
    const LdsLayout lay = make_lds_layout(LG, need);
#define BEEP_RUN(MW, WALK) launch_lds_p<P, MW, WALK>(cus, lay.bytes, st, g, pl, recs, bf, bc, b0, b1, cursor, lay, out)
    if (pl.closed) return dense ? BEEP_RUN(7, kWalkNone) : BEEP_RUN(1, kWalkNone);
    if constexpr (LG <= 3) {
        if (lds_lane_walk(pl, LG)) {
            if (pl.emit) return dense ? BEEP_RUN(LG == 3 ? 4 : 6, kWalkLaneEmit) : BEEP_RUN(1, kWalkLaneEmit);
            return dense ? BEEP_RUN(7, kWalkLane) : BEEP_RUN(1, kWalkLane);
        }
    }
    return dense ? BEEP_RUN(7, kWalkGroup) : BEEP_RUN(1, kWalkGroup);
#undef BEEP_RUN
}

hipError_t launch_lds_batches(int lg, int cus, hipStream_t st, const KGraph &g, const KPlan &pl,
                              const RootRec *recs, const uint32_t *bf, const uint32_t *bc,
                              uint32_t b0, uint32_t b1, unsigned long long *cursor, const KOut &out, bool dense)
{
    switch (lg) {
#define BEEP_CASE(LG) \
    case LG: return launch_lds_lg<LG>(cus, st, g, pl, recs, bf, bc, b0, b1, cursor, out, dense);
        BEEP_CASE(0) BEEP_CASE(1) BEEP_CASE(2) BEEP_CASE(3) BEEP_CASE(4) BEEP_CASE(5) BEEP_CASE(6)
#undef BEEP_CASE
    }
    return hipErrorInvalidValue;
}

// Zero fill (used instead of memset nodes so launch sequences can be captured).
// With dl set, a workgroup that starts after that deadline clears nothing: a
// hub round's arena is only read by kernels that stop at the same deadline.
__global__ void fill_zero_u32_kernel(uint32_t *p, uint64_t n, const unsigned long long *dl)
{
    if (dl && past(*dl)) return;
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        p[i] = 0u;
}

hipError_t launch_fill_zero(void *p, uint64_t bytes, hipStream_t st, const unsigned long long *dl)
{
    const uint64_t n = (bytes + 3) / 4;
    if (n == 0) return hipSuccess;
    uint64_t blocks = (n + 4 * kBlock - 1) / (4 * kBlock);
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(fill_zero_u32_kernel, dim3((uint32_t)blocks), dim3(kBlock), 0, st, (uint32_t *)p, n, dl);
    return hipGetLastError();
}

// First kernel of a launch sequence: clears the n counter words and writes
// the deadlines of the hub and the LDS kernels at words dl and dl + 1:
// now + ticks, or none (all ones).
__global__ void begin_sequence_kernel(unsigned long long *ctr, uint64_t n, uint64_t dl, uint64_t ticks_hub,
                                      uint64_t ticks_lds)
{
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        unsigned long long v = 0;
        if (i == dl || i == dl + 1) {
            const uint64_t t = i == dl ? ticks_hub : ticks_lds;
            v = t ? (unsigned long long)wall_clock64() + t : ~0ull;
        }
        if (i == dl + 3) v = (unsigned long long)wall_clock64();  // the sequence's start
        ctr[i] = v;
    }
}

// Last kernel of a launch sequence: copies the n result words to the record in
// host memory, with the time now as word t_end, followed by the stamps' maxima
// over their stripes.  (A copy command waits for the kernels on a queue of its
// own and took 15 to 20 us from the last kernel's end to the host.)
__global__ void end_sequence_kernel(const unsigned long long *ctr, uint32_t n, uint32_t t_end,
                                    const unsigned long long *stamp, unsigned long long *rec)
{
    for (uint32_t i = threadIdx.x; i < n; i += blockDim.x)
        rec[i] = i == t_end ? (unsigned long long)wall_clock64() : ctr[i];
    if (threadIdx.x < (uint32_t)kStampWords) {
        unsigned long long m = 0;
        for (int s = 0; s < kStripes; s++) {
            const unsigned long long x = stamp[s * kLine + threadIdx.x];
            m = x > m ? x : m;
        }
        rec[n + threadIdx.x] = m;
    }
}

hipError_t launch_end_sequence(const unsigned long long *ctr, uint32_t n, uint32_t t_end, const unsigned long long *stamp,
                               unsigned long long *rec, hipStream_t st)
{
    hipLaunchKernelGGL(end_sequence_kernel, dim3(1), dim3(kBlock), 0, st, ctr, n, t_end, stamp, rec);
    return hipGetLastError();
}

hipError_t launch_begin_sequence(unsigned long long *ctr, uint64_t n, uint64_t dl, uint64_t ticks_hub,
                                 uint64_t ticks_lds, hipStream_t st)
{
    const uint64_t blocks = (n + kBlock - 1) / kBlock;
    hipLaunchKernelGGL(begin_sequence_kernel, dim3((uint32_t)(blocks ? blocks : 1)), dim3(kBlock), 0, st, ctr, n, dl,
                       ticks_hub, ticks_lds);
    return hipGetLastError();
}

// One lane class's batches (lg: the widest of them) of several queries.
template <int P>
static hipError_t launch_lds_multi_p(int cus, hipStream_t st, const MultiQuery *qs, const MultiWork *work,
                                     uint32_t nwork, unsigned long long *cursor, const LdsLayout &lay)
{
    static LdsLaunchCache cache;
    int grid = cache.get((const void *)lds_multi_kernel<P>, lay.bytes) * cus;
    if ((uint32_t)grid > nwork) grid = (int)nwork;
    if (grid < 1) grid = 1;
    hipLaunchKernelGGL((lds_multi_kernel<P>), dim3(grid), dim3(kBlock), lay.bytes, st, qs, work, nwork, cursor, lay);
    return hipGetLastError();
}

hipError_t launch_lds_multi(int cus, hipStream_t st, const MultiQuery *qs, const MultiWork *work,
                            uint32_t nwork, unsigned long long *cursor, const LdsNeeds &need, int lg)
{
    const LdsLayout lay = make_lds_layout(lg, need);
    switch (lg) {
#define BEEP_CASE(LG) \
    case LG: return launch_lds_multi_p<(1 << LG)>(cus, st, qs, work, nwork, cursor, lay);
        BEEP_CASE(0) BEEP_CASE(1) BEEP_CASE(2) BEEP_CASE(3) BEEP_CASE(4) BEEP_CASE(5) BEEP_CASE(6)
#undef BEEP_CASE
    }
    return hipErrorInvalidValue;
}

hipError_t launch_hub_hash(int grid, hipStream_t st, const KGraph &g, const HubRec *hubs,
                           const uint32_t *hor, uint64_t g0, uint64_t g1, uint64_t *kv,
                           const unsigned long long *dl)
{
    hipLaunchKernelGGL(hub_hash_kernel, dim3(grid), dim3(kBlock), 0, st, g, hubs, hor, g0, g1, kv, dl);
    return hipGetLastError();
}

hipError_t launch_hub_encode(int grid, hipStream_t st, const KGraph &g, const HubRec *hubs,
                             const uint32_t *hor, const uint64_t *hrange, const uint64_t *rows, uint64_t nrows,
                             const uint64_t *kv, uint64_t *E, int upper, int count, const KOut &out)
{
    hipLaunchKernelGGL(hub_encode_kernel, dim3(grid), dim3(kBlock), 0, st, g, hubs, hor, hrange, rows, nrows, kv, E,
                       upper, count, out);
    return hipGetLastError();
}

// c2 set: count the slices' pairs per item (CLOSED); else build bitmap words in E.
hipError_t launch_hub_slices(hipStream_t st, const KGraph &g, const HubRec *hubs, const SliceRec *slices, uint32_t n,
                             const uint64_t *hrange, uint32_t kmax, uint32_t bin_ratio, uint64_t *E, uint32_t *c2,
                             uint64_t i0, const KOut &out)
{
    const SliceLayout lay = make_slice_layout(kmax, c2 != nullptr);
    static LdsLaunchCache cache[2];
    if (c2) {
        (void)cache[1].get((const void *)hub_slice_kernel<true>, lay.bytes);
        hipLaunchKernelGGL((hub_slice_kernel<true>), dim3(n), dim3(kBlock), lay.bytes, st, g, hubs, slices, hrange,
                           bin_ratio, E, c2, i0, lay, out);
    } else {
        (void)cache[0].get((const void *)hub_slice_kernel<false>, lay.bytes);
        hipLaunchKernelGGL((hub_slice_kernel<false>), dim3(n), dim3(kBlock), lay.bytes, st, g, hubs, slices, hrange,
                           bin_ratio, E, c2, i0, lay, out);
    }
    return hipGetLastError();
}

hipError_t launch_hub_closed(int grid, hipStream_t st, const HubRec *hubs, const uint32_t *hoi, uint64_t i0, uint64_t i1,
                             const uint32_t *c2, int closed, const KOut &out)
{
    hipLaunchKernelGGL(hub_closed_kernel, dim3(grid), dim3(kBlock), 0, st, hubs, hoi, i0, i1, c2, closed, out);
    return hipGetLastError();
}

// Dynamic LDS of the hub DFS: per wave nlev + 1 rows of wmax words (and a member list).
static size_t hub_lds_bytes(int nlev, uint32_t wmax, bool pair)
{
    return (size_t)(kBlock / 64) * hub_wave_words(nlev, wmax, pair) * 8;
}
constexpr size_t kHubLdsMax = 96 * 1024;

bool hub_dfs_in_lds(int nlev, uint32_t wmax, bool pair) { return hub_lds_bytes(nlev, wmax, pair) <= kHubLdsMax; }

// one cache per instantiation: [in LDS][pair]
static LdsLaunchCache &hub_dfs_cache(bool in_lds, bool pair)
{
    static LdsLaunchCache c[2][2];
    return c[in_lds][pair];
}

// The instantiation a plan runs: the stack in LDS or HBM, and the paired last
// levels compiled in only for the plans that have them (their counters cost
// registers, hence occupancy, that the other plans keep).
static const void *hub_dfs_fn(int nlev, uint32_t wmax, bool pair)
{
    if (hub_dfs_in_lds(nlev, wmax, pair))
        return pair ? (const void *)hub_dfs_kernel<true, true> : (const void *)hub_dfs_kernel<true, false>;
    return pair ? (const void *)hub_dfs_kernel<false, true> : (const void *)hub_dfs_kernel<false, false>;
}

hipError_t launch_hub_dfs(int grid, hipStream_t st, const KGraph &g, const KPlan &pl, const HubRec *hubs,
                          const uint32_t *hoi, uint64_t i0, uint64_t i1, unsigned long long *cursor,
                          const uint64_t *E, uint64_t *stk, uint32_t wmax, const KOut &out,
                          const HubQueue &hq, int mode)
{
    if (hub_pair5(pl.L, pl.pair != 0, wmax)) {
        hipLaunchKernelGGL(hub_pair5_kernel, dim3(grid), dim3(kBlock), 0, st, pl, hubs, hoi, i0, i1, cursor, E, out, hq,
                           mode);
        return hipGetLastError();
    }
    const int nlev = pl.L > 3 ? pl.L - 3 : 1;
    const bool in_lds = hub_dfs_in_lds(nlev, wmax, pl.pair != 0);
    const size_t lds = in_lds ? hub_lds_bytes(nlev, wmax, pl.pair != 0) : 0;
    const void *fn = hub_dfs_fn(nlev, wmax, pl.pair != 0);
    if (in_lds) (void)hub_dfs_cache(true, pl.pair != 0).get(fn, lds);
    void *args[] = {(void *)&g,  (void *)&pl,     (void *)&hubs, (void *)&hoi, (void *)&i0,
                    (void *)&i1, (void *)&cursor, (void *)&E,    (void *)&stk, (void *)&wmax,
                    (void *)&out, (void *)&hq,    (void *)&mode};
    return hipLaunchKernel(fn, dim3(grid), dim3(kBlock), args, lds, st);
}

int hub_dfs_occupancy(int nlev, uint32_t wmax, bool pair)
{
    if (hub_pair5(nlev + 3, pair, wmax)) {
        static LdsLaunchCache cache;
        return cache.get((const void *)hub_pair5_kernel, 0);
    }
    const void *fn = hub_dfs_fn(nlev, wmax, pair);
    const bool in_lds = hub_dfs_in_lds(nlev, wmax, pair);
    return hub_dfs_cache(in_lds, pair).get(fn, in_lds ? hub_lds_bytes(nlev, wmax, pair) : 0);
}

// Workgroups per CU the HBM stacks are sized for: those of the DFS kernel with
// the stack rows alone in LDS.
int hub_stack_occupancy(int nlev, uint32_t wmax, bool pair)
{
    const size_t lds = hub_lds_bytes(nlev, wmax, false);
    const bool in_lds = lds <= kHubLdsMax;
    return hub_dfs_cache(in_lds, pair).get(hub_dfs_fn(nlev, wmax, pair), in_lds ? lds : 0);
}

}  // namespace beep
