// engine.hpp -- device-side state of prepared queries and the launch
// sequence, shared by the single-query engine, batches and the server.
#pragma once

#include <hip/hip_runtime.h>

#include <vector>

#include "internal.hpp"
#include "sgm_kernels.hpp"

namespace beep {

#define HIP_CHECK(x)                                                                            \
    do {                                                                                        \
        hipError_t e_ = (x);                                                                    \
        if (e_ != hipSuccess)                                                                   \
            throw Error(BEEP_EDEVICE, std::string(#x) + ": " + hipGetErrorString(e_));         \
    } while (0)

// Counter words of one launch sequence (u64), in 128-byte lines of kLine
// words.  Read back after the run (kCtrWords): the kStripes accumulator
// stripes (kCtrAcc; see KOut::acc), then one line with the donation tail,
// slot tail and donated count, the deadlines of the hub and the LDS kernels,
// the stop flag and the sequence's start and end times.  Cleared but not read
// back: striped work cursors (kCurWords each) of the hub rounds (64), the
// donation drain and the LDS lane classes (31), and the stamps (KOut::stamp),
// whose maxima follow the read-back words in the host's record (kRecWords).
constexpr int kCtrAcc = 0;
constexpr int kCtrQTail = kStripes * kLine, kCtrSlot = kCtrQTail + 1, kCtrDonated = kCtrQTail + 2,
              kCtrDeadline = kCtrQTail + 3, kCtrStop = kCtrQTail + 5, kCtrT0 = kCtrQTail + 6,
              kCtrTEnd = kCtrQTail + 7;
constexpr int kCtrWords = (kStripes + 1) * kLine;
constexpr int kCurWords = kStripes * kLine;
constexpr int kCtrHub = kCtrWords, kCtrHead = kCtrHub + 64 * kCurWords, kCtrLds = kCtrHead + kCurWords,
              kCtrStamp = kCtrLds + 31 * kCurWords, kCtrTotal = kCtrStamp + kCurWords;
static_assert(kCurWords >= kStripes * kLine, "stamps fill a cursor's words");
constexpr int kRecWords = kCtrWords + kStampWords;

// HBM copy of a variant: oriented rows and per-vertex records.
struct DevGraph {
    int device = -1;
    uint32_t *ocol = nullptr;
    VInfo *vinfo = nullptr;
    uint32_t *htab = nullptr;  // lookup tables of the larger-key ranges (2 m slots)
    ~DevGraph();
};

struct HubRound {
    uint32_t h0, h1;      // hub index range
    uint64_t g0, g1;      // global row range (bitmap build)
    uint64_t i0, i1;      // global item range (DFS)
    uint64_t ewords;      // bitmap words used
    uint64_t hslots;      // hash slots used
    uint64_t er0 = 0, er1 = 0;  // its rows with a non-empty scan range outside slices: enc_rows[er0, er1)
    uint32_t s0 = 0, s1 = 0;    // its slices
};

// Read-only device records of one prepared root queue.
struct DevRoots {
    RootRec *recs = nullptr;
    uint32_t *batch_first = nullptr, *batch_count = nullptr;
    uint32_t nbatches = 0;
    HubRec *hubs = nullptr;
    uint32_t *hub_of_row = nullptr, *hub_of_item = nullptr;
    // per hub row: the part of the row vertex's larger-key range the bitmap
    // build streams (start | length << kRangeShift)
    uint64_t *hub_range = nullptr;
    uint64_t *enc_rows = nullptr;  // per round, the hub rows whose scan range is not empty and in no slice
    SliceRec *slices = nullptr;    // per round, heaviest first
    uint32_t slice_kept = 0;       // most kept rows of a hub in slices
    bool all_sliced = false;       // every hub row with a scan range is in a slice
    int skip_split = -1;  // plan property the hub items were built for
    uint32_t nhubs = 0;
    uint32_t wmax = 0;
    std::vector<HubRound> rounds;
    uint64_t arena_budget = 0;            // bytes the rounds were cut for
    uint64_t arena_words = 0, arena_slots = 0;
    uint64_t don_words = 0, don_records = 0, don_fine = 0;  // upper bounds of the donation ring
    void release();
};

// Scratch sizes of one launch sequence.
struct ScratchNeeds {
    uint64_t arena_words = 0, hash_slots = 0, stk_words = 0;
    uint64_t queue_cap = 0, slot_cap = 0, dbuf_words = 0, prof_words = 0;
    uint64_t queue_min = 0;  // what queue_cap may be cut to where space is short
    uint64_t bytes() const;
};

// Scratch of one launch sequence, carved out of one device region.
struct Scratch {
    uint64_t *arena = nullptr;
    uint64_t *kv = nullptr;  // hub hash slots: key (vertex + 1) | row index << 32
    uint64_t *stk = nullptr;
    HubChunk *queue = nullptr;
    uint64_t *slots = nullptr;
    uint32_t *dbuf = nullptr;
    unsigned long long *ctr = nullptr;
    unsigned long long *prof = nullptr;
    ScratchNeeds cap;
};
void carve(Scratch &s, char *base, const ScratchNeeds &n);

// Streams and events of one launch sequence: the heaviest LDS lane class on
// `main` right after the counters are cleared, the hub rounds on side[0], the
// other lane classes on the side streams (side[1..] when there are more).
struct Lane {
    static constexpr int kMaxSide = 3;  // with main: the 4 hardware queues a process gets by default
    int device = -1;
    int nside = 0;
    hipStream_t main = nullptr;
    hipStream_t side[kMaxSide] = {};
    hipEvent_t fork = nullptr, done = nullptr;  // main: counters cleared; everything done
    hipEvent_t side_done[kMaxSide] = {};
    static constexpr int kMaxClasses = 31;
    unsigned long long *rec = nullptr;  // the run's record (kRecWords), pinned
    void create(int device, int nside);
    ~Lane();
};

// Single-query device state of a Prep: its records, an owned scratch
// region and a lane.
struct DevPrep {
    int device = -1;
    int cus = 0;
    DevRoots roots;
    char *region = nullptr;
    uint64_t region_bytes = 0;
    Scratch scratch;
    Lane lane;
    ~DevPrep();
};

// Everything one enumeration launch sequence needs.
struct LaunchCfg {
    KPlan kp{};
    KGraph kg{};
    KOut out{};
    HubQueue hq{};  // q == nullptr: donation off
    int hub_grid = 0;
    int nlev = 1;
    int lmin = 0;
    bool donate = false;
    uint64_t deadline_ticks = 0;      // hub kernels
    uint64_t deadline_ticks_lds = 0;  // LDS kernels
};

// Zero fill kernel (no memset nodes, so sequences can be captured) and the
// first kernel of a launch sequence, which clears n counter words and writes
// the deadlines at words dl, dl + 1.
// dl: skip the clear once that deadline has passed (hub arenas only)
hipError_t launch_fill_zero(void *p, uint64_t bytes, hipStream_t st, const unsigned long long *dl = nullptr);
hipError_t launch_begin_sequence(unsigned long long *ctr, uint64_t n, uint64_t dl, uint64_t ticks_hub,
                                 uint64_t ticks_lds, hipStream_t st);

int device_cus(int device);
uint64_t wall_clock_khz(int device);

// Uploads the variant (once per variant) and the root records of pp, with hub
// rounds cut to arena_budget bytes (0: the default budget).
void upload(Prep &pp, int device, int skip_split, uint64_t arena_budget = 0);
ScratchNeeds scratch_needs(const Prep &pp, const Plan &p, const beep_opts &o, int cus);
// lds_deadline_ms < 0: the LDS kernels share o.deadline_ms
LaunchCfg make_launch(const Prep &pp, const Plan &p, const beep_opts &o, const Scratch &s, int cus,
                      double lds_deadline_ms = -1.0);
// clear counters + deadline, LDS classes and hub rounds on main and the side
// streams, join, record -> lane.rec; records lane.done at the end.
void enqueue_query(const Prep &pp, const LaunchCfg &c, const Scratch &s, Lane &lane);
hipError_t launch_end_sequence(const unsigned long long *ctr, uint32_t n, uint32_t t_end, const unsigned long long *stamp,
                               unsigned long long *rec, hipStream_t st);
void enqueue_hubs(const Prep &pp, const LaunchCfg &c, const Scratch &s, hipStream_t st);
// LDS lane classes, one launch each, on one stream.
void enqueue_lds_classes(const Prep &pp, const LaunchCfg &c, const Scratch &s, hipStream_t st);
// Device times of a run from its record (ms): t_enum_ms, t_hub_ms and t_lds_ms
// from the first kernel's start, and each lane class's launch.
void fill_times(const unsigned long long *rec, int device, beep_result &res);
void fill_result(const beep_opts &o, const unsigned long long *acc, beep_result &res);
// Balance figures from the busy-time accumulators (kProfPhases x kProfSlots).
void fill_profile(const unsigned long long *prof, beep_result &res);

}  // namespace beep
