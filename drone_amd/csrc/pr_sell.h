// fp64 pull PageRank of small and mid-size matrices: one launch per iteration.
//
// Such an iteration is bound by latency, not by bytes: R-MAT scale 12 / 16 (53 K / 955 K entries) took 17.1 / 18.7 us as
// two launches of the row-block path (zero 128 KB of accumulators, sweep, epilogue; then the fix-up with its two-level
// tickets for the dangling mass), where a launch that follows another on a stream costs 2.3 us and the bytes less than
// one.  Here a row belongs to one wavefront (or, a hub row, to one work-group), so nothing straddles and nothing is left
// to fix up, and the dangling mass travels as one partial per work-group that EVERY work-group of the next launch adds
// up for itself - a few KB out of L2, in flight beside the entries.
//
// Layout.  Rows are sorted by length, longest first, and that order is the plan's vertex order (sources are renumbered
// alike, so an iteration writes the next gather source with coalesced stores).  A row of L entries gets P = 1 ... 64
// lanes, the power of two that leaves a lane at most kSellDepth entries; 64 / P neighbouring rows form a slice, one
// wavefront.  A slice's entries are stored step by step, 64 consecutive source ids per step (lane = row in slice * P + q
// takes the row's entries q, q + P, ...), padded to the longest row of the slice - the first, and its neighbours in the
// sort are about as long - with the id of a source that is always 0.  Rows of more than 64 * kSellWaveSteps entries are
// hubs: a work-group each, T consecutive ids per step.  Every sum has a fixed order, so the results are bitwise repeatable.
//
// Measured, R-MAT edge factor 16, us per iteration (row blocks before, this): 1 K vertices 11.6 -> 4.05, 4 K 17.1 -> 4.3,
// 16 K 18.3 -> 4.7, 64 K 19.4 -> 8.0, 131 K 24.0 -> 14.2, 262 K 32.1 -> 24.3, 524 K 43.8 -> 41.3; the plan takes
// 0.13 ... 1.2 ms instead of 0.3 ... 2.7 ms.  Below 16 K vertices it is a launch (2.3 us) plus one chain of slice
// descriptor, ids, gathers and the partials' sum out of a cold L2; at 64 K and more the rate of gathers that hit L2.
// Lanes of 4 or 16 entries (kSellDepth) instead of 8: 10.0 / 9.3 us at 64 K.
//
// Larger matrices whose hubs are named often enough keep the first kSellHot sources - rows of many entries are named often, so
// they come first - in every CU's LDS (sell_iterate_hot_kernel): 131 K 14.2 -> 11.8, 262 K 24.3 -> 18.1, 524 K 41.3 -> 37.0, 0.4 M
// vertices and 7.0 M entries 35.7 -> 33.  What is left is the rate of the other gathers, and a round trip or two per slice
// (deeper lanes, 16 instead of 8 entries: 11.1 / 18.0 / 38.4 with an id array of their own; floats, whose rows are longer, have 16).
#pragma once
#include "spmv_merge.h"

namespace drone {

constexpr int kSellClasses = 7;      // P = 64, 32, ..., 1
constexpr int kSellDepth = 8;        // most entries of a lane in a slice with P < 64; gathers in flight per lane
// Gathers in flight per lane of a hub row's work-group, and most steps of a slice with P = 64 (longer rows are hubs) without / with
// the hottest sources in LDS.  In a small matrix the longest rows are what a launch waits for.  Runs of 20 iterations at 18 sizes, 700
// to 100,003 vertices and 4 to 30 entries a row, against 8 in flight and 16 steps, geometric mean and the two ends: 16 and 12 1.038 times as
// fast (40,009 vertices with 8 entries 119 -> 100 us, with 20 entries 130 -> 138), 12 and 10 1.041 (119 -> 100; 100,003 with 9 163 -> 170),
// 16 and 8 1.035 (119 -> 100; 130 -> 137), 12 and 12 1.034 (119 -> 100; 130 -> 135), 8 and 8 1.029, 8 and 12 1.020, 16 and 14 1.014: as good
// as any, and the best at R-MAT scale 16 with 16 entries (178 -> 162; 12 and 10 168, 12 and 12 169).
constexpr int kSellHubDepth = 16, kSellWaveSteps = 12, kSellWaveStepsWide = 16;
constexpr int kSellDepthF32 = 16, kSellWaveStepsF32 = 32;  // the same of float rows
constexpr int kSellHot = 20000;      // sources that a work-group of sell_iterate_hot_kernel keeps in LDS: 160,000 of 163,840 bytes

// When the work-groups of a run in one launch stop waiting for the others (sell_enter): not before `patience` looks, and when `places` have
// come.  A negative patience is that of a test: none for the others' sources either.
struct SellGate {
    int patience = 64, places = INT_MAX;
    int enough = 1, price = 0;  // work-groups as good as all, and looks that the run is worth to one: of the run
};

struct SellRows {
    int64_t n = 0, nnz = 0;
    int threads = 256;               // work-group size of the iteration, 256 or 512; 1,024 with the hot sources in LDS
    int hot = 0;                     // sources kept in LDS, or 0: ids from there on are one more, and that number is the padding
    int hubs = 0, slices = 0, blocks = 0;
    int row_begin[kSellClasses + 1] = {};    // first row of the class (row_begin[kSellClasses] = n)
    int slice_begin[kSellClasses + 1] = {};  // first slice of the class
    int32_t *order = nullptr;        // device [n]: row -> caller's id
    int32_t *hub_step = nullptr;     // device [hubs + 1]: first step (of `threads` ids) of a hub row in hub_col
    int4 *slice = nullptr;           // device [slices]: {first step (of 64 ids) in col, steps, first row, rows << 3 | log2 P}
    int32_t *hub_col = nullptr;
    int32_t *col = nullptr;
    double *c[2] = {nullptr, nullptr};     // device [n + 1]: gather sources; [n] stays 0
    double *inv = nullptr;           // device [n]: inverse out-degrees in row order, refreshed by every run
    double *part[2] = {nullptr, nullptr};  // device: dangling mass per work-group, of this iteration and the one before
    int init_blocks = 0;
    SellGate rule;                   // of sell_resident_kernel
    int resident = 0;                // work-groups of sell_resident_kernel, or 0: a launch per iteration
    int resident_iters = 0;          // iterations of the shortest run that it does
    int staged = 0;                  // slots that a lane of it brings into LDS
    size_t lds = 0;                  // bytes of its sources in LDS
    int live = 0, live_slices = 0;   // rows with entries, and the slices that have one of them
    unsigned long long *exchange = nullptr;  // device [4 n]: its sources on their way, kSellNone between runs
    unsigned *gate = nullptr;        // device [3 * kTicketStride]: who has come and who has left, 0 between runs; `failed`
    int *failed = nullptr;           // pinned: a work-group of a run has given up waiting for another, and no call has reported it yet
    DeviceArena arena;               // everything above
    DeviceArena entries;             // hub_col and col, whose sizes are known last
};

// Whether the layout suits the matrix (n rows, nnz entries).
bool sell_suits(int64_t n, int64_t nnz);
int sell_create(SellRows *sr, int64_t n, int64_t nnz, const int64_t *row_ptr, const int32_t *col, hipStream_t stream);
// The rows alone, for float sources of which a work-group keeps kSellHotF32: sr->hot is 0, and nothing built, where the entries name
// too few of them.  Fills `order` and the entries, and new_id (device [n]): caller's id -> source.
constexpr int kSellHotF32 = 2 * kSellHot;
bool sell_f32_suits(int64_t n, int64_t nnz);
int sell_create_f32(SellRows *sr, int64_t n, int64_t nnz, const int *row_ptr, const int32_t *col, int32_t *new_id, hipStream_t stream);
constexpr int kSellHotThreads = 1024, kSellHotBlocks = 256;
// One superstep's aggregation over it.  part, ticket: device [kSellHotBlocks] and [ticket_words(kSellHotBlocks)].
int sell_push(const SellRows &sr, const float *push, float *diff, int *active, double *part, unsigned int *ticket, const StoreStat &stat,
              hipStream_t stream);
void sell_destroy(SellRows *sr);
// The two kinds of launch of a run: sell_begin reads the caller's inverse out-degrees, makes the first gather source and
// its dangling mass; sell_iterate is one iteration (it = 0, 1, ...), the last of which passes rank_out.
int sell_begin(const SellRows &sr, const double *inv_user, hipStream_t stream);
int sell_iterate(const SellRows &sr, int it, double alpha, double *rank_out, hipStream_t stream);
// A whole run of iters >= 1 in one launch, where sr.resident is not 0.  Worth it from sr.resident_iters on: entering costs what two launches
// do (4 K vertices and 53 K entries, us for 1, 2, 3 and 20 iterations: 9.3, 11.9, 13.7, 48 instead of 7.2, 11.8, 16.6, 86).  Plans of more than
// 10 K rows stage 12 slots a lane, whose registers ask for an empty CU, and such a CU comes late on a busy chip: 12,000 vertices and 108 K entries alone
// 27, 33, 42, 48, 53 us for 3, 5, 8, 10, 12 iterations instead of 27, 35, 49-68, 56-72, 64-75, beside a stream that adds to 1 GiB of floats 178 for any
// of them instead of 75, 106, 150, 175, 193: from 8 on an idle chip gains more than a busy one loses (10,000 vertices and 200 K entries, which find
// their places, 62, 73, 88 for 3, 5, 8 instead of 81, 109, 155).
constexpr int kSellResidentIters = 3, kSellResidentItersEmptyCu = 8;
int sell_run(const SellRows &sr, const double *inv_user, int iters, double alpha, double *rank_out, hipStream_t stream);

}  // namespace drone
