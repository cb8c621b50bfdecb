// One-launch-per-iteration fp64 PageRank: see pr_sell.h.
#include "pr_sell.h"

#include <algorithm>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

namespace drone {
namespace {

// Up to here (rows + entries) the layout beats the row blocks: at 8.5 M items 37.0 (41.3 without sources in LDS) against 43.8 us
// per iteration, at 17 M (8 MB of gather source, twice an XCD's L2) 73.7 against the 63.8 of the row blocks' sorted gathers.
constexpr int64_t kSellMaxItems = 9 << 20;
// Work-groups of 256 / 512 / 1,024 lanes, us per iteration at 0.012 / 0.057 / 1.02 / 2.07 / 4.2 / 8.5 M items: 4.05 / 4.7 /
// 9.1 / 14.6 / 24.2 / 51.5, 4.2 / 5.1 / 9.6 / 14.1 / 24.3 / 41.3, 5.3 / 6.3 / 12.2 / 14.5 / 21.1 / 43.4: small ones for small
// matrices (more CUs at work), 512 once the partials of so many work-groups and the hub rows count.
constexpr int64_t kSellWideItems = 1200 << 10;
constexpr int kSellInitThreads = 256, kSellInitBlocks = 512;
// From kSellWideItems on the hottest sources sit in LDS, if that many of the entries name one of them (of kSellSamples looked
// at): us per iteration without / with, and the share, 2.0 M items (131,072 vertices) 14.1 / 11.8 at 0.89, 4.2 M 24.2 / 18.1 at 0.79,
// 8.5 M 41.3 / 37.0 at 0.71, 1 M vertices and 7.8 M entries 45.3 / 38.2 at 0.63; half as many sources in LDS 41.3 / 44.0 at 0.57,
// 45.3 / 45.8 at 0.50.  Bringing 160 KB into every CU's LDS takes 3 us whatever there is to do: 1.0 M items 9.0 / 9.6.
constexpr double kSellHotShare = 0.6;
// Float rows from here on: see ensure_sell_rows in pr_push.hip for both sides.
constexpr int64_t kSellF32Items = 4 << 20;
constexpr int kSellSamples = 1 << 16;
constexpr size_t kSellHotLds = sizeof(double) * kSellHot;
static_assert(kSellInitBlocks <= kSellHotThreads && kSellHotBlocks <= kSellHotThreads, "a partial per lane");
static_assert(sizeof(float) * kSellHotF32 == kSellHotLds, "the same LDS");
// Whole runs in one launch of up to kSellResidentBlocks work-groups, kSellResidentSlices slices to each as long as there are no more: a
// wavefront per SIMD gathers, and the fewer work-groups read every source the better (1 K vertices, 12 K entries, us per iteration with 1, 2, 4
// and 8 slices a work-group 1.45, 1.31, 1.26, 1.33; up to 128 work-groups at 8 K vertices 2.6 instead of 2.4).
constexpr int kSellResidentBlocks = 64, kSellResidentSlices = 4, kSellStaged = 12;
constexpr size_t kSellResidentLds = 152 << 10;  // of 160; the kernel's own arrays are 1
constexpr int kSellMassLoads = 4;  // partials of the dangling mass per lane that are requested ahead

// What a kernel needs of SellRows, by value.
struct SellShape {
    int n, hubs, slices;
    int row_begin[kSellClasses + 1], slice_begin[kSellClasses + 1];
};

// Class of a row of `len` entries: the smallest P with at most kSellDepth (kSellDepthF32) entries per lane; class k has P = 64 >> k.
__host__ __device__ inline int sell_class_limit(int k, bool f32, int hub_limit)  // longest row of class k
{
    return k == 0 ? hub_limit : (64 >> k) * (f32 ? kSellDepthF32 : kSellDepth);
}

__device__ __forceinline__ double wave_sum(double v)  // valid in every lane
{
#pragma unroll
    for (int m = kWave / 2; m > 0; m >>= 1) v += __shfl_xor(v, m, kWave);
    return v;
}

template <int T>
__device__ __forceinline__ double block_sum(double v, double *s_red)  // valid in every thread
{
    v = wave_sum(v);
    if ((threadIdx.x & (kWave - 1)) == 0) s_red[threadIdx.x / kWave] = v;
    __syncthreads();
    double t = 0.0;
#pragma unroll
    for (int w = 0; w < T / kWave; ++w) t += s_red[w];
    return t;
}

// inv = the caller's inverse out-degrees in row order, c0 = inv / n, dangling mass of the uniform ranks per work-group.
__global__ __launch_bounds__(kSellInitThreads) void sell_begin_kernel(int n, const int32_t *__restrict__ order,
                                                                      const double *__restrict__ inv_user, double inv_n,
                                                                      double *__restrict__ inv, double *__restrict__ c0,
                                                                      double *__restrict__ c1, double *__restrict__ part)
{
    __shared__ double s_red[kSellInitThreads / kWave];
    double stat = 0.0;
    for (int i = blockIdx.x * kSellInitThreads + threadIdx.x; i < n; i += gridDim.x * kSellInitThreads) {
        const double iv = inv_user[order[i]];
        inv[i] = iv;
        c0[i] = iv * inv_n;
        if (iv == 0.0) stat += inv_n;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) c0[n] = c1[n] = 0.0;  // what the padding gathers
    const double total = block_sum<kSellInitThreads>(stat, s_red);
    if (threadIdx.x == 0) part[blockIdx.x] = total;
}

// Sum of c_in over `steps` consecutive steps of T ids starting at `ids` (this lane's), D gathers in flight.
template <int T, int D>
__device__ __forceinline__ double sell_sum(const int32_t *__restrict__ ids, int steps, const double *__restrict__ c_in, int pad)
{
    double sum = 0.0;
    for (int s = 0; s < steps; s += D) {
        int id[D];
        double v[D];
#pragma unroll
        for (int k = 0; k < D; ++k) id[k] = s + k < steps ? ids[(size_t)(s + k) * T] : pad;  // uniform condition
#pragma unroll
        for (int k = 0; k < D; ++k) v[k] = s + k < steps ? c_in[id[k]] : 0.0;
#pragma unroll
        for (int k = 0; k < D; ++k) sum += v[k];
    }
    return sum;
}

// One iteration.  Work-groups [0, hubs) take a hub row each, the others T / 64 slices each.
template <int T>
__global__ __launch_bounds__(T) void sell_iterate_kernel(int n, int hubs, int slices, const int32_t *__restrict__ hub_step,
                                                         const int32_t *__restrict__ hub_col,
                                                         const int4 *__restrict__ slice,
                                                         const int32_t *__restrict__ col, const double *__restrict__ c_in,
                                                         const double *__restrict__ inv, double *__restrict__ c_out,
                                                         const double *__restrict__ part_in, int parts,
                                                         double *__restrict__ part_out, double alpha, double inv_n,
                                                         const int32_t *__restrict__ order, double *__restrict__ r_out)
{
    __shared__ double s_dang[T / kWave], s_hub[T / kWave], s_red[T / kWave];
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    // The partials are requested first and added up last: they travel beside the entries.
    double mass[kSellMassLoads];
#pragma unroll
    for (int k = 0; k < kSellMassLoads; ++k) mass[k] = part_in[tid + k * T < parts ? tid + k * T : 0];
    int row = -1;
    double sum = 0.0, iv = 0.0;
    if ((int)blockIdx.x < hubs) {
        const int s0 = hub_step[blockIdx.x], s1 = hub_step[blockIdx.x + 1];
        if (tid == 0) {
            row = blockIdx.x;
            iv = inv[row];
        }
        sum = sell_sum<T, kSellHubDepth>(hub_col + (size_t)s0 * T + tid, s1 - s0, c_in, n);
        sum = wave_sum(sum);
        if (lane == 0) s_hub[wave] = sum;
    } else {
        const int s = __builtin_amdgcn_readfirstlane(((int)blockIdx.x - hubs) * (T / kWave) + wave);
        if (s < slices) {  // the same for the whole wavefront
            const int4 d = slice[s];  // {first step, steps, first row, rows << 3 | log2(lanes per row)}
            const int lanes_log = d.w & 7, lanes = 1 << lanes_log, r = lane >> lanes_log;
            if ((lane & (lanes - 1)) == 0 && r < (d.w >> 3)) {
                row = d.z + r;
                iv = inv[row];
            }
            sum = sell_sum<kWave, kSellDepth>(col + (size_t)d.x * kWave + lane, d.y, c_in, n);
            for (int m = lanes >> 1; m > 0; m >>= 1) sum += __shfl_xor(sum, m, kWave);
        }
    }
    double all = 0.0;
#pragma unroll
    for (int k = 0; k < kSellMassLoads; ++k) all += tid + k * T < parts ? mass[k] : 0.0;
    for (int i = tid + kSellMassLoads * T; i < parts; i += T) all += part_in[i];
    const double dang = block_sum<T>(all, s_dang);  // its barrier is s_hub's too
    if ((int)blockIdx.x < hubs) {
        sum = 0.0;
#pragma unroll
        for (int w = 0; w < T / kWave; ++w) sum += s_hub[w];
    }
    double stat = 0.0;
    if (row >= 0) {
        const double rn = (1.0 - alpha) * inv_n + alpha * dang * inv_n + alpha * sum;
        c_out[row] = rn * iv;
        if (r_out) r_out[order[row]] = rn;
        if (iv == 0.0) stat = rn;
    }
    const double total = block_sum<T>(stat, s_red);
    if (tid == 0) part_out[blockIdx.x] = total;
}

// ---- whole runs in one launch -----------------------------------------------------------------------------------------
// Runs of a launch per iteration wait for launches: 2.3 us each, and then a chain of descriptor, ids and gathers out of a cold cache (4.1 us
// per iteration at 500 vertices as at 4 K).  What is left here is one trip of a value to memory and back (1.2 us for 1 K values between
// any number of work-groups, 1.4 for 4 K), bringing the sources into LDS at 30 bytes a cycle, and the chains of gathers and lane
// sums in between.  20 iterations, us, a launch per iteration / this: 500 vertices and 2 K entries 69 / 32, 4 K and 53 K 86 / 48, 6 K and
// 43 K 86 / 50, 12 K and 115 K 98 / 69, 12 K and 343 K 102 / 80.  More slices than wavefronts lose: 8 K and 595 K 102 / 139, 12 K and 622 K
// 119 / 170; so do more hub rows than work-groups (4 K and 464 K, 3 iterations 16.9 / 19.8, 20 96.7 / 93.5).  All 1,024 lanes bring sources
// in, the slots' loads and the LDS writes without a bounds check (with one 2.05 -> 2.4 us per iteration); work-groups of 256 or 512
// lanes take longer from 2 K vertices on (4 K 2.9 and 2.3 instead of 2.0).
//
// Small matrices: the work-groups stay for the whole run, with the entries of their rows in registers and all sources in LDS, and
// hand each other the new sources through memory.  A source is its own flag: a slot that holds kSellNone (a NaN that no sum makes)
// is not written yet, so a value that is there is the value, and no order between different slots is needed to read it.  Slots are
// 8-byte relaxed atomics at agent scope, which every XCD reads and writes at the same place.
//
// Four sets of slots.  Iteration `it` reads set it, writes set it + 1, and its owners clear set it - 1 (indexes modulo 4): whoever
// holds all of set it knows that every work-group, each of which owns a row, has finished reading set it - 1.  Set it - 1 is written
// again two iterations on and looked at three on; the owner waits for its clearing store (which writes through) before it publishes
// again, and who looks at the set has read what it published then.  The last work-group to leave clears the last set, and the counters.
//
// The work-groups wait for each other, so all that take part must have a place on the chip before any starts.  Each reports at a gate; one
// that has looked in vain for long enough closes it, those who have come by then do the run, and later ones go; every sum has the same order
// then.  (Behind the gate all are on the chip, and every wait ends.  kSellPolls is seconds; a lane that has waited for so long says so and goes
// on with the NaN.  The last work-group to leave then clears every set, and the plan's next run reports it instead of running.)
// Long enough: `patience` looks where who is there takes no more rounds of slices and hub rows than all would; else also as many as the run
// would take with them, at kSellLooksPerRound a round (1.2 us on an idle chip, four times that beside a stream of memory-bound kernels), so
// that the wait at most doubles it.  20 iterations beside a stream that adds to 1 GiB of floats, us, a launch per iteration / one
// work-group behind every closed gate / this: 4 K vertices and 53 K entries 289 / 111 / 119 (three 67 / 45 / 51), 12 K and 108 K 313 / 3,300 / 177, 12 K and
// 240 K 323 / - / 220-237, 12 K and 344 K 363 / - / 270, 12 K and 419 K 381 / 12,700 / 250-315; beside bf16 products of 8,192 rows, whose work-groups fill the
// chip for 0.7 ms each, 16,000 / 80-5,300 / 780.  What the runs of more than 10 K rows wait for are the places: 124 registers a lane ask for an
// empty CU (with 96, at the price of 27 spilled, 71 / 80 for three iterations, but 20 of an idle chip 78 -> 104 and 91 -> 132), so their short runs
// are a launch per iteration (kSellResidentItersEmptyCu).
constexpr int kSellResidentThreads = 1024;
constexpr unsigned long long kSellNone = 0x7ffc5e1100a1b2c3ull, kSellNan = 0x7ff8000000000000ull;
// The gate: who has come, and once it is closed how many of them do the run.
constexpr unsigned kSellClosed = 1u << 31, kSellCame = 0xff;
constexpr int kSellRunShift = 8, kSellLooksPerRound = 2, kSellMostLooks = 1 << 22;
static_assert(kSellResidentBlocks <= (int)kSellCame, "a byte each");
constexpr int kSellPolls = 1 << 22;
constexpr unsigned kSellGaveUp = 1u << 16;  // times those who gave up, beside the count of those who have left
constexpr int kSellWaitStores = 0x0f70;  // s_waitcnt vmcnt(0)

__device__ __forceinline__ void slot_store(unsigned long long *p, unsigned long long v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ unsigned long long slot_load(const unsigned long long *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

__device__ __forceinline__ bool slot_is_none(unsigned long long v) { return (unsigned)(v >> 32) == (unsigned)(kSellNone >> 32); }

// Four sets of `slots` slots of which `used` are, the gate, and behind its counters where the last work-group reports.
__global__ void sell_slots_kernel(int slots, int used, unsigned long long *__restrict__ exchange, unsigned *__restrict__ gate, int *failed)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < 4 * slots; i += gridDim.x * blockDim.x)
        exchange[i] = i % slots < used ? kSellNone : 0;
    if (blockIdx.x == 0 && threadIdx.x < 2 * kTicketStride) gate[threadIdx.x] = 0;
    if (blockIdx.x == 0 && threadIdx.x == 0) *reinterpret_cast<int **>(gate + 2 * kTicketStride) = failed;
}

// Through the gate: this work-group's number in the run and, from kSellRunShift on, how many do it, or -1 to leave.  ticket: the gate when
// it came.
__device__ __forceinline__ int sell_enter(unsigned *gate, unsigned ticket, const SellGate &rule)
{
    const int mine = (int)(ticket & kSellCame);
    unsigned seen = ticket + 1;
    for (int looks = -rule.patience;; ++looks) {
        if (seen & kSellClosed) {
            const int groups = (int)(seen >> kSellRunShift & kSellCame);
            return mine < groups ? mine | groups << kSellRunShift : -1;
        }
        const int came = (int)seen;
        if (came >= (int)gridDim.x && rule.places >= came) return mine | came << kSellRunShift;
        if (came >= rule.places || (looks >= 0 && (came >= rule.enough || looks * came >= rule.price))) {
            const unsigned closed = seen | kSellClosed | (unsigned)min(came, rule.places) << kSellRunShift;
            if (__hip_atomic_compare_exchange_strong(gate, &seen, closed, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) seen = closed;
        } else seen = __hip_atomic_load(gate, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

template <int Ctrl>
__device__ __forceinline__ double dpp_add(double v)
{
    const long long bits = __double_as_longlong(v);
    const unsigned lo = __builtin_amdgcn_update_dpp(0u, (unsigned)bits, Ctrl, 0xf, 0xf, true);
    const unsigned hi = __builtin_amdgcn_update_dpp(0u, (unsigned)(bits >> 32), Ctrl, 0xf, 0xf, true);
    return v + __longlong_as_double((long long)((unsigned long long)hi << 32 | lo));
}

template <int Lanes>
__device__ __forceinline__ double swap_add(double v)
{
    const long long bits = __double_as_longlong(v);
    const unsigned lo = (unsigned)bits, hi = (unsigned)(bits >> 32);
    const auto l = Lanes == 16 ? __builtin_amdgcn_permlane16_swap(lo, lo, false, false) : __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
    const auto h = Lanes == 16 ? __builtin_amdgcn_permlane16_swap(hi, hi, false, false) : __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
    const auto value = [](unsigned a, unsigned b) { return __longlong_as_double((long long)((unsigned long long)b << 32 | a)); };
    return value(l[0], h[0]) + value(l[1], h[1]);
}

// Sum over neighbouring `lanes` lanes (a power of two, the same for the whole wavefront), valid in each of them.  Without the LDS
// crossbar, whose six round trips would be a third of an iteration's work.
__device__ __forceinline__ double lanes_sum(double v, int lanes)
{
    if (lanes > 1) v = dpp_add<0xb1>(v);    // quad_perm 1 0 3 2
    if (lanes > 2) v = dpp_add<0x4e>(v);    // quad_perm 2 3 0 1
    if (lanes > 4) v = dpp_add<0x141>(v);   // row_half_mirror: the quads are even by now
    if (lanes > 8) v = dpp_add<0x140>(v);   // row_mirror
    if (lanes > 16) v = swap_add<16>(v);
    if (lanes > 32) v = swap_add<32>(v);
    return v;
}

// Rows [0, live) have entries.  The others' rank is the iteration's constant term, so nobody has to be told: every work-group makes
// their sources for itself.  A set has a slot per live row and is zeros up to S = K * T, of which a lane brings K into LDS.
template <int K>
__global__ __launch_bounds__(kSellResidentThreads) void sell_resident_kernel(
    int n, int live, int hubs, int slices, int hub_width, const int32_t *__restrict__ hub_step, const int32_t *__restrict__ hub_col,
    const int4 *__restrict__ slice, const int32_t *__restrict__ col, const int32_t *__restrict__ order,
    const double *__restrict__ inv_user, double *inv, unsigned long long *exchange, unsigned *gate, SellGate rule, int iters,
    double alpha, double inv_n, double *__restrict__ r_out)
{
    constexpr int T = kSellResidentThreads, S = K * T, D = kSellWaveSteps, kHubAhead = 4, kRest = 4;
    extern __shared__ __attribute__((aligned(16))) double s_c[];  // sources [S], of the rows without entries [n - live], 0; those rows' inverse out-degrees [n - live]
    __shared__ double s_mass[T / kWave], s_hub[T / kWave];
    __shared__ int s_group, s_last, s_dangling;
    __shared__ unsigned s_gave_up;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int rest = n - live;
    unsigned *left = gate + kTicketStride;
    double *s_rest = s_c + S + rest + 1;
    unsigned ticket = 0;
    if (tid == 0) {
        ticket = __hip_atomic_fetch_add(gate, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_dangling = 0;
    }
    __syncthreads();
    // The uniform ranks' sources, which every work-group makes for itself, and the inverse out-degrees that go with this lane's slots.
    int dangling = 0;
    unsigned dangles = 0;
    double ivs[K];
    {
        int vertex[K];
#pragma unroll
        for (int k = 0; k < K; ++k) vertex[k] = order[min(tid + k * T, n - 1)];
#pragma unroll
        for (int k = 0; k < K; ++k) ivs[k] = inv_user[vertex[k]];
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const bool there = tid + k * T < live;
        s_c[tid + k * T] = ivs[k] * inv_n;
        dangles |= (there && ivs[k] == 0.0) << k;
        if (!there) ivs[k] = 0.0;
    }
    dangling = __builtin_popcount(dangles);
    for (int i = tid; i < rest; i += kRest * T) {
        int vertex[kRest];
        double iv[kRest];
#pragma unroll
        for (int k = 0; k < kRest; ++k) vertex[k] = order[min(live + i + k * T, n - 1)];
#pragma unroll
        for (int k = 0; k < kRest; ++k) iv[k] = inv_user[vertex[k]];
#pragma unroll
        for (int k = 0; k < kRest; ++k)
            if (i + k * T < rest) {
                s_c[S + i + k * T] = iv[k] * inv_n;
                s_rest[i + k * T] = iv[k];
                dangling += iv[k] == 0.0;
            }
    }
    if (tid == 0) {
        s_c[S + rest] = 0.0;  // what the padding gathers
        s_group = sell_enter(gate, ticket, rule);
        s_last = 0;
        s_gave_up = 0;
    }
    if (dangling) atomicAdd(&s_dangling, dangling);
    __syncthreads();
    const int group = __builtin_amdgcn_readfirstlane(s_group < 0 ? -1 : s_group & (int)kSellCame);
    const int groups = __builtin_amdgcn_readfirstlane(s_group >> kSellRunShift);
    const auto leave = [&] {  // thread 0, when the work-group reads no slots any more
        const unsigned mine = 1 + s_gave_up, before = __hip_atomic_fetch_add(left, mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), all = before + mine;
        s_last = (all & (kSellGaveUp - 1)) != gridDim.x ? 0 : all < kSellGaveUp ? 1 : 4;  // sets to clear
    };
    const auto close = [&] {
        if (!s_last) return;
        if (iters > 1)
            for (int set = 0; set < s_last; ++set)
                for (int i = tid; i < live; i += T) slot_store(exchange + (size_t)((iters - 1 + set) & 3) * S + i, kSellNone);
        if (tid == 0) {
            if (s_last > 1) __hip_atomic_store(*reinterpret_cast<int **>(gate + 2 * kTicketStride), 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            __hip_atomic_store(gate, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(left, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    };
    if (group < 0) {
        if (tid == 0) leave();
        __syncthreads();
        close();
        return;
    }
    const int stride = groups * (T / kWave), first = group + groups * wave;
    const bool more = slices > stride || hubs > groups, hub = group < hubs;
    const auto place = [&](bool there, int row) { return !there ? S + rest : row < live ? row : row + (S - live); };  // in LDS
    const auto row_of = [&](const int4 &d) {
        const int lanes_log = d.w & 7, r = lane >> lanes_log;
        return (lane & ((1 << lanes_log) - 1)) == 0 && r < (d.w >> 3) && d.z + r < live ? d.z + r : -1;
    };
    // The first slice of the wavefront and the first hub of the work-group stay in registers.
    const int4 d0 = first < slices ? slice[first] : make_int4(0, 0, 0, 0);
    int id[D], hub_id[kHubAhead];
#pragma unroll
    for (int k = 0; k < D; ++k) id[k] = col[((size_t)d0.x + k) * kWave + lane];  // (the array goes on for D steps)
#pragma unroll
    for (int k = 0; k < D; ++k) id[k] = place(k < d0.y, id[k]);
    const int row0 = row_of(d0);
    const double iv0 = row0 >= 0 ? inv_user[order[row0]] : 1.0;
    // Steps of a hub taken at once, this lane's share of them.
    const int hub_lanes = T / hub_width, hub_sub = __builtin_amdgcn_readfirstlane(tid / hub_width), hub_lane = tid % hub_width;
    const auto hub_fetch = [&](int from, int to, int (&ids)[kHubAhead]) {
#pragma unroll
        for (int k = 0; k < kHubAhead; ++k) ids[k] = hub_col[(size_t)min(from + hub_sub + k * hub_lanes, to - 1) * hub_width + hub_lane];
#pragma unroll
        for (int k = 0; k < kHubAhead; ++k) ids[k] = place(from + hub_sub + k * hub_lanes < to, ids[k]);
    };
    int hub_from = 0, hub_to = 0;
    double hub_iv = 0.0;
    if (hub) {
        hub_from = hub_step[group];
        hub_to = hub_step[group + 1];
        hub_iv = inv_user[order[group]];
        hub_fetch(hub_from, hub_to, hub_id);
    }
    const double dangling_rows = s_dangling;
    for (int s = first + stride; s < slices; s += stride) {
        const int row = row_of(slice[s]);
        if (row >= 0) inv[row] = inv_user[order[row]];  // read again by this lane only
    }
    // A rank is base + alpha * sum, and base is the same everywhere: a slot holds alpha * sum, times the
    // inverse out-degree where that is not 0, and base, which takes a reduction, is added by the readers and not waited for.
    bool given_up = rule.patience < 0;
    if (given_up) s_gave_up = kSellGaveUp;
    double base = inv_n, mass = 0.0;  // of the ranks that the iteration starts from: base, and the dangling mass beyond base
    for (int it = 0; it < iters; ++it) {
        unsigned long long *out = exchange + (size_t)((it + 1) & 3) * S, *done = exchange + (size_t)((it + 3) & 3) * S;
        const bool last = it == iters - 1;
        if (it > 0) {
            const unsigned long long *in = exchange + (size_t)(it & 3) * S + tid;
            unsigned long long v[K];
#pragma unroll
            for (int k = 0; k < K; ++k) v[k] = slot_load(in + k * T);
            for (int i = tid; i < rest; i += T) s_c[S + i] = base * s_rest[i];
            for (int polls = 0; !given_up; ++polls) {
                bool missing = false;
#pragma unroll
                for (int k = 0; k < K; ++k) missing |= slot_is_none(v[k]);
                if (!missing) break;
                given_up = polls >= kSellPolls;
                if (given_up) s_gave_up = kSellGaveUp;
#pragma unroll
                for (int k = 0; k < K; ++k)
                    if (slot_is_none(v[k])) v[k] = slot_load(in + k * T);
            }
            mass = 0.0;
#pragma unroll
            for (int k = 0; k < K; ++k) {
                double x = __longlong_as_double((long long)v[k]);
                if (dangles >> k & 1) {
                    mass += x;
                    x *= 0.0;
                }
                s_c[tid + k * T] = x + base * ivs[k];
            }
            __builtin_amdgcn_s_waitcnt(kSellWaitStores);  // for the clearing stores of the iteration before
        }
        __syncthreads();
        if (last && tid == 0) leave();
        double sum = 0.0, part = 0.0;
        const auto gather = [&](auto steps) {
            double v[decltype(steps)::value];
#pragma unroll
            for (int k = 0; k < decltype(steps)::value; ++k) v[k] = s_c[id[k]];
#pragma unroll
            for (int k = 0; k < decltype(steps)::value; ++k) sum += v[k];
        };
        const auto hub_sum = [&](int from, int to, const int (&ahead)[kHubAhead]) {
            int ids[kHubAhead];
            double total = 0.0;
#pragma unroll
            for (int k = 0; k < kHubAhead; ++k) ids[k] = ahead[k];
            for (;;) {
#pragma unroll
                for (int k = 0; k < kHubAhead; ++k)
                    total += s_c[ids[k]];
                from += kHubAhead * hub_lanes;
                if (from >= to) return total;
                hub_fetch(from, to, ids);
            }
        };
        // A row's slots: filled for the next iteration, cleared of the one before.
        const auto hand_on = [&](int row, double iv, double total) {
            if (!last) {
                const unsigned long long bits = (unsigned long long)__double_as_longlong(iv == 0.0 ? alpha * total : alpha * total * iv);
                slot_store(out + row, slot_is_none(bits) ? kSellNan : bits);
            }
            if (it > 0) slot_store(done + row, kSellNone);
        };
        if (hub) {
            part = lanes_sum(hub_sum(hub_from, hub_to, hub_id), kWave);
            if (lane == 0) s_hub[wave] = part;
        }
        if (d0.y > 8) gather(std::integral_constant<int, D>());
        else if (d0.y > 4) gather(std::integral_constant<int, 8>());
        else if (d0.y > 0) gather(std::integral_constant<int, 4>());
        if (first < slices) {
            sum = lanes_sum(sum, 1 << (d0.w & 7));
            if (row0 >= 0) hand_on(row0, iv0, sum);
        }
        if (hub) {
            __syncthreads();
            if (wave == 0) {
                part = lanes_sum(s_hub[lane & (T / kWave - 1)], T / kWave);
                if (lane == 0) hand_on(group, hub_iv, part);
            }
        }
        // The constant term of this iteration's ranks.  Behind the barrier the sources in LDS may be replaced.
        mass = lanes_sum(mass, kWave);
        if (lane == 0) s_mass[wave] = mass;
        __syncthreads();
        const double dang = dangling_rows * base + lanes_sum(s_mass[lane & (T / kWave - 1)], T / kWave);
        base = (1.0 - alpha) * inv_n + alpha * dang * inv_n;
        const auto store = [&](int row, double total) {
            if (last) r_out[order[row]] = base + alpha * total;
        };
        if (row0 >= 0) store(row0, sum);
        if (hub && tid == 0) store(group, part);
        if (more) {
            for (int h = group + groups; h < hubs; h += groups) {
                int ids[kHubAhead];
                hub_fetch(hub_step[h], hub_step[h + 1], ids);
                const double wave_part = lanes_sum(hub_sum(hub_step[h], hub_step[h + 1], ids), kWave);
                if (lane == 0) s_hub[wave] = wave_part;
                __syncthreads();
                const double total = lanes_sum(s_hub[lane & (T / kWave - 1)], T / kWave);
                if (tid == 0) {
                    hand_on(h, inv_user[order[h]], total);
                    store(h, total);
                }
                __syncthreads();  // s_hub is used again
            }
            for (int s = first + stride; s < slices; s += stride) {
                const int4 d = slice[s];
                const int row = row_of(d);
                const double iv = row >= 0 ? inv[row] : 1.0;
                double total = 0.0;
                for (int step = 0; step < d.y; step += kSellDepth) {
                    int ids[kSellDepth];
#pragma unroll
                    for (int k = 0; k < kSellDepth; ++k) ids[k] = step + k < d.y ? place(true, col[((size_t)d.x + step + k) * kWave + lane]) : S + rest;
#pragma unroll
                    for (int k = 0; k < kSellDepth; ++k) total += s_c[ids[k]];
                }
                total = lanes_sum(total, 1 << (d.w & 7));
                if (row >= 0) {
                    hand_on(row, iv, total);
                    store(row, total);
                }
            }
            __syncthreads();  // the sources in LDS and s_hub are replaced next
        }
    }
    for (int i = live + group * T + tid; i < n; i += groups * T) r_out[order[i]] = base;
    __syncthreads();
    close();
}

// v[k] = source of id[k], the padding's 0.  Both kinds of load are under the lanes' own condition: a hot lane costs the L1 nothing.
template <int HOT, int D, typename V>
__device__ __forceinline__ void sell_hot_gather(const int (&id)[D], const V *s_hot, const V *__restrict__ c_in, V (&v)[D])
{
#pragma unroll
    for (int k = 0; k < D; ++k) {
        v[k] = V(0);
        if (id[k] > HOT) v[k] = c_in[id[k] - 1];
    }
#pragma unroll
    for (int k = 0; k < D; ++k)
        if (id[k] < HOT) v[k] = s_hot[id[k]];
}

// Calls add(value) for the sources of steps [s, steps) of T ids from `ids` on (this lane's).
template <int T, int HOT, int D, typename V, typename Add>
__device__ __forceinline__ void sell_hot_each(int s, int steps, const int32_t *__restrict__ ids, const V *s_hot, const V *__restrict__ c_in, Add add)
{
    for (; s < steps; s += D) {
        int id[D];
        V v[D];
#pragma unroll
        for (int k = 0; k < D; ++k) id[k] = s + k < steps ? ids[(size_t)(s + k) * T] : HOT;
        sell_hot_gather<HOT>(id, s_hot, c_in, v);
#pragma unroll
        for (int k = 0; k < D; ++k) add(v[k]);
    }
}

// The first D steps of a slice.
template <int HOT, int D>
__device__ __forceinline__ void sell_hot_fetch(const int4 &slice, const int32_t *__restrict__ col, int lane, int (&id)[D])
{
#pragma unroll
    for (int k = 0; k < D; ++k) id[k] = k < slice.y ? col[((size_t)slice.x + k) * kWave + lane] : HOT;
}

// s_hot[i] = c_in[i] for the first HOT of n sources, in pieces of 16 bytes.  Every CU of an XCD starts at another piece: otherwise they
// would all ask one L2 channel for the same line (2 M items 13.3 -> 11.9 us).
template <int HOT, typename V>
__device__ __forceinline__ void sell_hot_stage(int n, const V *__restrict__ c_in, V *s_hot)
{
    constexpr int W = 16 / sizeof(V), T = kSellHotThreads, kPieces = (HOT / W + T - 1) / T;
    static_assert(HOT % W == 0, "whole pieces");
    const int hot = n < HOT ? n : HOT, rot = ((int)blockIdx.x / 8) % kPieces;
#pragma unroll
    for (int k = 0; k < kPieces; ++k) {
        const int i = ((int)threadIdx.x + (k + rot < kPieces ? k + rot : k + rot - kPieces) * T) * W;
        if (i + W <= hot) *reinterpret_cast<float4 *>(s_hot + i) = *reinterpret_cast<const float4 *>(c_in + i);
        else
            for (int j = i; j < hot; ++j) s_hot[j] = c_in[j];
    }
}

// One iteration with the hottest sources in LDS; one work-group per CU, the slices dealt out to the wavefronts of all.
__global__ __launch_bounds__(kSellHotThreads) void sell_iterate_hot_kernel(
    int n, int hubs, int slices, const int32_t *__restrict__ hub_step, const int32_t *__restrict__ hub_col,
    const int4 *__restrict__ slice, const int32_t *__restrict__ col, const double *__restrict__ c_in,
    const double *__restrict__ inv, double *__restrict__ c_out, const double *__restrict__ part_in, int parts,
    double *__restrict__ part_out, double alpha, double inv_n, const int32_t *__restrict__ order, double *__restrict__ r_out)
{
    constexpr int T = kSellHotThreads;
    extern __shared__ __attribute__((aligned(16))) double s_hot[];  // [kSellHot], filled in pieces of 16 bytes
    __shared__ double s_dang[T / kWave], s_red[T / kWave];
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int stride = (int)gridDim.x * (T / kWave);
    // The first slice's ids, and the dangling mass, travel beside the hot sources.
    int s = (int)blockIdx.x + (int)gridDim.x * wave;
    const auto descriptor = [&](int at) { return at < slices ? slice[at] : make_int4(0, 0, 0, 0); };
    int4 d = descriptor(s), after = descriptor(s + stride);
    int id[kSellDepth];
    sell_hot_fetch<kSellHot>(d, col, lane, id);
    const double mass = tid < parts ? part_in[tid] : 0.0;
    sell_hot_stage<kSellHot>(n, c_in, s_hot);
    const double dang = block_sum<T>(mass, s_dang);
    const double base = (1.0 - alpha) * inv_n + alpha * dang * inv_n;
    double stat = 0.0;
    const auto finish = [&](int row, double iv, double sum) {
        const double rn = base + alpha * sum;
        c_out[row] = rn * iv;
        if (r_out) r_out[order[row]] = rn;
        if (iv == 0.0) stat += rn;
    };
    for (int h = blockIdx.x; h < hubs; h += gridDim.x) {
        const int s0 = hub_step[h], s1 = hub_step[h + 1];
        const double iv = inv[h];
        const int32_t *ids = hub_col + (size_t)s0 * T + tid;
        double sum = 0.0;
        sell_hot_each<T, kSellHot, kSellDepth>(0, s1 - s0, ids, s_hot, c_in, [&](double v) { sum += v; });
        sum = block_sum<T>(sum, s_red);
        if (tid == 0) finish(h, iv, sum);
        __syncthreads();  // s_red is used again
    }
    while (s < slices) {
        const int4 later = descriptor(s + 2 * stride);  // it takes a round trip before its ids can be asked for
        const int lanes_log = d.w & 7, lanes = 1 << lanes_log, r = lane >> lanes_log;
        const bool mine = (lane & (lanes - 1)) == 0 && r < (d.w >> 3);
        const double iv = mine ? inv[d.z + r] : 0.0;
        double sum = 0.0, v[kSellDepth];
        sell_hot_gather<kSellHot>(id, s_hot, c_in, v);
        sell_hot_fetch<kSellHot>(after, col, lane, id);
#pragma unroll
        for (int k = 0; k < kSellDepth; ++k) sum += v[k];
        sell_hot_each<kWave, kSellHot, kSellDepth>(kSellDepth, d.y, col + (size_t)d.x * kWave + lane, s_hot, c_in, [&](double x) { sum += x; });
        for (int m = lanes >> 1; m > 0; m >>= 1) sum += __shfl_xor(sum, m, kWave);
        if (mine) finish(d.z + r, iv, sum);
        d = after;
        after = later;
        s += stride;
    }
    const double total = block_sum<T>(stat, s_red);
    if (tid == 0) part_out[blockIdx.x] = total;
}

// diff[v] = sum of the pushes of v's row, active[v] = whether any is not 0; the number of active rows goes to `stat`.
__global__ __launch_bounds__(kSellHotThreads) void sell_push_kernel(int n, int hubs, int slices, const int32_t *__restrict__ hub_step,
                                                                    const int32_t *__restrict__ hub_col,
                                                                    const int4 *__restrict__ slice, const int32_t *__restrict__ col,
                                                                    const float *__restrict__ push, const int32_t *__restrict__ order,
                                                                    float *__restrict__ diff, int *__restrict__ active,
                                                                    double *part, unsigned int *ticket, StoreStat stat)
{
    constexpr int T = kSellHotThreads, H = kSellHotF32, D = kSellDepthF32;
    extern __shared__ __attribute__((aligned(16))) float s_push[];  // [kSellHotF32], filled in pieces of 16 bytes
    __shared__ double s_red[T / kWave];
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int stride = (int)gridDim.x * (T / kWave);
    int s = (int)blockIdx.x + (int)gridDim.x * wave;
    const auto descriptor = [&](int at) { return at < slices ? slice[at] : make_int4(0, 0, 0, 0); };
    int4 d = descriptor(s), after = descriptor(s + stride);
    int id[D];
    sell_hot_fetch<H>(d, col, lane, id);
    sell_hot_stage<H>(n, push, s_push);
    __syncthreads();
    int lowered = 0;
    const auto finish = [&](int v, float sum, bool any) {
        diff[v] = sum;
        active[v] = any;
        lowered += any;
    };
    for (int h = blockIdx.x; h < hubs; h += gridDim.x) {
        const int s0 = hub_step[h], s1 = hub_step[h + 1];
        const int32_t *ids = hub_col + (size_t)s0 * T + tid;
        float sum = 0.0f;
        bool any = false;
        sell_hot_each<T, H, D>(0, s1 - s0, ids, s_push, push, [&](float v) { sum += v; any |= v != 0.0f; });
        const bool some = __syncthreads_or(any);
        const double total = block_sum<T>((double)sum, s_red);
        if (tid == 0) finish(order[h], (float)total, some);
        __syncthreads();  // s_red is used again
    }
    while (s < slices) {
        const int4 later = descriptor(s + 2 * stride);
        const int lanes_log = d.w & 7, lanes = 1 << lanes_log, r = lane >> lanes_log;
        const int row = (lane & (lanes - 1)) == 0 && r < (d.w >> 3) ? order[d.z + r] : -1;
        float sum = 0.0f, v[D];
        bool any = false;
        const auto add = [&](float x) {
            sum += x;
            any |= x != 0.0f;
        };
        sell_hot_gather<H>(id, s_push, push, v);
        sell_hot_fetch<H>(after, col, lane, id);
#pragma unroll
        for (int k = 0; k < D; ++k) add(v[k]);
        sell_hot_each<kWave, H, D>(D, d.y, col + (size_t)d.x * kWave + lane, s_push, push, add);
        const unsigned long long some = __ballot(any);
        for (int m = lanes >> 1; m > 0; m >>= 1) sum += __shfl_xor(sum, m, kWave);
        if (row >= 0) finish(row, sum, ((some >> lane) & (lanes == kWave ? ~0ull : (1ull << lanes) - 1)) != 0);
        d = after;
        after = later;
        s += stride;
    }
    const double total = block_sum<T>((double)lowered, s_red);
    unsigned int one = 0;
    if (tid == 0) one = publish_part(part + blockIdx.x, total);
    if (!last_block_done(ticket, one)) return;
    const double all = block_sum<T>(tid < (int)gridDim.x ? load_agent(part + tid) : 0.0, s_red);
    if (tid == 0) stat(all);
}

// ---- building the layout ---------------------------------------------------------------------------------------------
template <typename Off>
__global__ void sell_lengths_kernel(int n, const Off *__restrict__ row_ptr, unsigned *__restrict__ len, int32_t *__restrict__ id)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        len[i] = (unsigned)(row_ptr[i + 1] - row_ptr[i]);
        id[i] = i;
    }
}

// new_id of every vertex; bounds[k] = rows (longest first) with more entries than class k takes, bounds[kSellClasses + 1] = rows with any
__global__ void sell_bounds_kernel(int n, const unsigned *__restrict__ len_sorted, const int32_t *__restrict__ order,
                                   bool f32, int hub_limit, int32_t *__restrict__ new_id, int *__restrict__ bounds)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) new_id[order[i]] = i;
    if (blockIdx.x != 0) return;
    if (threadIdx.x < kSellClasses || threadIdx.x == kSellClasses + 1) {
        const unsigned limit = threadIdx.x < kSellClasses ? (unsigned)sell_class_limit(threadIdx.x, f32, hub_limit) : 0;
        int lo = 0, hi = n;  // first row with at most `limit` entries
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (len_sorted[mid] > limit) lo = mid + 1; else hi = mid;
        }
        bounds[threadIdx.x] = lo;
    } else if (threadIdx.x == kSellClasses) {
        bounds[kSellClasses] = 0;  // for sell_sample_kernel
    }
}

// *named += entries, of kSellSamples from all over the matrix, whose source is one of the first `hot`
__global__ __launch_bounds__(256) void sell_sample_kernel(int64_t nnz, const int32_t *__restrict__ col, const int32_t *__restrict__ new_id,
                                                          int hot, int *__restrict__ named)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const unsigned long long names = __ballot(new_id[col[(int64_t)((double)i / kSellSamples * (double)nnz)]] < hot);
    if ((threadIdx.x & (kWave - 1)) == 0) atomicAdd(named, __popcll(names));
}

__device__ __forceinline__ void sell_slice_rows(const SellShape &sh, int s, int &k, int &first_row, int &last_row)
{
    k = 0;
    for (int q = 1; q < kSellClasses; ++q) k += s >= sh.slice_begin[q];
    first_row = sh.row_begin[k] + ((s - sh.slice_begin[k]) << k);
    last_row = sh.row_begin[k + 1];
}

// steps of every hub row and slice (the last element is the sentinel an exclusive scan turns into the total)
__global__ void sell_steps_kernel(SellShape sh, int threads, const unsigned *__restrict__ len_sorted,
                                  int32_t *__restrict__ hub_steps, int32_t *__restrict__ slice_steps)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i <= sh.hubs || i <= sh.slices; i += gridDim.x * blockDim.x) {
        if (i <= sh.hubs) hub_steps[i] = i < sh.hubs ? (int)((len_sorted[i] + threads - 1) / threads) : 0;
        if (i <= sh.slices) {
            int steps = 0;
            if (i < sh.slices) {
                int k, first_row, last_row;
                sell_slice_rows(sh, i, k, first_row, last_row);
                const unsigned lanes = 64u >> k;
                steps = (int)((len_sorted[first_row] + lanes - 1) / lanes);
            }
            slice_steps[i] = steps;
        }
    }
}

// The ids of every hub row and slice, one wavefront per slice and one work-group per hub row.
template <typename Off>
__global__ __launch_bounds__(256) void sell_fill_kernel(SellShape sh, int threads, const int32_t *__restrict__ order,
                                                        const Off *__restrict__ row_ptr, const int32_t *__restrict__ col,
                                                        const int32_t *__restrict__ new_id,
                                                        const int32_t *__restrict__ hub_step,
                                                        const int32_t *__restrict__ slice_step, int4 *__restrict__ slice,
                                                        int32_t *__restrict__ hub_out, int32_t *__restrict__ out, int hot)
{
    const auto source = [&](bool there, int64_t e) {
        if (!there) return hot ? hot : sh.n;
        const int id = new_id[col[e]];
        return id + (hot && id >= hot);
    };
    if ((int)blockIdx.x < sh.hubs) {
        const int64_t e0 = row_ptr[order[blockIdx.x]], e1 = row_ptr[order[blockIdx.x] + 1];
        const int64_t at = (int64_t)hub_step[blockIdx.x] * threads, count = (int64_t)hub_step[blockIdx.x + 1] * threads - at;
        for (int64_t i = threadIdx.x; i < count; i += 256) hub_out[at + i] = source(e0 + i < e1, e0 + i);
        return;
    }
    const int s = ((int)blockIdx.x - sh.hubs) * (256 / kWave) + threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
    if (s >= sh.slices) return;
    int k, first_row, last_row;
    sell_slice_rows(sh, s, k, first_row, last_row);
    const int lanes = 64 >> k, q = lane & (lanes - 1), r = first_row + (lane >> (6 - k));
    int64_t e0 = 0, e1 = 0;
    if (r < last_row) {
        e0 = row_ptr[order[r]] + q;
        e1 = row_ptr[order[r] + 1];
    }
    const int st0 = slice_step[s], st1 = slice_step[s + 1], rows = last_row - first_row < (1 << k) ? last_row - first_row : 1 << k;
    if (lane == 0) slice[s] = make_int4(st0, st1 - st0, first_row, rows << 3 | (6 - k));
    for (int st = st0; st < st1; ++st, e0 += lanes)
        out[(size_t)st * kWave + lane] = source(e0 < e1, e0);
}

using SellResident = decltype(&sell_resident_kernel<1>);

SellResident sell_resident_of(const SellRows &sr)
{
    switch (sr.staged) {
    case 1: return &sell_resident_kernel<1>;
    case 2: return &sell_resident_kernel<2>;
    case 3: return &sell_resident_kernel<3>;
    case 4: return &sell_resident_kernel<4>;
    case 5: return &sell_resident_kernel<5>;
    case 6: return &sell_resident_kernel<6>;
    case 8: return &sell_resident_kernel<8>;
    case 10: return &sell_resident_kernel<10>;
    default: return &sell_resident_kernel<kSellStaged>;
    }
}

// Whether runs are one launch, and of how many work-groups.
void choose_resident(SellRows *sr, int live)
{
    if (sr->n + sr->nnz > kSellWideItems) return;  // sell_resident_kernel keeps kSellWaveSteps steps of a slice; wide plans have longer ones
    sr->live = live;
    sr->live_slices = sr->slice_begin[kSellClasses - 1] + (int)ceil_div(live - sr->row_begin[kSellClasses - 1], kWave);
    sr->staged = 0;
    for (const int staged : {kSellStaged, 10, 8, 6, 5, 4, 3, 2, 1})
        if (staged * kSellResidentThreads >= live) sr->staged = staged;
    sr->lds = sizeof(double) * ((size_t)sr->staged * kSellResidentThreads + 2 * (size_t)(sr->n - live) + 1);
    if (!sr->staged || sr->lds > kSellResidentLds || sr->hubs > kSellResidentBlocks || sr->live_slices > kSellResidentBlocks * (kSellResidentThreads / kWave)) return;
    const int wanted = std::max((int)ceil_div(sr->live_slices, kSellResidentSlices), sr->hubs);
    sr->resident = std::max(1, std::min({wanted, kSellResidentBlocks, sr->live_slices}));  // each of several owns a row
    sr->resident_iters = sr->staged < kSellStaged ? kSellResidentIters : kSellResidentItersEmptyCu;
    const auto rounds = [&](int groups) { return ceil_div(sr->live_slices, groups * (kSellResidentThreads / kWave)) + ceil_div(sr->hubs, groups); };
    while (sr->rule.enough < sr->resident && rounds(sr->rule.enough) > rounds(sr->resident)) ++sr->rule.enough;
}

SellShape shape_of(const SellRows &sr)
{
    SellShape sh;
    sh.n = (int)sr.n;
    sh.hubs = sr.hubs;
    sh.slices = sr.slices;
    std::copy(sr.row_begin, sr.row_begin + kSellClasses + 1, sh.row_begin);
    std::copy(sr.slice_begin, sr.slice_begin + kSellClasses + 1, sh.slice_begin);
    return sh;
}

}  // namespace

bool sell_suits(int64_t n, int64_t nnz) { return n + nnz <= kSellMaxItems; }

namespace {

// f32_id: of sell_create_f32, or null.
template <typename Off>
int sell_build(SellRows *sr, int64_t n, int64_t nnz, const Off *row_ptr, const int32_t *col, int32_t *f32_id, hipStream_t s)
{
    const int hot = f32_id ? kSellHotF32 : kSellHot;
    sr->n = n;
    sr->nnz = nnz;
    sr->threads = n + nnz > kSellWideItems ? 512 : 256;
    constexpr int kWords = kSellClasses + 2;
    const int hub_limit = kWave * (f32_id ? kSellWaveStepsF32 : n + nnz > kSellWideItems ? kSellWaveStepsWide : kSellWaveSteps);
    unsigned *len = nullptr, *len_sorted = nullptr;
    int32_t *ids = nullptr, *new_id = f32_id, *hub_steps = nullptr, *slice_steps = nullptr, *slice_step = nullptr;
    int *bounds = nullptr, *h = nullptr;
    char *temp = nullptr;
    DeviceArena temps;
    const auto body = [&]() -> int {
        const size_t cnt = (size_t)n;
        // no more slices than rows of one lane each, plus one partly filled slice per class, plus 1 lane per kSellDepth / 2 entries
        const size_t most_slices = cnt / kWave + (size_t)nnz / (kWave * kSellDepth / 2) + 2 * kSellClasses + 1;
        const size_t most_hubs = (size_t)nnz / hub_limit + 1;
        size_t temp_bytes = 0, need = 0;
        sr->arena.want(&sr->order, cnt);
        sr->arena.want(&sr->hub_step, most_hubs + 1);
        sr->arena.want(&sr->slice, most_slices);
        if (!f32_id) {
            sr->arena.want(&sr->c[0], cnt + 1);
            sr->arena.want(&sr->c[1], cnt + 1);
            sr->arena.want(&sr->inv, cnt);
        }
        const size_t most_blocks = std::max<size_t>(most_hubs + ceil_div((int64_t)most_slices, sr->threads / kWave), kSellInitBlocks);
        if (!f32_id) {
            sr->arena.want(&sr->part[0], most_blocks);
            sr->arena.want(&sr->part[1], most_blocks);
        }
        DRONE_HIP_TRY(sr->arena.commit());
        DRONE_HIP_TRY(rocprim::radix_sort_pairs_desc(nullptr, temp_bytes, reinterpret_cast<unsigned *>(0x1000),
                                                     reinterpret_cast<unsigned *>(0x2000), reinterpret_cast<int32_t *>(0x3000),
                                                     sr->order, cnt, 0, 32, s));
        DRONE_HIP_TRY(rocprim::exclusive_scan(nullptr, need, reinterpret_cast<int32_t *>(0x1000), sr->hub_step, 0,
                                              std::max(most_slices, most_hubs) + 1, rocprim::plus<int32_t>(), s));
        temp_bytes = std::max(temp_bytes, need);
        temps.want(&len, cnt);
        temps.want(&len_sorted, cnt);
        temps.want(&ids, cnt);
        if (!f32_id) temps.want(&new_id, cnt);
        temps.want(&hub_steps, most_hubs + 1);
        temps.want(&slice_steps, most_slices + 1);
        temps.want(&slice_step, most_slices + 1);
        temps.want(&bounds, kWords);
        temps.want(&temp, temp_bytes);
        DRONE_HIP_TRY(temps.commit());
        DRONE_HIP_TRY(hipHostMalloc(&h, sizeof(int) * kWords));
        const int grid = (int)std::min<int64_t>(ceil_div(n, 256), 2048);
        int key_bits = 1;
        while (key_bits < 32 && (1ll << key_bits) <= nnz) ++key_bits;
        sell_lengths_kernel<<<grid, 256, 0, s>>>((int)n, row_ptr, len, ids);
        need = temp_bytes;
        DRONE_HIP_TRY(rocprim::radix_sort_pairs_desc(temp, need, len, len_sorted, ids, sr->order, cnt, 0, key_bits, s));
        sell_bounds_kernel<<<grid, 256, 0, s>>>((int)n, len_sorted, sr->order, f32_id != nullptr, hub_limit, new_id, bounds);
        if (n + nnz > kSellWideItems && nnz >= kSellSamples) sell_sample_kernel<<<kSellSamples / 256, 256, 0, s>>>(nnz, col, new_id, hot, bounds + kSellClasses);
        DRONE_HIP_TRY(hipMemcpyAsync(h, bounds, sizeof(int) * kWords, hipMemcpyDeviceToHost, s));
        DRONE_HIP_TRY(hipStreamSynchronize(s));
        if (h[kSellClasses] >= kSellHotShare * kSellSamples) {
            sr->hot = hot;
            sr->threads = kSellHotThreads;
            DRONE_HIP_TRY(hipFuncSetAttribute(f32_id ? reinterpret_cast<const void *>(&sell_push_kernel) : reinterpret_cast<const void *>(&sell_iterate_hot_kernel),
                                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)kSellHotLds));
        }
        if (f32_id && !sr->hot) return DRONE_OK;
        sr->hubs = h[0];
        for (int k = 0; k < kSellClasses; ++k) {
            sr->row_begin[k] = h[k];
            const int end = k + 1 < kSellClasses ? h[k + 1] : (int)n;
            sr->slice_begin[k + 1] = sr->slice_begin[k] + (int)ceil_div(end - h[k], 1 << k);
        }
        sr->row_begin[kSellClasses] = (int)n;
        sr->slices = sr->slice_begin[kSellClasses];
        DRONE_REQUIRE((size_t)sr->slices <= most_slices && (size_t)sr->hubs <= most_hubs, "slice bound");
        sr->blocks = sr->hot ? kSellHotBlocks : sr->hubs + (int)ceil_div(sr->slices, sr->threads / kWave);
        sr->init_blocks = (int)std::min<int64_t>(ceil_div(n, kSellInitThreads), kSellInitBlocks);
        if (!f32_id && !sr->hot) choose_resident(sr, h[kSellClasses + 1]);
        const SellShape sh = shape_of(*sr);
        sell_steps_kernel<<<(int)ceil_div(std::max(sr->slices, sr->hubs) + 1, 256), 256, 0, s>>>(sh, sr->threads, len_sorted, hub_steps, slice_steps);
        need = temp_bytes;
        DRONE_HIP_TRY(rocprim::exclusive_scan(temp, need, hub_steps, sr->hub_step, 0, (size_t)sr->hubs + 1, rocprim::plus<int32_t>(), s));
        need = temp_bytes;
        DRONE_HIP_TRY(rocprim::exclusive_scan(temp, need, slice_steps, slice_step, 0, (size_t)sr->slices + 1, rocprim::plus<int32_t>(), s));
        DRONE_HIP_TRY(hipMemcpyAsync(h, sr->hub_step + sr->hubs, sizeof(int), hipMemcpyDeviceToHost, s));
        DRONE_HIP_TRY(hipMemcpyAsync(h + 1, slice_step + sr->slices, sizeof(int), hipMemcpyDeviceToHost, s));
        DRONE_HIP_TRY(hipStreamSynchronize(s));
        sr->entries.want(&sr->hub_col, (size_t)h[0] * sr->threads);
        sr->entries.want(&sr->col, ((size_t)h[1] + kSellWaveSteps) * kWave);  // sell_resident_kernel reads so far beyond its slice
        const int slots = sr->staged * kSellResidentThreads;
        if (sr->resident) {
            sr->entries.want(&sr->exchange, 4 * (size_t)slots);
            sr->entries.want(&sr->gate, 3 * kTicketStride);
        }
        DRONE_HIP_TRY(sr->entries.commit());
        if (sr->resident) {
            sell_slots_kernel<<<64, 256, 0, s>>>(slots, sr->live, sr->exchange, sr->gate, h);
            // the limit belongs to the kernel, which plans of other sizes share
            DRONE_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(sell_resident_of(*sr)), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kSellResidentLds));
        }
        sell_fill_kernel<<<sr->hubs + (int)ceil_div(sr->slices, 256 / kWave), 256, 0, s>>>(
            sh, sr->threads, sr->order, row_ptr, col, new_id, sr->hub_step, slice_step, sr->slice, sr->hub_col, sr->col, sr->hot);
        DRONE_HIP_TRY(hipGetLastError());
        DRONE_HIP_TRY(hipStreamSynchronize(s));  // the temporaries go next
        if (sr->resident) {
            sr->failed = h;
            *sr->failed = 0;
            h = nullptr;
        }
        return DRONE_OK;
    };
    const int rc = body();
    temps.release();
    if (h) (void)hipHostFree(h);
    if (rc != DRONE_OK || (f32_id && !sr->hot)) sell_destroy(sr);
    return rc;
}

}  // namespace

int sell_create(SellRows *sr, int64_t n, int64_t nnz, const int64_t *row_ptr, const int32_t *col, hipStream_t s)
{
    return sell_build(sr, n, nnz, row_ptr, col, nullptr, s);
}

bool sell_f32_suits(int64_t n, int64_t nnz) { return n + nnz > kSellF32Items && n < INT32_MAX - 1; }

int sell_create_f32(SellRows *sr, int64_t n, int64_t nnz, const int *row_ptr, const int32_t *col, int32_t *new_id, hipStream_t s)
{
    return sell_build(sr, n, nnz, row_ptr, col, new_id, s);
}

void sell_destroy(SellRows *sr)
{
    sr->arena.release();
    sr->entries.release();
    if (sr->failed) (void)hipHostFree(sr->failed);
    *sr = SellRows{};
}

int sell_begin(const SellRows &sr, const double *inv_user, hipStream_t s)
{
    sell_begin_kernel<<<sr.init_blocks, kSellInitThreads, 0, s>>>((int)sr.n, sr.order, inv_user, 1.0 / (double)sr.n, sr.inv,
                                                                 sr.c[0], sr.c[1], sr.part[0]);
    DRONE_HIP_TRY(hipGetLastError());
    return DRONE_OK;
}

int sell_run(const SellRows &sr, const double *inv_user, int iters, double alpha, double *rank_out, hipStream_t s)
{
    if (__atomic_load_n(sr.failed, __ATOMIC_RELAXED)) {
        *sr.failed = 0;
        set_error(DRONE_ERR_HIP, "an earlier run of this plan waited in vain for one of its work-groups: its ranks are not valid");
        return DRONE_ERR_HIP;
    }
    SellGate rule = sr.rule;
    rule.price = (int)std::min<int64_t>((int64_t)iters * kSellLooksPerRound * (ceil_div(sr.live_slices, kSellResidentThreads / kWave) + sr.hubs), kSellMostLooks);
    sell_resident_of(sr)<<<sr.resident, kSellResidentThreads, sr.lds, s>>>(
        (int)sr.n, sr.live, sr.hubs, sr.live_slices, sr.threads, sr.hub_step, sr.hub_col, sr.slice, sr.col, sr.order, inv_user, sr.inv,
        sr.exchange, sr.gate, rule, iters, alpha, 1.0 / (double)sr.n, rank_out);
    DRONE_HIP_TRY(hipGetLastError());
    return DRONE_OK;
}

int sell_iterate(const SellRows &sr, int it, double alpha, double *rank_out, hipStream_t s)
{
    const int parts = it == 0 ? sr.init_blocks : sr.blocks, now = it & 1;
    const auto launch = [&](auto kernel, size_t lds) {
        kernel<<<sr.blocks, sr.threads, lds, s>>>((int)sr.n, sr.hubs, sr.slices, sr.hub_step, sr.hub_col, sr.slice, sr.col, sr.c[now], sr.inv,
                                                sr.c[now ^ 1], sr.part[now], parts, sr.part[now ^ 1], alpha,
                                                1.0 / (double)sr.n, sr.order, rank_out);
    };
    if (sr.hot) launch(sell_iterate_hot_kernel, kSellHotLds);
    else if (sr.threads == 512) launch(sell_iterate_kernel<512>, 0);
    else launch(sell_iterate_kernel<256>, 0);
    DRONE_HIP_TRY(hipGetLastError());
    return DRONE_OK;
}

int sell_push(const SellRows &sr, const float *push, float *diff, int *active, double *part, unsigned int *ticket, const StoreStat &stat,
              hipStream_t s)
{
    sell_push_kernel<<<sr.blocks, sr.threads, kSellHotLds, s>>>((int)sr.n, sr.hubs, sr.slices, sr.hub_step, sr.hub_col, sr.slice, sr.col,
                                                               push, sr.order, diff, active, part, ticket, stat);
    DRONE_HIP_TRY(hipGetLastError());
    return DRONE_OK;
}

}  // namespace drone
