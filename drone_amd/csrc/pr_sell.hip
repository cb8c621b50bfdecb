// One-launch-per-iteration fp64 PageRank: see pr_sell.h.
#include "pr_sell.h"

#include <algorithm>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

namespace drone {
namespace {

// Up to here (rows + entries) the layout beats the row blocks: at 8.5 M items 37.8 (41.3 without sources in LDS) against 43.8 us
// per iteration, at 17 M (8 MB of gather source, twice an XCD's L2) 73.7 against the 63.8 of the row blocks' sorted gathers.
constexpr int64_t kSellMaxItems = 9 << 20;
// Work-groups of 256 / 512 / 1,024 lanes, us per iteration at 0.012 / 0.057 / 1.02 / 2.07 / 4.2 / 8.5 M items: 4.05 / 4.7 /
// 9.1 / 14.6 / 24.2 / 51.5, 4.2 / 5.1 / 9.6 / 14.1 / 24.3 / 41.3, 5.3 / 6.3 / 12.2 / 14.5 / 21.1 / 43.4: small ones for small
// matrices (more CUs at work), 512 once the partials of so many work-groups and the hub rows count.
constexpr int64_t kSellWideItems = 1200 << 10;
constexpr int kSellInitThreads = 256, kSellInitBlocks = 512;
// From kSellWideItems on the hottest sources sit in LDS, if that many of the entries name one of them (of kSellSamples
// looked at): us per iteration without / with, and the share, 2.0 M items (131,072 vertices) 14.1 / 11.9 at 0.89, 4.2 M 24.2 / 18.5 at
// 0.79, 8.5 M 41.3 / 37.8 at 0.71, 1 M vertices and 7.8 M entries 45.3 / 40.6 at 0.63; half as many sources in LDS 41.3 / 44.0 at
// 0.57, 45.3 / 45.8 at 0.50.  Bringing 160 KB into every CU's LDS takes 3 us whatever there is to do: 1.0 M items 9.0 / 9.6.
constexpr double kSellHotShare = 0.6;
constexpr int kSellSamples = 1 << 16;
constexpr int kSellHotThreads = 1024, kSellHotBlocks = 256;
constexpr size_t kSellHotLds = sizeof(double) * kSellHot;
static_assert(kSellInitBlocks <= kSellHotThreads && kSellHot % 2 == 0, "a partial per lane; pairs");
constexpr int kSellMassLoads = 4;  // partials of the dangling mass per lane that are requested ahead

// What a kernel needs of SellRows, by value.
struct SellShape {
    int n, hubs, slices;
    int row_begin[kSellClasses + 1], slice_begin[kSellClasses + 1];
};

// Class of a row of `len` entries: the smallest P with at most kSellDepth entries per lane; class k has P = 64 >> k.
__host__ __device__ inline int sell_class_limit(int k, int hub_limit)  // longest row of class k
{
    return k == 0 ? hub_limit : (64 >> k) * kSellDepth;
}

template <int T>
__device__ __forceinline__ double block_sum(double v, double *s_red)  // valid in every thread
{
#pragma unroll
    for (int m = kWave / 2; m > 0; m >>= 1) v += __shfl_xor(v, m, kWave);
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

// Sum of c_in over `steps` consecutive steps of T ids starting at `ids` (this lane's), kSellDepth gathers in flight.
template <int T>
__device__ __forceinline__ double sell_sum(const int32_t *__restrict__ ids, int steps, const double *__restrict__ c_in, int pad)
{
    double sum = 0.0;
    for (int s = 0; s < steps; s += kSellDepth) {
        int id[kSellDepth];
        double v[kSellDepth];
#pragma unroll
        for (int k = 0; k < kSellDepth; ++k) id[k] = s + k < steps ? ids[(size_t)(s + k) * T] : pad;  // uniform condition
#pragma unroll
        for (int k = 0; k < kSellDepth; ++k) v[k] = s + k < steps ? c_in[id[k]] : 0.0;
#pragma unroll
        for (int k = 0; k < kSellDepth; ++k) sum += v[k];
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
    __shared__ double s_dang[T / kWave], s_red[T / kWave];
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
        sum = sell_sum<T>(hub_col + (size_t)s0 * T + tid, s1 - s0, c_in, n);
        sum = block_sum<T>(sum, s_red);
        __syncthreads();  // s_red is used again below
    } else {
        const int s = __builtin_amdgcn_readfirstlane(((int)blockIdx.x - hubs) * (T / kWave) + wave);
        if (s < slices) {  // the same for the whole wavefront
            const int4 d = slice[s];  // {first step, steps, first row, rows << 3 | log2(lanes per row)}
            const int lanes_log = d.w & 7, lanes = 1 << lanes_log, r = lane >> lanes_log;
            if ((lane & (lanes - 1)) == 0 && r < (d.w >> 3)) {
                row = d.z + r;
                iv = inv[row];
            }
            sum = sell_sum<kWave>(col + (size_t)d.x * kWave + lane, d.y, c_in, n);
            for (int m = lanes >> 1; m > 0; m >>= 1) sum += __shfl_xor(sum, m, kWave);
        }
    }
    double all = 0.0;
#pragma unroll
    for (int k = 0; k < kSellMassLoads; ++k) all += tid + k * T < parts ? mass[k] : 0.0;
    for (int i = tid + kSellMassLoads * T; i < parts; i += T) all += part_in[i];
    const double dang = block_sum<T>(all, s_dang);
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

// Sum of the sources of `steps` consecutive steps of T ids from `ids` on (this lane's), the first kSellDepth of which are there already.
// Both kinds of load are under the lanes' own condition: a hot lane costs the L1 nothing.
template <int T>
__device__ __forceinline__ double sell_hot_sum(int (&id)[kSellDepth], const int32_t *__restrict__ ids, int steps,
                                               const double *s_hot, const double *__restrict__ c_in)
{
    double sum = 0.0;
    for (int s = 0;;) {
        double v[kSellDepth];
#pragma unroll
        for (int k = 0; k < kSellDepth; ++k) {
            v[k] = 0.0;
            if (id[k] > kSellHot) v[k] = c_in[id[k] - 1];
        }
#pragma unroll
        for (int k = 0; k < kSellDepth; ++k)
            if (id[k] < kSellHot) v[k] = s_hot[id[k]];
        s += kSellDepth;
        if (s < steps) {
#pragma unroll
            for (int k = 0; k < kSellDepth; ++k) id[k] = s + k < steps ? ids[(size_t)(s + k) * T] : kSellHot;
        }
#pragma unroll
        for (int k = 0; k < kSellDepth; ++k) sum += v[k];
        if (s >= steps) return sum;
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
    extern __shared__ double s_hot[];  // [kSellHot]
    __shared__ double s_dang[T / kWave], s_red[T / kWave];
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int stride = (int)gridDim.x * (T / kWave);
    // The first slice's ids, and the dangling mass, travel beside the hot sources.
    int s = (int)blockIdx.x + (int)gridDim.x * wave;
    int4 d = s < slices ? slice[s] : make_int4(0, 0, 0, 0);
    int id[kSellDepth];
    const auto fetch = [&](int4 what, int (&to)[kSellDepth]) {
#pragma unroll
        for (int k = 0; k < kSellDepth; ++k) to[k] = k < what.y ? col[((size_t)what.x + k) * kWave + lane] : kSellHot;
    };
    fetch(d, id);
    const double mass = tid < parts ? part_in[tid] : 0.0;
    const int hot = n < kSellHot ? n : kSellHot;
    const double2 *c2 = reinterpret_cast<const double2 *>(c_in);
    constexpr int kPieces = (kSellHot / 2 + T - 1) / T;
    const int rot = ((int)blockIdx.x / 8) % kPieces;  // work-groups of an XCD would all ask one L2 channel for the same line: 2 M items 13.3 -> 11.9 us
#pragma unroll
    for (int k = 0; k < kPieces; ++k) {
        const int i = tid + (k + rot < kPieces ? k + rot : k + rot - kPieces) * T;
        if (2 * i + 1 < hot) reinterpret_cast<double2 *>(s_hot)[i] = c2[i];
        else if (2 * i < hot) s_hot[2 * i] = c_in[2 * i];
    }
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
        int hub_id[kSellDepth];
#pragma unroll
        for (int k = 0; k < kSellDepth; ++k) hub_id[k] = s0 + k < s1 ? ids[(size_t)k * T] : kSellHot;
        const double sum = block_sum<T>(sell_hot_sum<T>(hub_id, ids, s1 - s0, s_hot, c_in), s_red);
        if (tid == 0) finish(h, iv, sum);
        __syncthreads();  // s_red is used again
    }
    while (s < slices) {
        const int next = s + stride;
        const int4 after = next < slices ? slice[next] : make_int4(0, 0, 0, 0);
        const int lanes_log = d.w & 7, lanes = 1 << lanes_log, r = lane >> lanes_log;
        const bool mine = (lane & (lanes - 1)) == 0 && r < (d.w >> 3);
        const double iv = mine ? inv[d.z + r] : 0.0;
        int id_after[kSellDepth];
        fetch(after, id_after);
        double sum = sell_hot_sum<kWave>(id, col + (size_t)d.x * kWave + lane, d.y, s_hot, c_in);
        for (int m = lanes >> 1; m > 0; m >>= 1) sum += __shfl_xor(sum, m, kWave);
        if (mine) finish(d.z + r, iv, sum);
        d = after;
        s = next;
#pragma unroll
        for (int k = 0; k < kSellDepth; ++k) id[k] = id_after[k];
    }
    const double total = block_sum<T>(stat, s_red);
    if (tid == 0) part_out[blockIdx.x] = total;
}

// ---- building the layout ---------------------------------------------------------------------------------------------
__global__ void sell_lengths_kernel(int n, const int64_t *__restrict__ row_ptr, unsigned *__restrict__ len, int32_t *__restrict__ id)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        len[i] = (unsigned)(row_ptr[i + 1] - row_ptr[i]);
        id[i] = i;
    }
}

// new_id of every vertex; bounds[k] = rows (longest first) with more than limit[k] entries
__global__ void sell_bounds_kernel(int n, const unsigned *__restrict__ len_sorted, const int32_t *__restrict__ order,
                                   int hub_limit, int32_t *__restrict__ new_id, int *__restrict__ bounds)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) new_id[order[i]] = i;
    if (blockIdx.x != 0) return;
    if (threadIdx.x < kSellClasses) {
        const unsigned limit = (unsigned)sell_class_limit(threadIdx.x, hub_limit);
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

// *named += entries, of kSellSamples from all over the matrix, whose source is one of the first kSellHot
__global__ __launch_bounds__(256) void sell_sample_kernel(int64_t nnz, const int32_t *__restrict__ col, const int32_t *__restrict__ new_id,
                                                          int *__restrict__ named)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const unsigned long long hot = __ballot(new_id[col[(int64_t)((double)i / kSellSamples * (double)nnz)]] < kSellHot);
    if ((threadIdx.x & (kWave - 1)) == 0) atomicAdd(named, __popcll(hot));
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
__global__ __launch_bounds__(256) void sell_fill_kernel(SellShape sh, int threads, const int32_t *__restrict__ order,
                                                        const int64_t *__restrict__ row_ptr, const int32_t *__restrict__ col,
                                                        const int32_t *__restrict__ new_id,
                                                        const int32_t *__restrict__ hub_step,
                                                        const int32_t *__restrict__ slice_step, int4 *__restrict__ slice,
                                                        int32_t *__restrict__ hub_out, int32_t *__restrict__ out, bool hot)
{
    const auto source = [&](bool there, int64_t e) {
        if (!there) return hot ? kSellHot : sh.n;
        const int id = new_id[col[e]];
        return id + (hot && id >= kSellHot);
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

int sell_create(SellRows *sr, int64_t n, int64_t nnz, const int64_t *row_ptr, const int32_t *col, hipStream_t s)
{
    sr->n = n;
    sr->nnz = nnz;
    sr->threads = n + nnz > kSellWideItems ? 512 : 256;
    const int hub_limit = kWave * kSellWaveSteps;
    unsigned *len = nullptr, *len_sorted = nullptr;
    int32_t *ids = nullptr, *new_id = nullptr, *hub_steps = nullptr, *slice_steps = nullptr, *slice_step = nullptr;
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
        sr->arena.want(&sr->c[0], cnt + 1);
        sr->arena.want(&sr->c[1], cnt + 1);
        sr->arena.want(&sr->inv, cnt);
        const size_t most_blocks = std::max<size_t>(most_hubs + ceil_div((int64_t)most_slices, sr->threads / kWave), kSellInitBlocks);
        sr->arena.want(&sr->part[0], most_blocks);
        sr->arena.want(&sr->part[1], most_blocks);
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
        temps.want(&new_id, cnt);
        temps.want(&hub_steps, most_hubs + 1);
        temps.want(&slice_steps, most_slices + 1);
        temps.want(&slice_step, most_slices + 1);
        temps.want(&bounds, kSellClasses + 1);
        temps.want(&temp, temp_bytes);
        DRONE_HIP_TRY(temps.commit());
        DRONE_HIP_TRY(hipHostMalloc(&h, sizeof(int) * (kSellClasses + 1)));
        const int grid = (int)std::min<int64_t>(ceil_div(n, 256), 2048);
        int key_bits = 1;
        while (key_bits < 32 && (1ll << key_bits) <= nnz) ++key_bits;
        sell_lengths_kernel<<<grid, 256, 0, s>>>((int)n, row_ptr, len, ids);
        need = temp_bytes;
        DRONE_HIP_TRY(rocprim::radix_sort_pairs_desc(temp, need, len, len_sorted, ids, sr->order, cnt, 0, key_bits, s));
        sell_bounds_kernel<<<grid, 256, 0, s>>>((int)n, len_sorted, sr->order, hub_limit, new_id, bounds);
        if (n + nnz > kSellWideItems && nnz >= kSellSamples) sell_sample_kernel<<<kSellSamples / 256, 256, 0, s>>>(nnz, col, new_id, bounds + kSellClasses);
        DRONE_HIP_TRY(hipMemcpyAsync(h, bounds, sizeof(int) * (kSellClasses + 1), hipMemcpyDeviceToHost, s));
        DRONE_HIP_TRY(hipStreamSynchronize(s));
        if (h[kSellClasses] >= kSellHotShare * kSellSamples) {
            sr->hot = true;
            sr->threads = kSellHotThreads;
            DRONE_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(&sell_iterate_hot_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kSellHotLds));
        }
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
        sr->entries.want(&sr->col, (size_t)h[1] * kWave);
        DRONE_HIP_TRY(sr->entries.commit());
        sell_fill_kernel<<<sr->hubs + (int)ceil_div(sr->slices, 256 / kWave), 256, 0, s>>>(
            sh, sr->threads, sr->order, row_ptr, col, new_id, sr->hub_step, slice_step, sr->slice, sr->hub_col, sr->col, sr->hot);
        DRONE_HIP_TRY(hipGetLastError());
        DRONE_HIP_TRY(hipStreamSynchronize(s));  // the temporaries go next
        return DRONE_OK;
    };
    const int rc = body();
    temps.release();
    if (h) (void)hipHostFree(h);
    if (rc != DRONE_OK) sell_destroy(sr);
    return rc;
}

void sell_destroy(SellRows *sr)
{
    sr->arena.release();
    sr->entries.release();
    *sr = SellRows{};
}

int sell_begin(const SellRows &sr, const double *inv_user, hipStream_t s)
{
    sell_begin_kernel<<<sr.init_blocks, kSellInitThreads, 0, s>>>((int)sr.n, sr.order, inv_user, 1.0 / (double)sr.n, sr.inv,
                                                                 sr.c[0], sr.c[1], sr.part[0]);
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

}  // namespace drone
