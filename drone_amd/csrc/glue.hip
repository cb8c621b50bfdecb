// Element-wise and per-row kernels on the measured GCN step, semantics as in cuda_gcn/src/cuda/cuda_kernel.cu:
// ReLU (:384-399), dropout with an explicit keep mask (:403-420), soft-max cross-entropy (:295-379 with the
// host logic of cuda_module.cu:406-483), Adam (:450-460), plus SGD, accuracy (cuda_gcn.cu:226-246) and arg-max.
#include <algorithm>
#include <map>
#include <mutex>
#include <utility>

#include "spmv_merge.h"

namespace drone {
namespace {

constexpr int kThreads = 256;

inline int grid_for(int64_t n, int per_thread = 4)
{
    int64_t b = ceil_div(n, (int64_t)kThreads * per_thread);
    if (b < 1) b = 1;
    if (b > 65536) b = 65536;
    return (int)b;
}

__device__ __forceinline__ uint64_t splitmix64_dev(uint64_t x)
{
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}

// Four elements per lane when the count and the addresses allow 16-byte accesses (a float and a mask byte at a time: 10 us for
// 16,000 rows of 64, four: 5).
template <int V>
__global__ void relu_forward_kernel(float *__restrict__ x, uint8_t *__restrict__ mask, int64_t n, int training)
{
    for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q * V < n; q += (int64_t)gridDim.x * blockDim.x) {
        if constexpr (V == 4) {
            float4 t = reinterpret_cast<const float4 *>(x)[q];
            if (training) reinterpret_cast<uchar4 *>(mask)[q] = make_uchar4(t.x > 0, t.y > 0, t.z > 0, t.w > 0);
            if (!(t.x > 0)) t.x = 0;
            if (!(t.y > 0)) t.y = 0;
            if (!(t.z > 0)) t.z = 0;
            if (!(t.w > 0)) t.w = 0;
            reinterpret_cast<float4 *>(x)[q] = t;
        } else {
            const bool keep = x[q] > 0;
            if (training) mask[q] = keep;
            if (!keep) x[q] = 0;
        }
    }
}

template <int V>
__global__ void relu_backward_kernel(float *__restrict__ g, const uint8_t *__restrict__ mask, int64_t n)
{
    for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q * V < n; q += (int64_t)gridDim.x * blockDim.x) {
        if constexpr (V == 4) {
            float4 t = reinterpret_cast<const float4 *>(g)[q];
            const uchar4 m = reinterpret_cast<const uchar4 *>(mask)[q];
            if (!m.x) t.x = 0;
            if (!m.y) t.y = 0;
            if (!m.z) t.z = 0;
            if (!m.w) t.w = 0;
            reinterpret_cast<float4 *>(g)[q] = t;
        } else {
            if (!mask[q]) g[q] = 0;
        }
    }
}

inline bool four_wide(const float *x, const uint8_t *mask, int64_t n)
{
    return n % 4 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(mask) % 4 == 0;
}

// keep[i] = u(seed, step, i) >= p with u uniform in [0,1): a pure function of its arguments
__global__ void dropout_mask_kernel(uint8_t *__restrict__ keep, int64_t n, uint64_t seed, uint64_t step, float p)
{
    const uint64_t key = splitmix64_dev(splitmix64_dev(seed) ^ (step * 0xD1342543DE82EF95ull));
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const float u = (float)(splitmix64_dev(key + (uint64_t)i) >> 40) * (1.0f / 16777216.0f);
        keep[i] = u >= p;
    }
}

// cuda_kernel.cu:470-475: data[i] = (u - 0.5) * scale with u uniform in (0, 1], scale = 2 * sqrt(6 / (in + out)).
__global__ void glorot_kernel(float *__restrict__ w, int64_t n, uint64_t seed, float scale)
{
    const uint64_t key = splitmix64_dev(splitmix64_dev(seed) ^ 0x676C6F726F74ull);
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const float u = (float)((splitmix64_dev(key + (uint64_t)i) >> 40) + 1) * (1.0f / 16777216.0f);
        w[i] = (u - 0.5f) * scale;
    }
}

__global__ void dropout_apply_kernel(float *__restrict__ x, const uint8_t *__restrict__ keep, int64_t n, float scale)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        x[i] *= keep[i] ? scale : 0.0f;
}

// ReLU and the dropout that follows it in one pass over the activations (the two modules apart read and write them
// twice and the keep-mask three times): element by element the arithmetic of relu_forward_kernel, dropout_mask_kernel
// and dropout_apply_kernel in that order.  Four elements per lane when the count allows 16-byte accesses.
template <int V>
__global__ void relu_dropout_forward_kernel(float *__restrict__ x, uint8_t *__restrict__ mask, uint8_t *__restrict__ keep,
                                            int64_t n, uint64_t seed, uint64_t step, float p, float scale)
{
    const uint64_t key = splitmix64_dev(splitmix64_dev(seed) ^ (step * 0xD1342543DE82EF95ull));
    for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q * V < n; q += (int64_t)gridDim.x * blockDim.x) {
        float v[V];
        uint8_t m[V], k[V];
        if constexpr (V == 4) {
            const float4 t = reinterpret_cast<const float4 *>(x)[q];
            v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
        } else {
            v[0] = x[q];
        }
#pragma unroll
        for (int j = 0; j < V; ++j) {
            const int64_t i = q * V + j;
            m[j] = v[j] > 0;
            const float u = (float)(splitmix64_dev(key + (uint64_t)i) >> 40) * (1.0f / 16777216.0f);
            k[j] = u >= p;
            const float r = m[j] ? v[j] : 0.0f;
            v[j] = r * (k[j] ? scale : 0.0f);
        }
        if constexpr (V == 4) {
            reinterpret_cast<float4 *>(x)[q] = make_float4(v[0], v[1], v[2], v[3]);
            reinterpret_cast<uchar4 *>(mask)[q] = make_uchar4(m[0], m[1], m[2], m[3]);
            reinterpret_cast<uchar4 *>(keep)[q] = make_uchar4(k[0], k[1], k[2], k[3]);
        } else {
            x[q] = v[0];
            mask[q] = m[0];
            keep[q] = k[0];
        }
    }
}

// The two backward steps in the module list's order: g *= keep ? scale : 0 (dropout), then g = 0 where the ReLU was off.
template <int V>
__global__ void relu_dropout_backward_kernel(float *__restrict__ g, const uint8_t *__restrict__ mask,
                                             const uint8_t *__restrict__ keep, int64_t n, float scale)
{
    for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q * V < n; q += (int64_t)gridDim.x * blockDim.x) {
        if constexpr (V == 4) {
            float4 t = reinterpret_cast<const float4 *>(g)[q];
            const uchar4 m = reinterpret_cast<const uchar4 *>(mask)[q], k = reinterpret_cast<const uchar4 *>(keep)[q];
            t.x *= k.x ? scale : 0.0f; t.y *= k.y ? scale : 0.0f; t.z *= k.z ? scale : 0.0f; t.w *= k.w ? scale : 0.0f;
            if (!m.x) t.x = 0; if (!m.y) t.y = 0; if (!m.z) t.z = 0; if (!m.w) t.w = 0;
            reinterpret_cast<float4 *>(g)[q] = t;
        } else {
            float t = g[q] * (keep[q] ? scale : 0.0f);
            if (!mask[q]) t = 0;
            g[q] = t;
        }
    }
}

// L lanes per row, 64 / L rows per wavefront (L = the power of two that gives a lane at most four classes: a whole
// wavefront per 41-class row left a third of the lanes idle and took 74 us for 232,965 rows).  grad = softmax - onehot on
// labelled rows, 0 elsewhere; the per-block loss sum and labelled-row count go to block_loss / block_count.
// A lane keeps its (at most four) logits of a row in registers, and a wavefront has kCeGroups groups of 64 / L rows in
// flight: with one group, every step of the loop was a chain of two memory round trips (logits, then the store of the
// gradient behind them) and the kernel took 49 us for 232,965 x 41, twice what its 90 MB cost.
constexpr int kCeGroups = 2;
constexpr int kLossRowBlocks = 2048, kLossWeightBlocks = 64;  // most work-groups for the rows, for the weights
constexpr int kLossBlocks = kLossRowBlocks + kLossWeightBlocks;

// Parts of the work-groups: [0] loss, [1] labelled rows, [2] correct rows, [3] counted rows, [4] sum of squares.
struct LossScratch {
    double *part;          // [5][kLossBlocks]
    unsigned int *ticket;  // counters of last_block_done, zero between launches
    static constexpr size_t bytes() { return sizeof(double) * 5 * kLossBlocks + sizeof(unsigned int) * (kLossBlocks / kTicketGroup + 2) * kTicketStride; }
};

// A work-group's part of sum x[i]^2, in double: every lane four independent chains (one chain of dependent loads and fp64 adds
// in a single work-group took 117 us for the 77,056 weights of a 602 x 128 layer).  Valid in thread 0.
__device__ __forceinline__ double squares_part(const float *__restrict__ x, int64_t n, int block, int blocks)  // this lane's
{
    const int64_t step = (int64_t)blocks * kThreads;
    double t[4] = {0.0, 0.0, 0.0, 0.0};
    int64_t i = (int64_t)block * kThreads + threadIdx.x;
    for (; i + 3 * step < n; i += 4 * step) {
        const float a = x[i], b = x[i + step], c = x[i + 2 * step], d = x[i + 3 * step];
        t[0] += (double)a * (double)a;
        t[1] += (double)b * (double)b;
        t[2] += (double)c * (double)c;
        t[3] += (double)d * (double)d;
    }
    for (; i < n; i += step) t[0] += (double)x[i] * (double)x[i];
    return (t[0] + t[1]) + (t[2] + t[3]);
}

template <typename V>
__device__ __forceinline__ V sum_of_lanes(V v)
{
#pragma unroll
    for (int m = kWave / 2; m > 0; m >>= 1) v += __shfl_xor(v, m, kWave);
    return v;
}

// The loss, the gradient, and what is reported with them, in one launch: the last work-group adds the parts of all.
// Work-groups past row_blocks add up the squares of the weights meanwhile.  A training step and the report of its loss
// spent five launches and three copies on this (cross-entropy and its finish, accuracy and the clearing of its counts,
// sum of squares; ~5 us each where the graph is small): an epoch with its evaluation on 2,708
// vertices 310 -> 190 us.  (The five sums share a barrier on either side of the hand-over: 8.2 -> 6.3 us there.)
// With a split (drone_loss_pass_split_f32) the truth is chosen on the way, and written down for who reads it later: a launch
// less in either pass of an epoch, 151 -> 145 us for the two of it on 2,708 vertices.
struct TruthChoice {
    const int *split = nullptr, *label = nullptr;
    int which = 0;
    int *truth = nullptr;
};
template <int L>
__global__ __launch_bounds__(kThreads) void loss_kernel(drone_loss_pass p, TruthChoice choice, int row_blocks, LossScratch scratch)
{
    constexpr int R = kWave / L, kWaves = kThreads / kWave, U = kCeGroups;
    __shared__ double s_red[5][kWaves];
    static_assert(kWaves == 4, "the sums of four wavefronts");
    const int n = p.n, classes = p.classes, ld = p.ld, ldg = p.ldg;
    const float *__restrict__ logits = p.logits;
    const int *__restrict__ truth = p.truth;
    const auto truth_of = [&](int row, bool writes) {
        if (!choice.split) return truth[row];
        const int label = choice.label[row], t = choice.split[row] == choice.which ? label : -1;
        if (writes) choice.truth[row] = t;
        return t;
    };
    float *__restrict__ grad = p.grad;
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int li = lane % L, sub = lane / L;
    const int per_lane = (classes + L - 1) / L;  // more than 4 only in the 64-lane instance
    double loss = 0.0;
    int cnt = 0, correct = 0, counted = 0;
    double squares = 0.0;
    if ((int)blockIdx.x >= row_blocks)
        squares = squares_part(p.weights, p.weight_count, (int)blockIdx.x - row_blocks, (int)gridDim.x - row_blocks);
    const int mean_over = p.mean_over && grad ? *p.mean_over : 0;
    const float grad_scale = p.mean_over ? (mean_over > 0 ? 1.0f / (float)mean_over : 1.0f) : p.grad_scale;
    for (int64_t base = ((int64_t)blockIdx.x * kWaves + wave) * R * U; base < n && (int)blockIdx.x < row_blocks;
         base += (int64_t)row_blocks * kWaves * R * U) {
        const int row0 = (int)base;
        if (per_lane <= 4) {
            float z[U][4];
            int t[U];
            bool skip[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int row = row0 + u * R + sub;
                const float *src = logits + (size_t)(row < n ? row : n - 1) * ld;
#pragma unroll
                for (int k = 0; k < 4; ++k) z[u][k] = li + k * L < classes ? src[li + k * L] : -INFINITY;
                t[u] = row < n ? truth_of(row, li == 0) : -1;
                skip[u] = p.skip && row < n && p.skip[row] != -1;
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int row = row0 + u * R + sub;
                const bool labelled = t[u] >= 0 && t[u] < classes;  // a label outside the classes counts as none
                float mx = fmaxf(fmaxf(z[u][0], z[u][1]), fmaxf(z[u][2], z[u][3]));
#pragma unroll
                for (int m = L / 2; m > 0; m >>= 1) mx = fmaxf(mx, __shfl_xor(mx, m, kWave));
                float e[4], sum = 0.0f;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    e[k] = li + k * L < classes ? expf(z[u][k] - mx) : 0.0f;
                    sum += e[k];
                }
#pragma unroll
                for (int m = L / 2; m > 0; m >>= 1) sum += __shfl_xor(sum, m, kWave);
                // the true class's logit sits in lane t % L, register t / L
                float zt = 0.0f;
#pragma unroll
                for (int k = 0; k < 4; ++k) zt = (labelled && t[u] / L == k) ? z[u][k] : zt;
                zt = __shfl(zt, labelled ? sub * L + t[u] % L : lane, kWave);
                if (grad && row < n) {
                    const float inv = 1.0f / sum;
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const int j = li + k * L;
                        if (j < classes) {
                            float g = 0.0f;
                            if (labelled) {
                                g = e[k] * inv;
                                if (j == t[u]) g -= 1.0f;
                                g *= grad_scale;
                            }
                            grad[(size_t)row * ldg + j] = g;
                        }
                    }
                }
                if (li == 0 && labelled) {
                    loss += (double)(logf(sum) - (zt - mx));
                    cnt += 1;
                    if (!skip[u]) {
                        counted += 1;
                        correct += !(mx > zt);
                    }
                }
            }
        } else {
            for (int u = 0; u < U; ++u) {
                const int row = row0 + u * R + sub;
                const bool valid = row < n;
                const float *z = logits + (size_t)(valid ? row : 0) * ld;
                const int t = valid ? truth_of(row, li == 0) : -1;
                const bool labelled = t >= 0 && t < classes;
                float mx = -INFINITY;
                for (int j = li; j < classes; j += L) mx = fmaxf(mx, z[j]);
#pragma unroll
                for (int m = L / 2; m > 0; m >>= 1) mx = fmaxf(mx, __shfl_xor(mx, m, kWave));
                float sum = 0.0f;
                for (int j = li; j < classes; j += L) sum += expf(z[j] - mx);
#pragma unroll
                for (int m = L / 2; m > 0; m >>= 1) sum += __shfl_xor(sum, m, kWave);
                if (grad && valid)
                    for (int j = li; j < classes; j += L) {
                        float g = 0.0f;
                        if (labelled) {
                            g = expf(z[j] - mx) / sum;
                            if (j == t) g -= 1.0f;
                            g *= grad_scale;
                        }
                        grad[(size_t)row * ldg + j] = g;
                    }
                if (li == 0 && labelled) {
                    loss += (double)(logf(sum) - (z[t] - mx));
                    cnt += 1;
                    if (!p.skip || p.skip[row] == -1) {
                        counted += 1;
                        correct += !(mx > z[t]);
                    }
                }
            }
        }
    }
    // (whole numbers below 2^53: exact)
    const auto to_lds = [&](const double (&v)[5]) {
        if (lane == 0) {
#pragma unroll
            for (int k = 0; k < 5; ++k) s_red[k][wave] = v[k];
        }
        __syncthreads();
    };
    const auto of_block = [&](int k) { return (s_red[k][0] + s_red[k][1]) + (s_red[k][2] + s_red[k][3]); };
    to_lds({sum_of_lanes(loss), (double)sum_of_lanes(cnt), (double)sum_of_lanes(correct), (double)sum_of_lanes(counted), sum_of_lanes(squares)});
    unsigned int one = 0;
    // five lanes, one instruction: it has returned for all of them when it has for thread 0
    if (threadIdx.x < 5) one = publish_part(scratch.part + threadIdx.x * kLossBlocks + blockIdx.x, of_block(threadIdx.x));
    if (!last_block_done(scratch.ticket, one)) return;
    double sum[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    for (int i = threadIdx.x; i < (int)gridDim.x; i += kThreads)
#pragma unroll
        for (int k = 0; k < 5; ++k) sum[k] += load_agent(scratch.part + k * kLossBlocks + i);
#pragma unroll
    for (int k = 0; k < 5; ++k) sum[k] = sum_of_lanes(sum[k]);
    to_lds(sum);
    if (threadIdx.x != 0) return;
#pragma unroll
    for (int k = 0; k < 5; ++k) sum[k] = of_block(k);
    const float mean = (float)(sum[0] / sum[1]);  // over the labelled rows
    if (p.loss) *p.loss = mean;
    if (p.labelled) *p.labelled = (int)sum[1];
    if (p.report) *p.report = drone_loss_report{mean, (float)sum[4], (int)sum[1], (int)sum[2], (int)sum[3]};
}

// cuda_gcn.cu:226-246: a labelled row is wrong iff some logit is strictly greater than the true-class logit; rows of
// mirrors (skip[row] != -1, the reference's Mirror2WorkerHost) are left out of the counts (:234).
// pred[row] = arg-max with ties to the lowest index (optional).  counts[0] += correct, counts[1] += labelled.
// kAccGroups groups of 64 / L rows are in flight per wavefront, their logits in registers (see loss_kernel).
constexpr int kAccGroups = 4;
// Work-groups of 1024 lanes, at most one per CU: every work-group ends with two atomics on the same two counters, and
// those cost about 9 ns each (1024 work-groups of 256 lanes: 40 us for 232,965 x 41, 2048: 58 us).
constexpr int kAccThreads = 1024, kAccBlocks = 256;
template <int L>  // lanes per row, as in loss_kernel
__global__ __launch_bounds__(kAccThreads) void accuracy_kernel(int n, int classes, const float *__restrict__ logits, int ld,
                                                            const int *__restrict__ truth, const int *__restrict__ skip,
                                                            int *__restrict__ pred, int *__restrict__ counts)
{
    constexpr int R = kWave / L, kWaves = kAccThreads / kWave, U = kAccGroups;
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int li = lane % L, sub = lane / L;
    const int per_lane = (classes + L - 1) / L;  // more than 4 only in the 64-lane instance
    int correct = 0, total = 0;
    for (int row0 = (blockIdx.x * kWaves + wave) * R * U; row0 < n; row0 += gridDim.x * kWaves * R * U) {
        float best[U], zt[U];
        int arg[U], t[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int row = row0 + u * R + sub;
            const bool valid = row < n;
            const float *z = logits + (size_t)(valid ? row : n - 1) * ld;
            best[u] = -INFINITY;
            arg[u] = INT32_MAX;
            t[u] = (valid && truth) ? truth[row] : -1;
            if (skip && valid && skip[row] != -1) t[u] = -1;
            if (t[u] >= classes) t[u] = -1;
            if (per_lane <= 4) {
                float v[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) v[k] = li + k * L < classes ? z[li + k * L] : -INFINITY;
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (v[k] > best[u]) { best[u] = v[k]; arg[u] = li + k * L; }
                // the true class's logit sits in lane t % L, register t / L: no second trip to memory behind the label
                float mine = 0.0f;
#pragma unroll
                for (int k = 0; k < 4; ++k) mine = (t[u] >= 0 && t[u] / L == k) ? v[k] : mine;
                zt[u] = __shfl(mine, t[u] >= 0 ? sub * L + t[u] % L : lane, kWave);
            } else {
                for (int j = li; j < classes; j += L) {
                    const float v = z[j];
                    if (v > best[u]) { best[u] = v; arg[u] = j; }
                }
                zt[u] = t[u] >= 0 ? z[t[u]] : 0.0f;
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int row = row0 + u * R + sub;
#pragma unroll
            for (int m = L / 2; m > 0; m >>= 1) {
                const float ob = __shfl_xor(best[u], m, kWave);
                const int oa = __shfl_xor(arg[u], m, kWave);
                if (ob > best[u] || (ob == best[u] && oa < arg[u])) { best[u] = ob; arg[u] = oa; }
            }
            if (li == 0 && row < n) {
                if (pred) pred[row] = arg[u];
                if (t[u] >= 0) {
                    total++;
                    if (!(best[u] > zt[u])) correct++;
                }
            }
        }
    }
#pragma unroll
    for (int m = kWave / 2; m > 0; m >>= 1) {
        correct += __shfl_xor(correct, m, kWave);
        total += __shfl_xor(total, m, kWave);
    }
    // one pair of atomics per work-group, not per wavefront: they all hit the same two addresses
    __shared__ int s_correct[kWaves], s_total[kWaves];
    if (lane == 0) { s_correct[wave] = correct; s_total[wave] = total; }
    __syncthreads();
    if (counts && threadIdx.x == 0) {
        int c = 0, t = 0;
        for (int w = 0; w < kWaves; ++w) { c += s_correct[w]; t += s_total[w]; }
        if (t) {
            atomicAdd(&counts[0], c);
            atomicAdd(&counts[1], t);
        }
    }
}

// out[0] = sum of x[i]^2, accumulated in double by one work-group of 1024 in a fixed order (weights are small).  Four
// independent chains per thread: one chain of dependent loads and fp64 adds took 117 us for the 77,056 weights of a
// 602 x 128 layer.
__global__ __launch_bounds__(1024) void sum_squares_kernel(const float *__restrict__ x, int64_t n, float *__restrict__ out)
{
    __shared__ double s_part[1024 / kWave];
    double t[4] = {0.0, 0.0, 0.0, 0.0};
    int64_t i = threadIdx.x;
    for (; i + 3 * 1024 < n; i += 4 * 1024) {
        const float a = x[i], b = x[i + 1024], c = x[i + 2 * 1024], d = x[i + 3 * 1024];
        t[0] += (double)a * (double)a;
        t[1] += (double)b * (double)b;
        t[2] += (double)c * (double)c;
        t[3] += (double)d * (double)d;
    }
    for (; i < n; i += 1024) t[0] += (double)x[i] * (double)x[i];
    double v = (t[0] + t[1]) + (t[2] + t[3]);
#pragma unroll
    for (int m = kWave / 2; m > 0; m >>= 1) v += __shfl_xor(v, m, kWave);
    if ((threadIdx.x & (kWave - 1)) == 0) s_part[threadIdx.x / kWave] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double total = 0.0;
        for (int w = 0; w < 1024 / kWave; ++w) total += s_part[w];
        out[0] = (float)total;
    }
}

// One launch for all tensors of an optimiser step: blockIdx.y is the tensor.
constexpr int kStepTensors = 4;
struct StepTensors {
    drone_step_tensor t[kStepTensors];
    drone_step_sums sums[kStepTensors];
};
struct SgdStep {
    float lr;
    __device__ __forceinline__ void operator()(const drone_step_tensor &t, int64_t i, float g) const { t.w[i] -= lr * g; }
};

// cuda_kernel.cu:450-460
struct AdamStep {
    float weight_decay, beta1, beta2, eps, step_size;
    __device__ __forceinline__ void operator()(const drone_step_tensor &t, int64_t i, float g) const
    {
        const float w = t.w[i];
        if (t.decay) g += weight_decay * w;
        const float mi = (float)(beta1 * t.m[i] + (1.0 - beta1) * g);
        const float vi = (float)(beta2 * t.v[i] + (1.0 - beta2) * g * g);
        t.m[i] = mi;
        t.v[i] = vi;
        t.w[i] = w - step_size * mi / (sqrtf(vi) + eps);
    }
};

// A tensor's gradient is there, or still the partial sums of a split reduction, which are then added up as sgemm_reduce_kernel does
// it: 32 outputs to 256 lanes, eight sums of an output in flight, a fixed order.  Bound by launches: a reduction of its own for each of two
// weights, and the step, were 3.4 to 4.7 us each (epoch on 2,708 vertices and its evaluation 145 -> 138 us, 30,011-vertex step, whose layer 1 keeps its reduction, 226 -> 224).
template <typename Step>
__global__ __launch_bounds__(kThreads) void step_kernel(StepTensors tensors, Step step)
{
    constexpr int G = 8, O = kThreads / G;
    __shared__ float s_sum[G][O];
    const drone_step_tensor t = tensors.t[blockIdx.y];
    const drone_step_sums from = tensors.sums[blockIdx.y];
    if (from.splits <= 0) {
        for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < t.n; i += (int64_t)gridDim.x * kThreads) step(t, i, t.grad[i]);
        return;
    }
    const int o = threadIdx.x % O, g = threadIdx.x / O;
    for (int64_t base = (int64_t)blockIdx.x * O; base < t.n; base += (int64_t)gridDim.x * O) {
        const int64_t i = base + o;
        float sum = 0.0f;
        if (i < t.n) {
            int z = g;
            for (; z + 7 * G < from.splits; z += 8 * G) {
                float v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = from.sums[(size_t)(z + u * G) * t.n + i];
#pragma unroll
                for (int u = 0; u < 8; ++u) sum += v[u];
            }
            for (; z < from.splits; z += G) sum += from.sums[(size_t)z * t.n + i];
        }
        s_sum[g][o] = sum;
        __syncthreads();
        if (g == 0 && i < t.n) {
#pragma unroll
            for (int k = 1; k < G; ++k) sum += s_sum[k][o];
            const_cast<float *>(t.grad)[i] = sum;
            step(t, i, sum);
        }
        __syncthreads();
    }
}

__global__ void fill_f32_kernel(float *__restrict__ x, int64_t n, float value)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        x[i] = value;
}

// LossScratch, one per (device, stream): calls on one stream are
// ordered and share it, calls on different streams may overlap
std::mutex g_mutex;
std::map<std::pair<int, hipStream_t>, void *> g_loss_scratch;

// Zeroed on a stream of its own and waited for: the caller's may be recording a graph, and then a fill on it would run at
// the replays instead of now.
int loss_scratch_create(void **out)
{
    void *p = nullptr;
    hipStream_t once = nullptr;
    DRONE_HIP_TRY(hipMalloc(&p, LossScratch::bytes()));
    hipError_t e = hipStreamCreateWithFlags(&once, hipStreamNonBlocking);
    if (e == hipSuccess) {
        fill_f32_kernel<<<64, kThreads, 0, once>>>(static_cast<float *>(p), (int64_t)(LossScratch::bytes() / sizeof(float)), 0.0f);
        e = hipGetLastError();
        const hipError_t waited = hipStreamSynchronize(once);
        if (e == hipSuccess) e = waited;
        (void)hipStreamDestroy(once);
    }
    if (e != hipSuccess) {
        (void)hipFree(p);
        set_error(DRONE_ERR_HIP, "scratch of the loss: %s", hipGetErrorString(e));
        return DRONE_ERR_HIP;
    }
    *out = p;
    return DRONE_OK;
}

}  // namespace
}  // namespace drone

using namespace drone;

extern "C" int drone_relu_forward_f32(float *x, uint8_t *mask, int64_t n, int training, drone_stream_t stream)
{
    clear_error();
    DRONE_REQUIRE(n >= 0 && (n == 0 || x) && (!training || mask || n == 0), "null operand");
    if (n == 0) return DRONE_OK;
    if (four_wide(x, mask, n)) relu_forward_kernel<4><<<grid_for(n / 4, 1), kThreads, 0, as_stream(stream)>>>(x, mask, n, training);
    else relu_forward_kernel<1><<<grid_for(n), kThreads, 0, as_stream(stream)>>>(x, mask, n, training);
    DRONE_HIP_TRY(hipGetLastError());
    return DRONE_OK;
}

extern "C" int drone_relu_backward_f32(float *grad, const uint8_t *mask, int64_t n, drone_stream_t stream)
{
    clear_error();
    DRONE_REQUIRE(n >= 0 && (n == 0 || (grad && mask)), "null operand");
    if (n == 0) return DRONE_OK;
    if (four_wide(grad, mask, n)) relu_backward_kernel<4><<<grid_for(n / 4, 1), kThreads, 0, as_stream(stream)>>>(grad, mask, n);
    else relu_backward_kernel<1><<<grid_for(n), kThreads, 0, as_stream(stream)>>>(grad, mask, n);
    DRONE_HIP_TRY(hipGetLastError());
    return DRONE_OK;
}

extern "C" int drone_dropout_mask(uint8_t *keep, int64_t n, uint64_t seed, uint64_t step, float p, drone_stream_t stream)
{
    clear_error();
    DRONE_REQUIRE(n >= 0 && (n == 0 || keep) && p >= 0.0f && p < 1.0f, "mask / probability");
    if (n == 0) return DRONE_OK;
    dropout_mask_kernel<<<grid_for(n), kThreads, 0, as_stream(stream)>>>(keep, n, seed, step, p);
    DRONE_HIP_TRY(hipGetLastError());
    return DRONE_OK;
}

// cuda_variable.cu:18-24 (CUDAVariable::glorot): n weights uniform in (-r, r], r = sqrtf(6 / (in_size + out_size)).
// The reference draws from cuRAND states seeded with 1234 (cuda_kernel.cu:423-426), whose bit stream cannot be
// reproduced without cuRAND; here element i is a function of (seed, i) alone.
extern "C" int drone_glorot_uniform_f32(float *w, int64_t n, int in_size, int out_size, uint64_t seed, drone_stream_t stream)
{
    clear_error();
    DRONE_REQUIRE(n >= 0 && (n == 0 || w) && in_size > 0 && out_size > 0, "weights / fan-in / fan-out");
    if (n == 0) return DRONE_OK;
    const float range = sqrtf(6.0f / (float)(in_size + out_size));
    glorot_kernel<<<grid_for(n), kThreads, 0, as_stream(stream)>>>(w, n, seed, range * 2);
    DRONE_HIP_TRY(hipGetLastError());
    return DRONE_OK;
}

// Forward and backward are the same scaling (cuda_kernel.cu:403-420): x *= keep ? 1/(1-p) : 0.
extern "C" int drone_dropout_apply_f32(float *x, const uint8_t *keep, int64_t n, float p, drone_stream_t stream)
{
    clear_error();
    DRONE_REQUIRE(n >= 0 && (n == 0 || (x && keep)) && p >= 0.0f && p < 1.0f, "operand / probability");
    if (n == 0) return DRONE_OK;
    dropout_apply_kernel<<<grid_for(n), kThreads, 0, as_stream(stream)>>>(x, keep, n, 1 / (1 - p));
    DRONE_HIP_TRY(hipGetLastError());
    return DRONE_OK;
}

extern "C" int drone_relu_dropout_forward_f32(float *x, uint8_t *mask, uint8_t *keep, int64_t n, uint64_t seed,
                                              uint64_t step, float p, drone_stream_t stream)
{
    clear_error();
    DRONE_REQUIRE(n >= 0 && (n == 0 || (x && mask && keep)) && p >= 0.0f && p < 1.0f, "operands / probability");
    if (n == 0) return DRONE_OK;
    const bool wide = n % 4 == 0 && (reinterpret_cast<uintptr_t>(x) % 16 == 0) &&
                      (reinterpret_cast<uintptr_t>(mask) % 4 == 0) && (reinterpret_cast<uintptr_t>(keep) % 4 == 0);
    if (wide)
        relu_dropout_forward_kernel<4><<<grid_for(n / 4, 2), kThreads, 0, as_stream(stream)>>>(x, mask, keep, n, seed, step, p, 1 / (1 - p));
    else
        relu_dropout_forward_kernel<1><<<grid_for(n), kThreads, 0, as_stream(stream)>>>(x, mask, keep, n, seed, step, p, 1 / (1 - p));
    DRONE_HIP_TRY(hipGetLastError());
    return DRONE_OK;
}

extern "C" int drone_relu_dropout_backward_f32(float *grad, const uint8_t *mask, const uint8_t *keep, int64_t n, float p,
                                               drone_stream_t stream)
{
    clear_error();
    DRONE_REQUIRE(n >= 0 && (n == 0 || (grad && mask && keep)) && p >= 0.0f && p < 1.0f, "operands / probability");
    if (n == 0) return DRONE_OK;
    const bool wide = n % 4 == 0 && (reinterpret_cast<uintptr_t>(grad) % 16 == 0) &&
                      (reinterpret_cast<uintptr_t>(mask) % 4 == 0) && (reinterpret_cast<uintptr_t>(keep) % 4 == 0);
    if (wide)
        relu_dropout_backward_kernel<4><<<grid_for(n / 4, 2), kThreads, 0, as_stream(stream)>>>(grad, mask, keep, n, 1 / (1 - p));
    else
        relu_dropout_backward_kernel<1><<<grid_for(n), kThreads, 0, as_stream(stream)>>>(grad, mask, keep, n, 1 / (1 - p));
    DRONE_HIP_TRY(hipGetLastError());
    return DRONE_OK;
}

namespace {
int loss_pass(const drone_loss_pass &p, const TruthChoice &choice, drone_stream_t stream)
{
    DRONE_REQUIRE(p.n > 0 && p.classes > 0 && p.logits && (p.truth || choice.split) && p.ld >= p.classes, "operands");
    DRONE_REQUIRE(p.grad == nullptr || p.ldg >= p.classes, "ldg < classes");
    DRONE_REQUIRE(p.weight_count >= 0 && (p.weights || p.weight_count == 0), "weights");
    int dev = 0;
    DRONE_HIP_TRY(hipGetDevice(&dev));
    hipStream_t s = as_stream(stream);
    void *ws = nullptr;
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        void *&slot = g_loss_scratch[std::make_pair(dev, s)];
        if (!slot) {
            const int rc = loss_scratch_create(&slot);
            if (rc != DRONE_OK) return rc;
        }
        ws = slot;
    }
    double *part = static_cast<double *>(ws);
    const LossScratch scratch{part, reinterpret_cast<unsigned int *>(part + 5 * kLossBlocks)};
    const int lanes = p.classes <= 16 ? 4 : p.classes <= 32 ? 8 : p.classes <= 64 ? 16 : p.classes <= 128 ? 32 : 64;  // per row
    const int row_blocks = (int)std::min<int64_t>(ceil_div(p.n, kThreads / lanes * kCeGroups), kLossRowBlocks);
    const int weight_blocks = (int)std::min<int64_t>(ceil_div(p.weight_count, kThreads * 8), kLossWeightBlocks);
    const int blocks = row_blocks + weight_blocks;
    if (lanes == 4) loss_kernel<4><<<blocks, kThreads, 0, s>>>(p, choice, row_blocks, scratch);
    else if (lanes == 8) loss_kernel<8><<<blocks, kThreads, 0, s>>>(p, choice, row_blocks, scratch);
    else if (lanes == 16) loss_kernel<16><<<blocks, kThreads, 0, s>>>(p, choice, row_blocks, scratch);
    else if (lanes == 32) loss_kernel<32><<<blocks, kThreads, 0, s>>>(p, choice, row_blocks, scratch);
    else loss_kernel<64><<<blocks, kThreads, 0, s>>>(p, choice, row_blocks, scratch);
    DRONE_HIP_TRY(hipGetLastError());
    return DRONE_OK;
}
}  // namespace

extern "C" int drone_loss_pass_f32(const drone_loss_pass *pass, drone_stream_t stream)
{
    clear_error();
    DRONE_REQUIRE(pass != nullptr, "null pass");
    return loss_pass(*pass, TruthChoice{}, stream);
}

extern "C" int drone_loss_pass_split_f32(const drone_loss_pass *pass, const int *split, const int *label, int which, int *truth,
                                         drone_stream_t stream)
{
    clear_error();
    DRONE_REQUIRE(pass != nullptr && split && label && truth, "null pass / split / label / truth");
    TruthChoice choice;
    choice.split = split;
    choice.label = label;
    choice.which = which;
    choice.truth = truth;
    return loss_pass(*pass, choice, stream);
}

extern "C" int drone_cross_entropy_f32(int n, int classes, const float *logits, int ld, const int *truth, float *grad,
                                       int ldg, float grad_scale, float *loss_out, int *count_out,
                                       drone_stream_t stream)
{
    drone_loss_pass p{};
    p.n = n;
    p.classes = classes;
    p.logits = logits;
    p.ld = ld;
    p.truth = truth;
    p.grad = grad;
    p.ldg = ldg;
    p.grad_scale = grad_scale;
    p.loss = loss_out;
    p.labelled = count_out;
    return drone_loss_pass_f32(&p, stream);
}

extern "C" int drone_sum_squares_f32(const float *x, int64_t n, float *out, drone_stream_t stream)
{
    clear_error();
    DRONE_REQUIRE(n >= 0 && (n == 0 || x) && out, "null operand");
    sum_squares_kernel<<<1, 1024, 0, as_stream(stream)>>>(x, n, out);
    DRONE_HIP_TRY(hipGetLastError());
    return DRONE_OK;
}

extern "C" int drone_accuracy_f32(int n, int classes, const float *logits, int ld, const int *truth, const int *skip,
                                  int *pred, int *counts, drone_stream_t stream)
{
    clear_error();
    DRONE_REQUIRE(n > 0 && classes > 0 && logits && ld >= classes, "operands");
    hipStream_t s = as_stream(stream);
    int blocks = (int)ceil_div(n, kAccThreads / kWave);
    if (blocks > kAccBlocks) blocks = kAccBlocks;
    if (classes <= 16) accuracy_kernel<4><<<blocks, kAccThreads, 0, s>>>(n, classes, logits, ld, truth, skip, pred, counts);
    else if (classes <= 32) accuracy_kernel<8><<<blocks, kAccThreads, 0, s>>>(n, classes, logits, ld, truth, skip, pred, counts);
    else if (classes <= 64) accuracy_kernel<16><<<blocks, kAccThreads, 0, s>>>(n, classes, logits, ld, truth, skip, pred, counts);
    else if (classes <= 128) accuracy_kernel<32><<<blocks, kAccThreads, 0, s>>>(n, classes, logits, ld, truth, skip, pred, counts);
    else accuracy_kernel<64><<<blocks, kAccThreads, 0, s>>>(n, classes, logits, ld, truth, skip, pred, counts);
    DRONE_HIP_TRY(hipGetLastError());
    return DRONE_OK;
}

namespace {
template <typename Step>
int launch_steps(const drone_step_tensor *t, const drone_step_sums *sums, int tensors, const Step &step, hipStream_t s)
{
    StepTensors all{};
    int grid = 1;
    for (int i = 0; i < tensors; ++i) {
        all.t[i] = t[i];
        if (sums) all.sums[i] = sums[i];
        grid = std::max(grid, all.sums[i].splits > 0 ? grid_for(8 * t[i].n, 1) : grid_for(t[i].n));
    }
    step_kernel<<<dim3(grid, tensors), kThreads, 0, s>>>(all, step);
    DRONE_HIP_TRY(hipGetLastError());
    return DRONE_OK;
}
bool sums_fit(const drone_step_tensor *t, const drone_step_sums *sums, int tensors)
{
    for (int i = 0; sums && i < tensors; ++i)
        if (sums[i].splits > 0 && t[i].n > 0 && !sums[i].sums) return false;
    return true;
}
}  // namespace

extern "C" int drone_sgd_steps_f32(const drone_step_tensor *t, int tensors, float lr, drone_stream_t stream)
{
    return drone_sgd_steps_sums_f32(t, nullptr, tensors, lr, stream);
}

extern "C" int drone_sgd_steps_sums_f32(const drone_step_tensor *t, const drone_step_sums *sums, int tensors, float lr, drone_stream_t stream)
{
    clear_error();
    DRONE_REQUIRE(t && tensors >= 1 && tensors <= kStepTensors, "tensors");
    for (int i = 0; i < tensors; ++i) DRONE_REQUIRE(t[i].n >= 0 && (t[i].n == 0 || (t[i].w && t[i].grad)), "null operand");
    DRONE_REQUIRE(sums_fit(t, sums, tensors), "null sums");
    return launch_steps(t, sums, tensors, SgdStep{lr}, as_stream(stream));
}

extern "C" int drone_sgd_step_f32(float *w, const float *g, int64_t n, float lr, drone_stream_t stream)
{
    const drone_step_tensor t{w, g, nullptr, nullptr, n, 0};
    return drone_sgd_steps_f32(&t, 1, lr, stream);
}

// cuda_module.cu:590-600: step_count is the value after the increment.
extern "C" int drone_adam_steps_f32(const drone_step_tensor *t, int tensors, float weight_decay, float lr, float beta1,
                                    float beta2, float eps, int step_count, drone_stream_t stream)
{
    return drone_adam_steps_sums_f32(t, nullptr, tensors, weight_decay, lr, beta1, beta2, eps, step_count, stream);
}

extern "C" int drone_adam_steps_sums_f32(const drone_step_tensor *t, const drone_step_sums *sums, int tensors, float weight_decay, float lr,
                                         float beta1, float beta2, float eps, int step_count, drone_stream_t stream)
{
    clear_error();
    DRONE_REQUIRE(t && tensors >= 1 && tensors <= kStepTensors && step_count >= 1, "tensors / step_count");
    for (int i = 0; i < tensors; ++i)
        DRONE_REQUIRE(t[i].n >= 0 && (t[i].n == 0 || (t[i].w && t[i].grad && t[i].m && t[i].v)), "operands");
    const float step_size = lr * sqrtf(1 - powf(beta2, (float)step_count)) / (1 - powf(beta1, (float)step_count));
    DRONE_REQUIRE(sums_fit(t, sums, tensors), "null sums");
    return launch_steps(t, sums, tensors, AdamStep{weight_decay, beta1, beta2, eps, step_size}, as_stream(stream));
}

extern "C" int drone_adam_step_f32(float *w, const float *g, float *m, float *v, int64_t n, int decay,
                                   float weight_decay, float lr, float beta1, float beta2, float eps, int step_count,
                                   drone_stream_t stream)
{
    const drone_step_tensor t{w, g, m, v, n, decay};
    return drone_adam_steps_f32(&t, 1, weight_decay, lr, beta1, beta2, eps, step_count, stream);
}

extern "C" int drone_fill_f32(float *x, int64_t n, float value, drone_stream_t stream)
{
    clear_error();
    DRONE_REQUIRE(n >= 0 && (n == 0 || x), "null operand");
    if (n == 0) return DRONE_OK;
    fill_f32_kernel<<<grid_for(n), kThreads, 0, as_stream(stream)>>>(x, n, value);
    DRONE_HIP_TRY(hipGetLastError());
    return DRONE_OK;
}
