// Products with A transposed, C (M x N) = alpha * A^T * B + beta * C, A stored K x M and B stored K x N: the weight gradients
// of cuda_gcn's CUDAMatmul (cuda_module.cu:92-105), whose reduction runs over the vertices and whose output is small.
//
// Both operands come straight from memory into matrix-core registers (DirectOperand, gemm_direct.h): a lane reads up to four
// consecutive columns of a row.  A work-group is four wavefronts, one per SIMD; they share a block of MT x NT tiles of 16 x 16 and
// split its rows, and add their blocks in wavefront order through LDS.  What it took:
//  * Work-groups go round the eight XCDs, so that blocks of the same rows, which are neighbours in launch order, each fetched these
//    rows into another XCD's L2: 1.2 M lines over the fabric per product of 320 x 100 over 30,720 rows where 0.42 M suffice.  Now an XCD gets a
//    contiguous run of (split, block), and reads a row once.
//  * One wavefront a SIMD: with two the same loops, which then issue the same loads and matrix instructions in all, take 1.6 times as long
//    (18.8 / 30.8 us per 30,720 rows of 320 x 100; the matrix instructions alone 17.3).
//  * With the rows in the L2 a block may be small, which leaves few splits and partial sums: 6 of 32 x 32 blocks against 25 of 64 x 64.
//  * Three groups of 16 rows in flight (two: 5 % slower on blocks of up to 8 tiles), two of the larger blocks, as the registers allow.
// us with the sum of the splits, before (four kernels, the reduction of a block shared by 8 or 16 wavefronts, or staged through LDS) / now: 320 x 100
// over 30,011 rows 36.6 / 32.2, 1,536 x 64 over 2,708 17.2 / 12.4, 480 x 40 over 189,106 148 / 96, 128 x 41 over 232,965 47 / 36,
// 640 x 128 over 232,965 324 / 297, 62 x 8 over 71,791 17.8 / 9.7, 100 x 50 over 45,000 25.2 / 14.7, 602 x 300 over 100,000 432 / 316, 1,000 x
// 1,000 over 5,000 106 / 94; 94 shapes, mostly of two-layer models, 1.27 times as fast in the mean.  Bound by the matrix pipe and by the L1, which
// overlap in part (the estimate below); small ones by a launch and a few round trips.
//
// Sums: a wavefront's matrix instructions add row after row to one accumulator, whose rounding errors grow with the length of such a chain.  Every
// 16, 48 or 64 rows the accumulators are added to a second set and the next chain starts from zero; in blocks of 32 tiles, whose loop is not unrolled
// that far, every 384 rows, as a pass of its own that takes a 100th of their matrix instructions' time.  (These blocks had one chain of all rows of a split's
// quarter, 2,336 for 640 x 128 over 232,965, and three groups in flight, of which the second set leaves two: 310 / 297 us, and with the second set in
// LDS 321).  Error against double, before / now, normal operands: 2.4e-7 / 1.7e-7, 1.6e-7 / 1.5e-7, 5.0e-7 / 1.8e-7, 2.6e-7 / 1.8e-7, 8.6e-7 / 3.6e-7, 1.9e-7 / 1.4e-7,
// 1.8e-7 / 1.6e-7, 9.7e-7 / 3.6e-7, 4.5e-7 / 1.7e-7 for the shapes above; 1,358 x 235 over 73,123 1.0e-6 / 3.6e-7, operands of one sign 1.8e-7 / 4.9e-8.
#pragma once
#include "gemm_direct.h"

namespace drone {
namespace {

constexpr int kGradWaves = 4;
constexpr int grad_depth(int tiles) { return tiles >= 16 ? 2 : 3; }  // groups of 16 rows in flight, as the registers allow
constexpr int grad_waves(int tiles) { return tiles <= 16 ? 2 : 1; }   // a SIMD, as the registers allow
constexpr int kGradXcds = 8;
constexpr int kGradChain = 24;  // groups a chain in blocks of 32 tiles

// (Registers for two wavefronts a SIMD where they suffice: with more of them the compiler keeps the sums in accumulation registers, and adding to
// them takes three instructions.)
template <int MT, int NT>
__global__ __launch_bounds__(kGradWaves * kWave) __attribute__((amdgpu_waves_per_eu(grad_waves(MT * NT), grad_waves(MT * NT)))) void
sgemm_grad_kernel(int M, int N, int K, float alpha, const float *__restrict__ A, int lda, const float *__restrict__ B, int ldb, float beta,
                  float *__restrict__ C, int ldc, int k_chunk, int splits, float *__restrict__ partial)
{
    constexpr int RP = 16 * MT, CP = 16 * NT, D = grad_depth(MT * NT);
    constexpr bool kShortChains = MT * NT <= 16;  // which end inside a round of the unrolled loop
    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int x = lane & 15, q = lane >> 4;
    // work-group blockIdx.x runs on XCD blockIdx.x % 8, which takes `per` consecutive (split, block)
    const int col_blocks = (N + CP - 1) / CP, blocks = (M + RP - 1) / RP * col_blocks;
    const int per = (blocks * splits + kGradXcds - 1) / kGradXcds;
    const int at = (int)(blockIdx.x % kGradXcds) * per + (int)(blockIdx.x / kGradXcds);
    if (at >= blocks * splits) return;  // the whole work-group
    const int split = at / blocks, block = at - split * blocks;
    const int m0 = block / col_blocks * RP, n0 = block % col_blocks * CP;
    const int kb = split * k_chunk, ke = kb + k_chunk < K ? kb + k_chunk : K;
    direct_f4 acc[MT][NT], sum[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[i][t] = sum[i][t] = direct_f4{0.0f, 0.0f, 0.0f, 0.0f};
    DirectOperand<MT, false> oa;
    DirectOperand<NT, false> ob;
    oa.init(A, lda, m0, M, x, q);
    ob.init(B, ldb, n0, N, x, q);
    // first: the group starts a chain (an accumulator of zeros is a constant to the instruction)
    const auto multiply = [&](const float (&a)[MT][4], const float (&b)[NT][4], bool first) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int t = 0; t < NT; ++t)
                    acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][j], b[t][j], first && j == 0 ? direct_f4{0.0f, 0.0f, 0.0f, 0.0f} : acc[i][t], 0, 0, 0);
    };
    const auto end_chain = [&]() {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int t = 0; t < NT; ++t) sum[i][t] += acc[i][t];
    };
    // whole groups of 16 rows are dealt out evenly to the wavefronts, the partial group goes to the last of them
    const int groups = (ke - kb) / 16;
    const int g0 = (int)((long long)groups * wave / kGradWaves), g1 = (int)((long long)groups * (wave + 1) / kGradWaves);
    float a[D][MT][4], b[D][NT][4];
    const auto reduce = [&](auto length) {  // of a chain, in groups
        constexpr int kRound = kShortChains ? (D + decltype(length)::value - 1) / decltype(length)::value * decltype(length)::value : D;
        const auto starts = [](int r) { return kShortChains && r % decltype(length)::value == 0; };
        const auto fetch = [&](int d, int g) {  // the last group once more instead of one behind it
            oa.load(kb + 16 * (g < g1 ? g : g1 - 1), a[d]);
            ob.load(kb + 16 * (g < g1 ? g : g1 - 1), b[d]);
        };
#pragma unroll
        for (int d = 0; d < D; ++d) fetch(d, g0 + d);
        static_assert(kRound % D == 0 && kGradChain % D == 0, "a group's registers are the same in every round");
        int g = g0;
        const auto round = [&]() {
#pragma unroll
            for (int r = 0; r < kRound; ++r) {
                // (the barriers keep the compiler from moving a group's loads down to their use)
                __builtin_amdgcn_sched_barrier(0);
                multiply(a[r % D], b[r % D], starts(r));
                __builtin_amdgcn_sched_barrier(0);
                fetch(r % D, g + r + D);
                if (starts(r + 1)) end_chain();
            }
        };
        if constexpr (kShortChains) {
            for (; g + kRound <= g1; g += kRound) round();
        } else {
            while (g + kRound <= g1) {
                const int end = g + kGradChain < g1 ? g + kGradChain : g1;
                for (; g + kRound <= end; g += kRound) round();
                end_chain();
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int t = 0; t < NT; ++t) acc[i][t] = direct_f4{0.0f, 0.0f, 0.0f, 0.0f};
            }
        }
#pragma unroll
        for (int r = 0; r < kRound; ++r)
            if (g + r < g1) {
                multiply(a[r % D], b[r % D], starts(r));
                if (r + D < kRound) fetch(r % D, g + r + D);
                if (kShortChains && (starts(r + 1) || g + r + 1 == g1)) end_chain();
            }
    };
    // A short chain is a group where a wavefront has a dozen of them or fewer, else three or four, whose end takes a twentieth of the time of
    // their matrix instructions.
    if (g0 < g1) {
        constexpr int kChain = D == 2 ? 4 : 3, kShort = MT * NT <= 8 ? 1 : kChain;
        if (kShort < kChain && g1 - g0 <= 12) reduce(std::integral_constant<int, kShort>());
        else reduce(std::integral_constant<int, kChain>());
    }
    if (wave == kGradWaves - 1 && kb + 16 * groups < ke) {
        oa.load_tail(kb + 16 * groups, ke, q, a[0]);
        ob.load_tail(kb + 16 * groups, ke, q, b[0]);
        multiply(a[0], b[0], kShortChains);
        if (kShortChains) end_chain();
    }
    if (!kShortChains) end_chain();
    extern __shared__ float s_tile[];  // [wavefront][MT * NT][4][64]: the sums as they lie
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) s_tile[((wave * MT * NT + i * NT + t) * 4 + v) * kWave + lane] = sum[i][t][v];
    __syncthreads();
    // Register v of lane x + 16 q of tile (i, t) is row position 4 q + v and column position x of the tile.  Columns fastest, so
    // that C is written in runs of consecutive lanes.
    float *out = partial ? partial + (size_t)split * M * N : C;
    const int ldo = partial ? N : ldc;
    for (int c = threadIdx.x; c < RP * CP; c += kGradWaves * kWave) {
        const int row = m0 + c / CP, col = n0 + c % CP;
        if (row >= M || col >= N) continue;
        int i, xr, t, xc;
        direct_place<MT, false>(m0, M, row, i, xr);
        direct_place<NT, false>(n0, N, col, t, xc);
        const int from = ((i * NT + t) * 4 + xr % 4) * kWave + (xr / 4) * 16 + xc;
        float total = 0.0f;
#pragma unroll
        for (int k = 0; k < kGradWaves; ++k) total += s_tile[k * MT * NT * 4 * kWave + from];
        float *dst = out + (size_t)row * ldo + col;
        if (!partial) {
            total *= alpha;
            if (beta != 0.0f) total += beta * *dst;
        }
        *dst = total;
    }
}

// How the output is cut into blocks of mt x nt tiles, and the reduction into splits: the cheapest of the instances by an estimate that
// was fitted to 84 products (8 to 1,500 rows of output, 2 to 300 columns, reductions of 300 to 233,000 rows).  Its choice takes 2 %
// longer than the best instance in the mean.
struct GradShape {
    int mt, nt, splits, k_chunk;
};
GradShape grad_shape(int M, int N, int K)
{
    static constexpr int kInstances[][2] = {{1, 1}, {2, 1}, {1, 2}, {2, 2}, {4, 3}, {4, 4}, {8, 2}, {8, 4}};
    constexpr int kGroups = 256;     // a work-group per CU
    constexpr int kLeastRows = 256;  // of a split: four groups of 16 a wavefront (46 x 2 over 7,306 rows in 114 splits 7.3 us, in 28 6.9)
    GradShape best{0, 0, 0, 0};
    double least = 0.0;
    for (const auto &tiles : kInstances) {
        const int mt = tiles[0], nt = tiles[1];
        // no block of which half lies outside (a lane's piece of up to four columns then fits the rows), and a single tile only where it does
        if (mt * nt == 1 ? M > 16 && N > 16 : (mt > 1 && 16 * mt >= M + 8 * mt) || (nt > 1 && 16 * nt >= N + 16)) continue;
        const int64_t blocks = ceil_div(M, 16 * mt) * ceil_div(N, 16 * nt);
        int splits = (int)std::max<int64_t>(1, std::min<int64_t>(kGroups / blocks, K / kLeastRows));
        const int k_chunk = (int)ceil_div(ceil_div(K, splits), 16) * 16;
        splits = (int)ceil_div(K, k_chunk);
        // us: a wavefront's matrix instructions and what a group of rows costs besides, the work-group's bytes through the L1 (64 a
        // clock, partly behind them), the wavefronts' sums through LDS, and partial sums (written, read again in another launch)
        const double rounds = (double)ceil_div(blocks * splits, kGroups), groups = (double)ceil_div(k_chunk / 16, kGradWaves);
        const double clocks = groups * (mt * nt * 4 * 32 + 180) + 0.7 * (double)k_chunk * (mt + nt);
        const double us = rounds * (clocks / 2400.0 + 0.3 * mt * nt) + (splits > 1 ? 2.3 + 3.5e-6 * splits * (double)M * N : 0.0);
        if (best.mt == 0 || us < least) {
            least = us;
            best = GradShape{mt, nt, splits, k_chunk};
        }
    }
    return best;
}

template <int MT, int NT>
void launch_grad(const GradShape &g, int M, int N, int K, float alpha, const float *A, int lda, const float *B, int ldb, float beta, float *C,
                 int ldc, float *partial, hipStream_t s)
{
    const int64_t all = ceil_div(M, 16 * MT) * ceil_div(N, 16 * NT) * g.splits;
    sgemm_grad_kernel<MT, NT><<<(unsigned)(ceil_div(all, kGradXcds) * kGradXcds), kGradWaves * kWave, sizeof(float) * kGradWaves * MT * NT * 4 * kWave, s>>>(
        M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, g.k_chunk, g.splits, partial);
}
// partial: null where there is one split.
void sgemm_grad(const GradShape &g, int M, int N, int K, float alpha, const float *A, int lda, const float *B, int ldb, float beta, float *C,
                int ldc, float *partial, hipStream_t s)
{
    const auto go = [&](auto mt, auto nt) {
        if (g.mt == decltype(mt)::value && g.nt == decltype(nt)::value)
            launch_grad<decltype(mt)::value, decltype(nt)::value>(g, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, partial, s);
    };
#define DRONE_GRAD(MT_, NT_) go(std::integral_constant<int, MT_>(), std::integral_constant<int, NT_>());
    DRONE_GRAD(1, 1)
    DRONE_GRAD(2, 1)
    DRONE_GRAD(1, 2)
    DRONE_GRAD(2, 2)
    DRONE_GRAD(4, 3)
    DRONE_GRAD(4, 4)
    DRONE_GRAD(8, 2)
    DRONE_GRAD(8, 4)
#undef DRONE_GRAD
}

}  // namespace
}  // namespace drone
