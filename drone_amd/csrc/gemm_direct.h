// fp32 products whose tiles would not fill the GPU: operands straight from memory into matrix-core registers.
//
// v_mfma_f32_16x16x4_f32 retires 64 multiply-adds per clock and SIMD, so a wavefront that holds an MT x NT block of 16 x 16
// tiles needs (MT + NT) / (MT * NT) KB per 32 clocks from L1 / L2 - little enough to leave LDS staging, its barriers and its
// 128-row tiles out.  What that buys is parallelism: a wavefront owns 16 (32) rows instead of a work-group 128, and the
// KS wavefronts of a work-group share one output block by splitting the reduction, adding their blocks in wavefront order
// through LDS.  A 2,708 x 1,433 x 64 layer product ran as 22 tiles of the tiled kernel on 22 of 256 CUs (66 us; here 12.5),
// 1,000 x 608 x 128 56 -> 7.  (Weight gradients: gemm_grad.h.)  Small
// products are bound by their chain of loads, mid-size ones by the L2 -> L1 traffic above (70 - 80 TFLOP/s), which is why
// large ones stay with the tiled kernel (100 - 130).
//
// Operand layouts.  Lane l = x + 16 q of a wavefront holds, for matrix instruction j of a group of 16 reduction steps, the
// elements of op(A) / op(B) at step k0 + 4 q + j.  An operand whose reduction index is contiguous in memory comes with one
// 16-byte load per tile and group (row 16 t + x, steps k0 + 4 q ..+ 3); one whose outer index is contiguous comes with
// loads of w = 4 / 2 / 1 floats per step, which feed w tiles: outer indices base + w x + i for tile i.  A lane whose piece
// would reach past the matrix slides back to the last whole piece: it then multiplies elements that another lane owns,
// and stores none of those (no masks, no reads past a row's end).  Only the reduction's last, partial group is guarded
// element by element.
#pragma once
#include "common.h"

namespace drone {
namespace {

typedef float direct_f4 __attribute__((ext_vector_type(4)));
struct alignas(4) DirectF4U { float v[4]; };
struct alignas(4) DirectF2U { float v[2]; };

// Where tile t of an outer-contiguous operand sits: the tiles are taken in pieces of 4, 2 and 1.
constexpr int direct_piece_width(int tiles, int t) { return t < tiles / 4 * 4 ? 4 : t < tiles / 2 * 2 ? 2 : 1; }
constexpr int direct_piece_first(int tiles, int t) { return t < tiles / 4 * 4 ? t / 4 * 4 : t < tiles / 2 * 2 ? t / 2 * 2 : t; }

// Outer index of (tile t, lane position x), and whether that lane owns it.
template <int TILES, bool K_CONTIG>
__device__ __forceinline__ int direct_outer(int base, int end, int t, int x, bool &own)
{
    if constexpr (K_CONTIG) {
        const int o = base + 16 * t + x;
        own = o < end;
        return o < end ? o : end - 1;
    } else {
        const int w = direct_piece_width(TILES, t), first = direct_piece_first(TILES, t);
        const int nominal = base + 16 * first + w * x;
        const int start = nominal + w <= end ? nominal : end - w;
        const int o = start + (t - first);
        own = o >= nominal && o < end;
        return o;
    }
}

// The other way round: the tile and lane position that hold outer index o of the block at `base` (base <= o < end).
template <int TILES, bool K_CONTIG>
__device__ __forceinline__ void direct_place(int base, int end, int o, int &t, int &x)
{
    const int p = o - base;
    if constexpr (K_CONTIG) {
        t = p / 16;
        x = p % 16;
    } else {
        constexpr int f2 = TILES / 4 * 4, f1 = TILES / 2 * 2;
        const int first = p < 16 * f2 ? p / 64 * 4 : p < 16 * f1 ? f2 + (p - 16 * f2) / 32 * 2 : f1 + (p - 16 * f1) / 16;
        const int w = p < 16 * f2 ? 4 : p < 16 * f1 ? 2 : 1;
        x = (p - 16 * first) / w;
        const int nominal = base + 16 * first + w * x;
        const int start = nominal + w <= end ? nominal : end - w;
        t = first + (o - start);
    }
}

template <int TILES, bool K_CONTIG>
struct DirectOperand {
    const float *at[K_CONTIG ? TILES : (TILES / 4 + (TILES % 4) / 2 + TILES % 2)];
    int ld;
    // base: first outer index of the block; end: extent of the outer dimension; q: the lane's quarter of a group
    __device__ __forceinline__ void init(const float *p, int ld_, int base, int end, int x, int q)
    {
        ld = ld_;
        bool own;
        if constexpr (K_CONTIG) {
#pragma unroll
            for (int t = 0; t < TILES; ++t)
                at[t] = p + (size_t)direct_outer<TILES, true>(base, end, t, x, own) * ld + 4 * q;
        } else {
            int piece = 0;
#pragma unroll
            for (int t = 0; t < TILES; t += direct_piece_width(TILES, t))
                at[piece++] = p + (size_t)(4 * q) * ld + direct_outer<TILES, false>(base, end, t, x, own);
        }
    }
    // v[t][j]: tile t, matrix instruction j, of the group that starts at step k0
    __device__ __forceinline__ void load(int k0, float (&v)[TILES][4]) const
    {
        if constexpr (K_CONTIG) {
#pragma unroll
            for (int t = 0; t < TILES; ++t) {
                const DirectF4U r = *reinterpret_cast<const DirectF4U *>(at[t] + k0);
#pragma unroll
                for (int j = 0; j < 4; ++j) v[t][j] = r.v[j];
            }
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                int piece = 0;
#pragma unroll
                for (int t = 0; t < TILES;) {
                    const float *src = at[piece++] + (size_t)(k0 + j) * ld;
                    const int w = direct_piece_width(TILES, t);
                    if (w == 4) {
                        const DirectF4U r = *reinterpret_cast<const DirectF4U *>(src);
#pragma unroll
                        for (int i = 0; i < 4; ++i) v[t + (i < TILES - t ? i : 0)][j] = r.v[i];
                    } else if (w == 2) {
                        const DirectF2U r = *reinterpret_cast<const DirectF2U *>(src);
                        v[t][j] = r.v[0];
                        v[t + (t + 1 < TILES ? 1 : 0)][j] = r.v[1];
                    } else {
                        v[t][j] = *src;
                    }
                    t += w;
                }
            }
        }
    }
    // the same for a group that reaches past step k_end: zeros there, nothing read past the matrix
    __device__ __forceinline__ void load_tail(int k0, int k_end, int q, float (&v)[TILES][4]) const
    {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const bool live = k0 + 4 * q + j < k_end;
            // a step past the end reads the lane's element of step k_end - 1 instead and counts it as zero
            const int back = live ? 0 : k0 + 4 * q + j - (k_end - 1);
            int piece = 0;
#pragma unroll
            for (int t = 0; t < TILES;) {
                if constexpr (K_CONTIG) {
                    const float r = at[t][k0 + j - back];
                    v[t][j] = live ? r : 0.0f;
                    ++t;
                } else {
                    const float *src = at[piece++] + ((ptrdiff_t)(k0 + j) - back) * ld;
                    const int w = direct_piece_width(TILES, t);
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (i < w && t + i < TILES) v[t + i][j] = live ? src[i] : 0.0f;
                    t += w;
                }
            }
        }
    }
};

// C (M x N) = alpha A op(B) + beta C.  A work-group owns MT x NT tiles of 16 x 16 per output block, its KS wavefronts a share of
// the reduction each (KS = 1: four wavefronts, an output block each).
template <int MT, int NT, bool B_K_CONTIG, int KS>
__global__ __launch_bounds__((KS > 4 ? KS : 4) * kWave) void sgemm_direct_kernel(int M, int N, int K, float alpha,
                                                                             const float *__restrict__ A, int lda,
                                                                             const float *__restrict__ B, int ldb,
                                                                             float beta, float *__restrict__ C, int ldc)
{
    constexpr int kWaves = KS > 4 ? KS : 4, kBlocks = kWaves / KS;
    constexpr int RP = 16 * MT, CP = 16 * NT;
    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int x = lane & 15, q = lane >> 4;
    const int share = wave % KS, block = wave / KS;
    // column blocks of the same rows are neighbours in launch order: they read the same part of A
    const int col_blocks = (N + CP - 1) / CP, row_group = blockIdx.x / col_blocks;
    const int m0 = (row_group * kBlocks + block) * RP, n0 = (blockIdx.x - row_group * col_blocks) * CP;
    direct_f4 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[i][t] = direct_f4{0.0f, 0.0f, 0.0f, 0.0f};
    if (m0 < M) {  // the same for the whole wavefront
        DirectOperand<MT, true> oa;
        DirectOperand<NT, B_K_CONTIG> ob;
        oa.init(A, lda, m0, M, x, q);
        ob.init(B, ldb, n0, N, x, q);
        // whole groups of 16 steps are dealt out evenly to the KS wavefronts, the partial group goes to the last of them
        const int groups = K / 16;
        const int g0 = (int)((long long)groups * share / KS), g1 = (int)((long long)groups * (share + 1) / KS);
        const auto multiply = [&](const float (&a)[MT][4], const float (&b)[NT][4]) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int t = 0; t < NT; ++t)
                        acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][j], b[t][j], acc[i][t], 0, 0, 0);
        };
        float a0[MT][4], b0[NT][4], a1[MT][4], b1[NT][4];
        // (Two forms of one loop, which the compiler schedules differently.  The first is for deep reductions: 2,708 x 1,433 x 64 13.2 ->
        // 11.4 us, 5,000 x 1,400 x 128 32.3 -> 29.0; blocks of a wavefront of their own lose by it, 15,003 x 100 x 50 7.7 -> 11.4.)
        if constexpr (KS == 8) {
            if (g0 < g1) {
                const auto group = [&](int g) { return 16 * (g < g1 ? g : g1 - 1); };  // the last group again behind it
                oa.load(16 * g0, a0);
                ob.load(16 * g0, b0);
                for (int g = g0;;) {
                    bool over = false;
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        oa.load(group(g + 1), j == 0 ? a1 : a0);
                        ob.load(group(g + 1), j == 0 ? b1 : b0);
                        multiply(j == 0 ? a0 : a1, j == 0 ? b0 : b1);
                        if (++g >= g1) {
                            over = true;
                            break;
                        }
                    }
                    if (over) break;
                }
            }
        } else if (g0 < g1) {
            oa.load(16 * g0, a0);
            ob.load(16 * g0, b0);
            for (int g = g0;;) {
                // the last group is fetched once more instead of the one behind it
                int next = g + 1 < g1 ? g + 1 : g;
                oa.load(16 * next, a1);
                ob.load(16 * next, b1);
                multiply(a0, b0);
                if (++g >= g1) break;
                next = g + 1 < g1 ? g + 1 : g;
                oa.load(16 * next, a0);
                ob.load(16 * next, b0);
                multiply(a1, b1);
                if (++g >= g1) break;
            }
        }
        if (share == KS - 1 && 16 * groups < K) {
            oa.load_tail(16 * groups, K, q, a0);
            ob.load_tail(16 * groups, K, q, b0);
            multiply(a0, b0);
        }
    }
    const auto put = [&](int row, int col, float sum) {
        float *dst = C + (size_t)row * ldc + col;
        float r = alpha * sum;
        if (beta != 0.0f) r += beta * *dst;
        *dst = r;
    };
    // Register v of lane x + 16 q of tile (i, t) is row position 4 q + v and column position x of the tile.
    if constexpr (KS == 1) {
        if (m0 >= M) return;
        const bool wide = beta == 0.0f && ldc % 4 == 0 && (reinterpret_cast<uintptr_t>(C) & 15) == 0;
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                bool own_row;
                const int row = direct_outer<MT, true>(m0, M, i, 4 * q + v, own_row);
                if (!own_row) continue;
#pragma unroll
                for (int t = 0; t < NT;) {
                    const int w = B_K_CONTIG ? 1 : direct_piece_width(NT, t);
                    // four tiles of one piece: the lane holds four consecutive columns
                    const int first = n0 + 16 * t + 4 * x;
                    if (w == 4 && wide && first + 4 <= N) {
                        direct_f4 r;
#pragma unroll
                        for (int k = 0; k < 4; ++k) r[k] = alpha * acc[i][t + k < NT ? t + k : t][v];
                        *reinterpret_cast<direct_f4 *>(C + (size_t)row * ldc + first) = r;
                    } else {
#pragma unroll
                        for (int k = 0; k < 4; ++k)
                            if (k < w && t + k < NT) {
                                bool own;
                                const int col = direct_outer<NT, B_K_CONTIG>(n0, N, t + k, x, own);
                                if (own) put(row, col, acc[i][t + k][v]);
                            }
                    }
                    t += w;
                }
            }
    } else {
        extern __shared__ float s_tile[];  // [wavefront][MT * NT][4][64]: the accumulators as they lie
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int v = 0; v < 4; ++v) s_tile[((wave * MT * NT + i * NT + t) * 4 + v) * kWave + lane] = acc[i][t][v];
        __syncthreads();
        // columns fastest, so that C is written in runs of consecutive lanes
        for (int c = threadIdx.x; c < kBlocks * RP * CP; c += kWaves * kWave) {
            const int blk = c / (RP * CP), pr = (c / CP) % RP, pc = c % CP;
            const int row = (row_group * kBlocks + blk) * RP + pr, col = n0 + pc;
            if (row >= M || col >= N) continue;
            int i, xr, t, xc;
            direct_place<MT, true>((row_group * kBlocks + blk) * RP, M, row, i, xr);
            direct_place<NT, B_K_CONTIG>(n0, N, col, t, xc);
            const int at = ((i * NT + t) * 4 + xr % 4) * kWave + (xr / 4) * 16 + xc;
            float sum = 0.0f;
#pragma unroll
            for (int k = 0; k < KS; ++k) sum += s_tile[(blk * KS + k) * MT * NT * 4 * kWave + at];
            put(row, col, sum);
        }
    }
}

// The same sums for few blocks, at most one per CU: four wavefronts, one per SIMD, take two of the eight shares each, side by side, two groups of
// either in flight.  What bounds such a product is a wavefront's chain of loads and matrix instructions; two wavefronts on a SIMD take longer for
// the two shares than one that alternates between them, and their eight tiles' worth of independent sums hide the instructions' latency.
// us by the kernel above / here: 2,708 x 1,440 x 64 12.8 / 10.7, 376 x 1,201 x 112 10.5 / 4.9, 1,726 x 1,440 x 25 8.8 / 5.9, 3,986 x 1,104 x 68 18.2 / 13.0;
// over 68 shapes 1.13 times as fast.  Three groups of either in flight: 1.13 -> 1.08.  One share after the other instead: 2,708 x 1,440 x 64 12.9.
constexpr int kTwinWaves = 4, kTwinShares = 2 * kTwinWaves, kTwinBlocks = 256;

template <int NT, bool B_K_CONTIG>
__global__ __launch_bounds__(kTwinWaves * kWave) void sgemm_twin_kernel(int M, int N, int K, float alpha, const float *__restrict__ A, int lda,
                                                                   const float *__restrict__ B, int ldb, float beta,
                                                                   float *__restrict__ C, int ldc)
{
    constexpr int D = 2, CP = 16 * NT;
    extern __shared__ float s_sums[];  // [share][NT][4][64], as the accumulators lie
    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int x = lane & 15, q = lane >> 4;
    const int col_blocks = (N + CP - 1) / CP, row_group = blockIdx.x / col_blocks;
    const int m0 = row_group * 16, n0 = (blockIdx.x - row_group * col_blocks) * CP;
    direct_f4 acc[2][NT];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[h][t] = direct_f4{0.0f, 0.0f, 0.0f, 0.0f};
    DirectOperand<1, true> oa;
    DirectOperand<NT, B_K_CONTIG> ob;
    oa.init(A, lda, m0, M, x, q);
    ob.init(B, ldb, n0, N, x, q);
    const int groups = K / 16, share = 2 * wave;
    const auto begin_of = [&](int s) { return (int)((long long)groups * s / kTwinShares); };
    const int begin[2] = {begin_of(share), begin_of(share + 1)}, end[2] = {begin[1], begin_of(share + 2)};
    const auto multiply = [&](int h, const float (&a)[1][4], const float (&b)[NT][4]) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[h][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[0][j], b[t][j], acc[h][t], 0, 0, 0);
    };
    float a[D][2][1][4], b[D][2][NT][4];
    const auto fetch = [&](int d, int h, int i) {  // the last group again instead of one behind it
        const int g = begin[h] + i < end[h] ? begin[h] + i : end[h] - 1;
        oa.load(16 * g, a[d][h]);
        ob.load(16 * g, b[d][h]);
    };
    const int both = min(end[0] - begin[0], end[1] - begin[1]);  // >= 1
#pragma unroll
    for (int d = 0; d < D; ++d)
#pragma unroll
        for (int h = 0; h < 2; ++h) fetch(d, h, d);
    int i = 0;
    for (; i + D <= both; i += D) {
#pragma unroll
        for (int d = 0; d < D; ++d)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                __builtin_amdgcn_sched_barrier(0);
                multiply(h, a[d][h], b[d][h]);
                __builtin_amdgcn_sched_barrier(0);
                fetch(d, h, i + d + D);
            }
    }
#pragma unroll
    for (int d = 0; d < D; ++d)
#pragma unroll
        for (int h = 0; h < 2; ++h)
            if (i + d < end[h] - begin[h]) multiply(h, a[d][h], b[d][h]);
    if (wave == kTwinWaves - 1 && 16 * groups < K) {
        oa.load_tail(16 * groups, K, q, a[0][0]);
        ob.load_tail(16 * groups, K, q, b[0][0]);
        multiply(1, a[0][0], b[0][0]);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) s_sums[(((share + h) * NT + t) * 4 + v) * kWave + lane] = acc[h][t][v];
    __syncthreads();
    for (int c = threadIdx.x; c < 16 * CP; c += kTwinWaves * kWave) {
        const int row = m0 + c / CP, col = n0 + c % CP;
        if (row >= M || col >= N) continue;
        int t, xr, i_, xc;
        direct_place<1, true>(m0, M, row, i_, xr);
        direct_place<NT, B_K_CONTIG>(n0, N, col, t, xc);
        const int from = (t * 4 + xr % 4) * kWave + (xr / 4) * 16 + xc;
        float sum = 0.0f;
        for (int k = 0; k < kTwinShares; ++k) sum += s_sums[k * NT * 4 * kWave + from];
        float *dst = C + (size_t)row * ldc + col;
        float r = alpha * sum;
        if (beta != 0.0f) r += beta * *dst;
        *dst = r;
    }
}

}  // namespace
}  // namespace drone
