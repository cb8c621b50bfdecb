// C (M x N) = alpha * A * op(B) for short rows on both sides (K <= 64, N <= 128) and many of them: the class-wide products of the model,
// H1 W2 and dT2 W2^T.  What bounds them is memory, mostly C.
//
// op(B) goes through LDS into registers once per work-group, in the order in which the lanes of v_mfma_f32_16x16x4_f32 want it, and stays there; a
// wavefront walks over strips of 16 rows with the next strip's rows in flight and leaves each in pieces of up to 16 bytes a lane: tile t of a
// piece of four holds columns 4 x + t, so a lane's four sums of a row are neighbours.  The tiled kernel, which had most of these, waits at barriers for
// single depth-32 steps and writes 4 bytes a lane; the direct one reads op(B) from L2 once per 16 or 32 rows.
//
// us before / here: 227,087 x 13 x 50 29.3 / 15.3 (4.0 TB/s), 227,087 x 3 x 120 47 / 28, 71,791 x 13 x 50 14.7 / 7.8, 30,011 x 16 x 41 7.3 / 4.4, 211,549 x 4 x 30
// 23.4 / 9.4, 227,087 x 50 x 7 25.6 / 15.3; 114 products of its range and around it 1.17 times as fast, and 30,011 x 23 x 100 in a training step 10.9 / 8.7.  Every
// wavefront loading op(B) for itself: 227,087 x 62 x 81 57 instead of 42.  Eight wavefronts a work-group: 5 % slower below 16,000 rows and with long op(B), 2 %
// faster in between.  1,024 work-groups are 7 % better than 512 for one group of 16 steps and 10 % worse for more.  With a beta the other kernels serve.
//
// Sums: in the order of the kernel that it stands in for, bit by bit, as in gemm_strip.h.
#pragma once
#include "gemm_strip.h"

namespace drone {
namespace {

constexpr int kFlatWaves = 4, kFlatMost = 24;  // kFlatMost: groups of steps times tiles are fewer

template <int KG, int NT>
__global__ __launch_bounds__(kFlatWaves * kWave) void sgemm_flat_kernel(int M, int N, int K, bool ascending, float alpha, const float *__restrict__ A,
                                                                   int lda, const float *__restrict__ B, int b_step, int b_col,
                                                                   float *__restrict__ C, int ldc)
{
    __shared__ direct_f4 s_b[KG * NT * kWave];  // op(B): [group][tile][lane]
    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), x = lane & 15, q = lane >> 4;
    const int strips = (int)(((int64_t)M + 15) / 16), waves = gridDim.x * kFlatWaves;
    const int whole = K / 16;                      // KG, or KG - 1 and a partial group
    const int past = 16 * whole + 4 * q + 4 - K;   // how far this lane's piece of the partial group reaches past the row: it slides back
    direct_f4 a[KG];
    const auto fetch = [&](int s) {
        const int64_t r = (int64_t)s * 16 + x;
        const float *row = A + (size_t)(r < M ? r : M - 1) * lda;
        const auto load4 = [&](int k) {
            const DirectF4U v = *reinterpret_cast<const DirectF4U *>(row + k);
            return direct_f4{v.v[0], v.v[1], v.v[2], v.v[3]};
        };
#pragma unroll
        for (int g = 0; g < KG; ++g) {
            if (g < KG - 1 || whole == KG) a[g] = load4(16 * g + 4 * q);
            else if (K >= 4) a[g] = load4(16 * g + 4 * q - (past > 0 ? past : 0));
            else a[g] = direct_f4{row[0], row[K > 1 ? 1 : 0], row[K - 1], 0.0f};
        }
    };
    int s = blockIdx.x * kFlatWaves + wave;
    if (s < strips) fetch(s);  // in flight while op(B) comes
    for (int i = wave; i < KG * NT; i += kFlatWaves) {
        const int g = i / NT, t = i - g * NT;
        const int w = direct_piece_width(NT, t), first = direct_piece_first(NT, t);  // as in direct_outer
        const int nominal = 16 * first + w * x, n = (nominal + w <= N ? nominal : N - w) + t - first;
        const float *src = B + (size_t)n * b_col;
        direct_f4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int k = 16 * g + (ascending ? 4 * j + q : 4 * q + j);
            const float e = src[(size_t)(k < K ? k : K - 1) * b_step];
            v[j] = k < K ? e : 0.0f;
        }
        s_b[i * kWave + lane] = v;
    }
    __syncthreads();
    direct_f4 b[KG][NT];
#pragma unroll
    for (int g = 0; g < KG; ++g)
#pragma unroll
        for (int t = 0; t < NT; ++t) b[g][t] = s_b[(g * NT + t) * kWave + lane];
    for (; s < strips; s += waves) {
        direct_f4 acc[NT], now[KG];
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = direct_f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int g = 0; g < KG; ++g) now[g] = a[g];
        if (s + waves < strips) fetch(s + waves);
#pragma unroll
        for (int g = 0; g < KG; ++g) {
            direct_f4 v = now[g];
            if (g == KG - 1 && whole < KG) {  // zeros past the row
                if (K >= 4) {
                    if (past > 0) {
                        if (past & 1) v = direct_f4{v[1], v[2], v[3], 0.0f};
                        if (past & 2) v = direct_f4{v[2], v[3], 0.0f, 0.0f};
                        if (past >= 4) v = direct_f4{0.0f, 0.0f, 0.0f, 0.0f};
                    }
                } else {
#pragma unroll
                    for (int j = 0; j < 3; ++j) v[j] = q == 0 && j < K ? v[j] : 0.0f;
                }
            }
            if (ascending) v = strip_ascending(v);
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[j], b[g][t][j], acc[t], 0, 0, 0);
        }
        // register v of lane x + 16 q of a tile is row 4 q + v; a piece of w tiles is w columns in a row, and only the last piece can reach past N
        int at_row = 4 * q;
        asm volatile("" : "+v"(at_row));  // keeps the compiler from holding an address per row and column (100 registers)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int64_t r = (int64_t)s * 16 + (at_row + v);
            if (r >= M) continue;
            float *dst = C + (size_t)r * ldc;
#pragma unroll
            for (int t = 0; t < NT;) {
                const int w = direct_piece_width(NT, t), first = 16 * t + w * x;
                const auto at = [&](int i) { return alpha * acc[t + i < NT ? t + i : t][v]; };
                if (t + w < NT || first + w <= N) {
                    if (w == 4) *reinterpret_cast<DirectF4U *>(dst + first) = DirectF4U{at(0), at(1), at(2), at(3)};
                    else if (w == 2) *reinterpret_cast<DirectF2U *>(dst + first) = DirectF2U{at(0), at(1)};
                    else dst[first] = at(0);
                } else if (first < N) {  // the piece begins at column N - w
#pragma unroll
                    for (int i = 1; i < w; ++i)
                        if (N - w + i >= first) dst[N - w + i] = at(i);
                }
                t += w;
            }
        }
    }
}

// Instead of the tiled kernel from 8,000 rows on (us by it / here: 9,110 x 7 x 116 7.1 / 4.8, 14,976 x 10 x 110 7.2 / 5.3, below that 6,054 x 5 x 109 4.2 / 4.7),
// instead of the direct or the strip kernel from 24,000 (26,727 x 46 x 46 7.3 / 5.7, 29,188 x 38 x 40 6.7 / 6.0; 18,665 x 55 x 49 7.6 / 8.0, 10,190 x 2 x 54
// 4.1 / 4.3).  Not where op(B) asks for more registers than leave two work-groups a CU (60,507 x 62 x 81 16.6 / 18.7, 209,407 x 42 x 105 42.8 / 44.5, but
// 104,863 x 41 x 83 22.9 / 20.3), and single tiles of whole groups are the direct kernel's best case (42,244 x 16 x 13 3.4 / 3.8).
bool flat_covers(bool tiled, int M, int N, int K)
{
    if (K < 1 || K > 64 || N > 128) return false;
    const int n16 = (int)ceil_div(N, 16), tiles = n16 <= 4 ? n16 : n16 <= 6 ? 6 : 8;
    if (ceil_div(K, 16) * tiles >= kFlatMost) return false;
    return tiled ? M >= 8000 : M >= 24000 && !(K % 16 == 0 && N <= 16);
}

template <int KG>
void launch_flat(bool tb, bool ascending, int M, int N, int K, float alpha, const float *A, int lda, const float *B, int ldb, float *C, int ldc,
                 hipStream_t s)
{
    const unsigned grid = (unsigned)std::min<int64_t>(KG == 1 ? 1024 : 512, ceil_div(ceil_div(M, 16), kFlatWaves));
    const int n16 = (int)ceil_div(N, 16);
    const auto go = [&](auto tiles) {
        constexpr int NT = decltype(tiles)::value;
        if constexpr (KG * NT < kFlatMost)
            sgemm_flat_kernel<KG, NT><<<grid, kFlatWaves * kWave, 0, s>>>(M, N, K, ascending, alpha, A, lda, B, tb ? 1 : ldb, tb ? ldb : 1, C, ldc);
    };
    if (n16 == 1) go(std::integral_constant<int, 1>());
    else if (n16 == 2) go(std::integral_constant<int, 2>());
    else if (n16 == 3) go(std::integral_constant<int, 3>());
    else if (n16 == 4) go(std::integral_constant<int, 4>());
    else if (n16 <= 6) go(std::integral_constant<int, 6>());
    else go(std::integral_constant<int, 8>());
}
void sgemm_flat(bool tb, bool ascending, int M, int N, int K, float alpha, const float *A, int lda, const float *B, int ldb, float *C, int ldc,
                hipStream_t s)
{
    const int kg = (int)ceil_div(K, 16);
    if (kg == 1) launch_flat<1>(tb, ascending, M, N, K, alpha, A, lda, B, ldb, C, ldc, s);
    else if (kg == 2) launch_flat<2>(tb, ascending, M, N, K, alpha, A, lda, B, ldb, C, ldc, s);
    else if (kg == 3) launch_flat<3>(tb, ascending, M, N, K, alpha, A, lda, B, ldb, C, ldc, s);
    else launch_flat<4>(tb, ascending, M, N, K, alpha, A, lda, B, ldb, C, ldc, s);
}

}  // namespace
}  // namespace drone
