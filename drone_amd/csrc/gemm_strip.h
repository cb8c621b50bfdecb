// C (M x N) = alpha * A * op(B) + beta * C for many rows of A and a small op(B): the layer products of the model on mid-size and large graphs.
//
// op(B) sits in LDS as a whole (K x N up to 160 KB), in the order in which the lanes of v_mfma_f32_16x16x4_f32 read it, so the loop over
// the reduction has no barrier and reads it once per 16 rows with 16 bytes a lane; a wavefront owns 16 rows and all columns, padded to 16 and not
// to 64 or 128, and reads its rows straight from memory, 16 bytes a lane, four groups of 16 steps ahead.  What it took: the fetch of op(B)
// addressed by scalar registers, a wavefront a block of 16 x 16 at a time (one index per lane took 12 us for 140 KB, this 6), beginning at
// another place in every work-group, as all ask for the same lines at once; no branch for columns past op(B) (with N no multiple of 16 all blocks of the last tile,
// which are one wavefront's where there are eight tiles, took a path of single loads: 31,465 x 224 x 113 28.8 / 22.7); op(B) transposed by 16-byte loads for either order of
// sums (31,465 x 312 x 116 48.9 / 31.6, by the tiled kernel 31.0); and LDS reads a group ahead of the matrix instructions, kept there
// by scheduling barriers (21 -> 20 us per 32,768 rows of 320 x 100, of which the matrix instructions are 15).  Two strips a wavefront, 4, 12 or 16
// wavefronts, 8 groups ahead, op(B) by rows (four times the LDS instructions), one run of groups over the seams between strips: none better
// over 100 shapes, several worse.
//
// us by the kernels that it stands in for / here: 30,011 x 320 x 100 30.5 / 27.8, 64,530 x 96 x 93 27.2 / 19.5, 103,955 x 288 x 84 90 / 63, 121,197 x 192 x 38
// 39.5 / 28.7, 196,368 x 352 x 30 91 / 55, 208,773 x 576 x 62 187 / 147, 227,087 x 92 x 23 31.6 / 24.3, transposed 64,593 x 244 x 110 45.7 / 42.0; 680 shapes 1.32 times as fast in the
// mean, six slower by 2.5 to 5 % (mostly 38,000 to 49,000 rows, where the tiled kernel's rounds come out even, and its 128 columns are all used).  Bound by
// op(B)'s fetch (a launch and 7 us in front of 140 KB) on few rows, by memory (3.9 TB/s of A and C) or the matrix pipe on many.
//
// Sums: one accumulator per output takes the reduction's steps one after the other, as v_mfma_f32_16x16x4_f32 and v_mfma_f32_32x32x2_f32 both do (their
// sums are those of a chain of fused multiply-adds).  ASC: in ascending order, like the tiled kernel; else as the direct kernel's groups of 16 take
// them (steps 4 q + j, for j = 0 ... 3 the quarters q in turn).  The results are therefore those of the kernel it stands in for, bit by bit.
#pragma once
#include "gemm_direct.h"

namespace drone {
namespace {

constexpr int kStripWaves = 8, kStripDepth = 4, kStripGroups = 256;  // work-groups: one per CU
constexpr size_t kStripLds = 160 << 10;
inline size_t strip_lds(int N, int K) { return (size_t)ceil_div(K, 16) * (size_t)ceil_div(N, 16) * kWave * sizeof(direct_f4); }

// Lane x + 16 q holds steps 4 q + j of a group in component j, and is to hold steps 4 j + q: the transposition of (q, j).
__device__ __forceinline__ direct_f4 strip_ascending(direct_f4 a)
{
    const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(a[0]), __float_as_uint(a[2]), false, false);
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a[1]), __float_as_uint(a[3]), false, false);
    const auto s = __builtin_amdgcn_permlane16_swap(p[0], r[0], false, false);
    const auto t = __builtin_amdgcn_permlane16_swap(p[1], r[1], false, false);
    return direct_f4{__uint_as_float(s[0]), __uint_as_float(s[1]), __uint_as_float(t[0]), __uint_as_float(t[1])};
}

template <int NT, bool TB, bool ASC>
__global__ __launch_bounds__(kStripWaves * kWave) void sgemm_strip_kernel(int M, int N, int K, float alpha, const float *__restrict__ A, int lda,
                                                                      const float *__restrict__ B, int ldb, float beta,
                                                                      float *__restrict__ C, int ldc)
{
    constexpr int D = kStripDepth;
    extern __shared__ direct_f4 s_strip[];  // op(B): [group][tile][lane]
    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), x = lane & 15, q = lane >> 4;
    const int whole = K / 16, groups = (K + 15) / 16;  // whole >= 1
    // the strips are dealt out evenly
    const int64_t strips = ((int64_t)M + 15) / 16, waves = (int64_t)gridDim.x * kStripWaves, w = (int64_t)blockIdx.x * kStripWaves + wave;
    const int first = (int)(w * strips / waves), end = (int)((w + 1) * strips / waves);
    direct_f4 ring[D], tail = {0.0f, 0.0f, 0.0f, 0.0f};
    const float *row = nullptr;
    const auto load4 = [&](int k) {
        const DirectF4U r = *reinterpret_cast<const DirectF4U *>(row + k);
        return direct_f4{r.v[0], r.v[1], r.v[2], r.v[3]};
    };
    const auto fetch = [&](int g) { return load4(16 * (g < whole ? g : whole - 1)); };  // the last group again instead of one behind it
    const int past = 16 * whole + 4 * q + 4 - K;  // how far this lane's piece of the partial group reaches past the row: it slides back
    const auto begin = [&](int s) {
        const int64_t r = (int64_t)s * 16 + x;
        row = A + (size_t)(r < M ? r : M - 1) * lda + 4 * q;
#pragma unroll
        for (int d = 0; d < D; ++d) ring[d] = fetch(d);
        if (whole < groups) tail = load4(16 * whole - (past > 0 ? past : 0));
    };
    if (first < end) begin(first);  // in flight while op(B) comes
    {
        // Columns past op(B) read its last one: nobody stores their sums.  Transposed, four steps of a lane are one 16-byte load, brought into order as A's are.
        constexpr int U = 4;
        const int blocks = groups * NT, turn = (int)((blockIdx.x / 8) % 32) * blocks / 32;
        const int lane_k = ASC && !TB ? q : 4 * q;
        constexpr int kStep = ASC && !TB ? 4 : 1;
        const int x_last = 16 * (NT - 1) + x < N ? x : N - 1 - 16 * (NT - 1);  // of the last tile
        const float *lane_b = TB ? B + (size_t)x * ldb + lane_k : B + (size_t)lane_k * ldb + x;
        const float *lane_b_last = TB ? B + (ptrdiff_t)x_last * ldb + lane_k : B + (size_t)lane_k * ldb + x_last;
        for (int b0 = wave; b0 < blocks; b0 += U * kStripWaves) {
            direct_f4 v[U];
            int at[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                int b = b0 + u * kStripWaves < blocks ? b0 + u * kStripWaves : b0;
                b = b + turn < blocks ? b + turn : b + turn - blocks;
                at[u] = b;
                const int g = b / NT, t = b - g * NT;
                const float *src = (t < NT - 1 ? lane_b : lane_b_last) + (TB ? (size_t)(16 * t) * ldb + 16 * g : (size_t)(16 * g) * ldb + 16 * t);
                if (16 * g + 16 <= K) {
                    if constexpr (TB) {
                        const DirectF4U r = *reinterpret_cast<const DirectF4U *>(src);
                        v[u] = direct_f4{r.v[0], r.v[1], r.v[2], r.v[3]};
                    } else {
#pragma unroll
                        for (int j = 0; j < 4; ++j) v[u][j] = src[(size_t)(kStep * j) * ldb];
                    }
                } else {  // the partial group: zeros past the reduction, the last step's element read again instead
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int k = 16 * g + lane_k + kStep * j, over = k < K ? 0 : k - (K - 1);
                        const float e = TB ? src[kStep * j - over] : src[(ptrdiff_t)(kStep * j - over) * ldb];
                        v[u][j] = k < K ? e : 0.0f;
                    }
                }
            }
            if constexpr (TB && ASC)
#pragma unroll
                for (int u = 0; u < U; ++u) v[u] = strip_ascending(v[u]);
#pragma unroll
            for (int u = 0; u < U; ++u) s_strip[at[u] * kWave + lane] = v[u];
        }
    }
    __syncthreads();
    const auto operand = [&](int g, direct_f4 (&b)[NT]) {
        g = g < groups ? g : groups - 1;
#pragma unroll
        for (int t = 0; t < NT; ++t) b[t] = s_strip[(g * NT + t) * kWave + lane];
    };
    for (int s = first; s < end; ++s) {
        direct_f4 acc[NT], b0[NT], b1[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = direct_f4{0.0f, 0.0f, 0.0f, 0.0f};
        const auto multiply = [&](const direct_f4 (&b)[NT], direct_f4 a) {
            if constexpr (ASC) a = strip_ascending(a);
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[t][j], acc[t], 0, 0, 0);
        };
        operand(0, b0);
        static_assert(D % 2 == 0, "the two operand buffers take turns");
        int g = 0;
        for (; g + D <= whole; g += D) {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                operand(g + d + 1, d % 2 ? b0 : b1);
                __builtin_amdgcn_sched_barrier(0);
                multiply(d % 2 ? b1 : b0, ring[d]);
                ring[d] = fetch(g + d + D);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int d = 0; d < D; ++d)
            if (g + d < whole) {
                operand(g + d + 1, d % 2 ? b0 : b1);
                __builtin_amdgcn_sched_barrier(0);
                multiply(d % 2 ? b1 : b0, ring[d]);
            }
        if (whole < groups) {
            operand(whole, b0);
            direct_f4 a = tail;  // zeros past the row
            if (past > 0) {
                if (past & 1) a = direct_f4{a[1], a[2], a[3], 0.0f};
                if (past & 2) a = direct_f4{a[2], a[3], 0.0f, 0.0f};
                if (past >= 4) a = direct_f4{0.0f, 0.0f, 0.0f, 0.0f};
            }
            multiply(b0, a);
        }
        if (s + 1 < end) begin(s + 1);
        // register v of lane x + 16 q of a tile is row 4 q + v, column x
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int64_t r = (int64_t)s * 16 + 4 * q + v;
            if (r >= M) continue;
            float *dst = C + (size_t)r * ldc + x;
#pragma unroll
            for (int t = 0; t < NT; ++t)
                if (16 * t + x < N) {
                    float sum = alpha * acc[t][v];
                    if (beta != 0.0f) sum += beta * dst[16 * t];
                    dst[16 * t] = sum;
                }
        }
    }
}

// Enough rows, and enough to multiply, to pay for op(B) in every CU's LDS (us by the other kernels / here, in millions of multiply-adds: 30,647 x 90 x 5
// (14) 5.1 / 6.4, 46,375 x 119 x 4 (22) 7.7 / 8.4, 81,311 x 131 x 7 (75) 13.4 / 13.9, 28,200 x 224 x 32 (202) 11.6 / 8.7).
bool strip_covers(int M, int N, int K)
{
    return M >= 28000 && N <= 128 && K >= 16 && (int64_t)M * N * K >= 80'000'000 && strip_lds(N, K) <= kStripLds;
}

template <int NT>
void launch_strip(bool tb, bool ascending, int M, int N, int K, float alpha, const float *A, int lda, const float *B, int ldb, float beta, float *C,
                  int ldc, hipStream_t s)
{
    const unsigned grid = (unsigned)std::min<int64_t>(kStripGroups, ceil_div(ceil_div(M, 16), kStripWaves));
    const auto go = [&](auto kernel) {
        kernel<<<grid, kStripWaves * kWave, strip_lds(N, K), s>>>(M, N, K, alpha, A, lda, B, ldb, beta, C, ldc);
    };
    if (tb && ascending) go(sgemm_strip_kernel<NT, true, true>);
    else if (tb) go(sgemm_strip_kernel<NT, true, false>);
    else if (ascending) go(sgemm_strip_kernel<NT, false, true>);
    else go(sgemm_strip_kernel<NT, false, false>);
}
void sgemm_strip(bool tb, bool ascending, int M, int N, int K, float alpha, const float *A, int lda, const float *B, int ldb, float beta, float *C,
                 int ldc, hipStream_t s)
{
    const int nt = (int)ceil_div(N, 16);
#define DRONE_STRIP(NT_) if (nt == NT_) launch_strip<NT_>(tb, ascending, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, s);
    DRONE_STRIP(1)
    DRONE_STRIP(2)
    DRONE_STRIP(3)
    DRONE_STRIP(4)
    DRONE_STRIP(5)
    DRONE_STRIP(6)
    DRONE_STRIP(7)
    DRONE_STRIP(8)
#undef DRONE_STRIP
}

}  // namespace
}  // namespace drone
