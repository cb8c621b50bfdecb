// Row-major fp32 GEMM on the gfx950 matrix cores:  C(MxN) = alpha * op(A)(MxK) * op(B)(KxN) + beta * C.
// Replaces the three cublasSgemm calls of cuda_gcn's CUDAMatmul (cuda_gcn/src/cuda/cuda_module.cu:25-38
// forward, :72-85 input gradient, :92-105 weight gradient), which are tall-skinny: M or K is the vertex
// count, the other dimensions are feature widths (41..602).
//
// Work-group = 512 lanes: 4 product wavefronts computing a BM x BN tile of C (128 x 128, 64 x 128 or 128 x 64) with
// v_mfma_f32_32x32x2_f32 - every one owns a (BM/WM) x (BN/WN) sub-tile as 32x32 accumulators - and 4 loader
// wavefronts that move the A and B tiles of depth 32 from global memory into LDS.  The split exists because a
// wavefront that issues a global load into a backed-up memory pipeline stalls at the issue, in order, for
// thousands of cycles (measured with the cycle counter: issuing one tile's loads took longer than multiplying
// it), and a stalled wavefront issues no MFMAs either; with separate roles the loaders absorb that stall while
// the product wavefronts only ever touch LDS.  One barrier per tile hands tile i + 1 over (double-buffered LDS)
// while tile i + 2 is in flight in the loaders' registers.
// Tiles are staged k-major ([k][m], [k][n]) so that the lanes of one MFMA operand read consecutive addresses;
// the operands of the next k-step are read before the current step's four MFMAs are issued.  A tile that lies
// inside the matrix is fetched with 16-byte loads (rows whose leading dimension is a multiple of 4 floats get
// them aligned, which measured 10-20 % faster than odd strides such as 602); edge tiles take dword loads with a
// bounds check per element, so M, N, K and the leading dimensions are arbitrary.
// Measured on one MI355X: 232,965 x 602 x 128 100 TFLOP/s (640-wide aligned rows 110), 65,536 x 32,768 x 128 (the
// dense-core shape of the SpMM) 133 TFLOP/s = 84 % of the 157 TFLOP/s fp32 MFMA peak.
// A long reduction with few tiles is split over grid.z; the partial tiles go to a scratch buffer and are summed in split order by a
// second kernel.  Weight gradients (A transposed, K = vertex count) have a kernel of their own, gemm_grad.h.
#include <algorithm>
#include <map>
#include <mutex>
#include <utility>

#include "common.h"
#include "gemm_direct.h"
#include "gemm_flat.h"
#include "gemm_grad.h"
#include "gemm_strip.h"

namespace drone {
namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kTileRows = 128;
constexpr int BK = 32;
constexpr int PAD = 4;

// Four consecutive floats that are only known to be 4-byte aligned (leading dimensions such as 602 or 41 are
// odd multiples of a dword); the hardware takes such a 16-byte load in one instruction.
struct alignas(4) Float4U {
    float v[4];
};

// Loads a (BK x EXT) k-major tile of op(X) into registers: element (k, i) for k in [0,BK), i in [0,EXT).
// K_CONTIG: memory holds X[i][k] (k contiguous) - lanes walk k fastest; else X[k][i] - lanes walk i fastest.
// A tile with all BK steps of the reduction is fetched as 16-byte loads without masks (`full`, uniform over the
// work-group), also where it reaches past the matrix in i (not INSIDE): what stands there only reaches outputs that
// nobody stores, so a lane past the end reads the last row again, or slides back to the row's last four elements and puts
// those of its own that exist in their place (store(): doing it here would wait for the load).  The last, partial tile of
// the reduction takes dword loads with a check per element.  The two paths distribute the elements over the lanes
// differently, so store() must be told which one filled the registers.  With checked dword loads for every tile that
// reaches past the matrix, 30,011 x 301 x 100 took 41 us (36 now), 602 x 128 over 232,965 rows 384 (336; the model pads that operand), 1,000 x 3,000 x
// 1,001 transposed 350 (208).
template <int EXT, bool K_CONTIG, bool INSIDE>
struct TileLoader {
    static constexpr int PER = BK * EXT / 256;
    static constexpr int VPER = PER / 4;
    float r[PER];
    // How far this lane's piece of i slid back, modulo 4 (a piece that lies wholly outside: any).
    static __device__ __forceinline__ int slid(int t, int i0, int i_end)
    {
        const int i = i0 + 4 * (t % (EXT / 4));
        return K_CONTIG || INSIDE || i + 4 <= i_end ? 0 : (i + 4 - i_end) & 3;
    }
    __device__ __forceinline__ void load(int t, const float *__restrict__ X, int ld, int i0, int i_end, int k0, int k_end, bool full)
    {
        const auto fetch = [&](int p, const float *src) {
            const Float4U q = *reinterpret_cast<const Float4U *>(src);
#pragma unroll
            for (int j = 0; j < 4; ++j) r[4 * p + j] = q.v[j];
        };
        if (full) {
#pragma unroll
            for (int p = 0; p < VPER; ++p) {
                if constexpr (K_CONTIG) {
                    const int i = i0 + t / (BK / 4) + p * (1024 / BK);
                    fetch(p, X + (size_t)(INSIDE || i < i_end ? i : i_end - 1) * ld + k0 + 4 * (t % (BK / 4)));
                } else {
                    const int i = i0 + 4 * (t % (EXT / 4));
                    fetch(p, X + (size_t)(k0 + t / (EXT / 4) + p * (1024 / EXT)) * ld + (INSIDE || i + 4 <= i_end ? i : i_end - 4));
                }
            }
            return;
        }
#pragma unroll
        for (int p = 0; p < PER; ++p) {
            int k, i;
            if constexpr (K_CONTIG) { k = t % BK; i = t / BK + p * (256 / BK); }
            else { i = t % EXT; k = t / EXT + p * (256 / EXT); }
            const int gi = i0 + i, gk = k0 + k;
            float v = 0.0f;
            if (gi < i_end && gk < k_end) v = K_CONTIG ? X[(size_t)gi * ld + gk] : X[(size_t)gk * ld + gi];
            r[p] = v;
        }
    }
    __device__ __forceinline__ void store(int t, float *s /* [BK][EXT+PAD] */, bool full, int slid) const
    {
        if (full) {
#pragma unroll
            for (int p = 0; p < VPER; ++p) {
                if constexpr (K_CONTIG) {
                    const int i = t / (BK / 4) + p * (1024 / BK), k = 4 * (t % (BK / 4));
#pragma unroll
                    for (int j = 0; j < 4; ++j) s[(k + j) * (EXT + PAD) + i] = r[4 * p + j];
                } else {
                    const int k = t / (EXT / 4) + p * (1024 / EXT), i = 4 * (t % (EXT / 4));
                    float4 v = make_float4(r[4 * p], r[4 * p + 1], r[4 * p + 2], r[4 * p + 3]);
                    if constexpr (!INSIDE) {
                        if (slid & 1) v.x = v.y, v.y = v.z, v.z = v.w;
                        if (slid & 2) v.x = v.z, v.y = v.w;
                    }
                    *reinterpret_cast<float4 *>(s + k * (EXT + PAD) + i) = v;
                }
            }
            return;
        }
#pragma unroll
        for (int p = 0; p < PER; ++p) {
            int k, i;
            if constexpr (K_CONTIG) { k = t % BK; i = t / BK + p * (256 / BK); }
            else { i = t % EXT; k = t / EXT + p * (256 / EXT); }
            s[k * (EXT + PAD) + i] = r[p];
        }
    }
};

// op(A) is M x K: TA=false -> A stored M x K (k contiguous); TA=true -> A stored K x M (m contiguous).
// op(B) is K x N: TB=false -> B stored K x N (n contiguous); TB=true -> B stored N x K (k contiguous).
template <int BM, int BN, bool TA, bool TB>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4, 4))) void sgemm_mfma_kernel(
    int M, int N, int K, float alpha, const float *__restrict__ A, int lda, const float *__restrict__ B, int ldb,
    float beta, float *__restrict__ C, int ldc, int k_chunk, float *__restrict__ partial)
{
    constexpr int WN = BN / 64;        // wavefronts along n (2 or 1)
    constexpr int WM = 4 / WN;         // wavefronts along m
    constexpr int TM = BM / WM / 32;   // 32x32 accumulators per wavefront along m (2 or 1)
    constexpr int TN = 2;              // and along n (64 columns per wavefront)
    __shared__ __attribute__((aligned(16))) float sA[2][BK * (BM + PAD)];
    __shared__ __attribute__((aligned(16))) float sB[2][BK * (BN + PAD)];

    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const int kb = blockIdx.z * k_chunk;
    const int ke = kb + k_chunk < K ? kb + k_chunk : K;
    const int tiles = (ke - kb + BK - 1) / BK;
    const int t = threadIdx.x & 255;

    if (threadIdx.x >= 256) {
        // ---- loader wavefronts: tile i + 1 goes to LDS while tile i is multiplied, tile i + 2 is in flight ----
        const auto run = [&](auto inside) {
            constexpr bool kInside = decltype(inside)::value;
            TileLoader<BM, !TA, kInside> la;
            TileLoader<BN, TB, kInside> lb;
            const bool wide_a = !TA || M >= 4, wide_b = TB || N >= 4;  // there is a piece of four to slide back to
            const int slid_a = la.slid(t, m0, M), slid_b = lb.slid(t, n0, N);
            auto fetch = [&](int i) {
                const int k0 = kb + i * BK;
                const bool full = k0 + BK <= ke;
                la.load(t, A, lda, m0, M, k0, ke, full && wide_a);
                lb.load(t, B, ldb, n0, N, k0, ke, full && wide_b);
            };
            auto put = [&](int i) {
                const bool full = kb + (i + 1) * BK <= ke;
                la.store(t, sA[i & 1], full && wide_a, slid_a);
                lb.store(t, sB[i & 1], full && wide_b, slid_b);
            };
            if (tiles > 0) {
                fetch(0);
                put(0);
            }
            if (tiles > 1) fetch(1);
            __syncthreads();
            for (int i = 0; i < tiles; ++i) {
                if (i + 1 < tiles) put(i + 1);
                if (i + 2 < tiles) fetch(i + 2);
                __syncthreads();
            }
        };
        // the tile's extent in m / n lies inside C
        if (m0 + BM <= M && n0 + BN <= N) run(std::true_type{});
        else run(std::false_type{});
        return;
    }

    // ---- product wavefronts ----
    const int wave = t / kWave, lane = t & (kWave - 1);
    const int wm = wave / WN, wn = wave % WN;
    const int lr = lane & 31, lk = lane >> 5;

    floatx16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

    __syncthreads();
    for (int it = 0; it < tiles; ++it) {
        const float *a = sA[it & 1], *b = sB[it & 1];
        // Operands of step kk + 2 are read before the products of step kk are issued (the scheduling barriers keep
        // the compiler from sinking the reads back to their use), so the LDS latency hides behind 4 MFMAs.
        float av[2][TM], bv[2][TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) av[0][i] = a[lk * (BM + PAD) + wm * (TM * 32) + i * 32 + lr];
#pragma unroll
        for (int j = 0; j < TN; ++j) bv[0][j] = b[lk * (BN + PAD) + wn * 64 + j * 32 + lr];
#pragma unroll
        for (int kk = 0; kk < BK; kk += 2) {
            const int cur = (kk / 2) & 1;
            if (kk + 2 < BK) {
#pragma unroll
                for (int i = 0; i < TM; ++i) av[cur ^ 1][i] = a[(kk + 2 + lk) * (BM + PAD) + wm * (TM * 32) + i * 32 + lr];
#pragma unroll
                for (int j = 0; j < TN; ++j) bv[cur ^ 1][j] = b[(kk + 2 + lk) * (BN + PAD) + wn * 64 + j * 32 + lr];
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[cur][i], bv[cur][j], acc[i][j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();
    }

    // 32x32 accumulator layout: register v of lane l holds row 8*(v/4) + 4*(l/32) + v%4, column l%32.
    float *out = partial ? partial + (size_t)blockIdx.z * M * N : C;
    const int ldo = partial ? N : ldc;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int row = m0 + wm * (TM * 32) + i * 32 + 8 * (v / 4) + 4 * lk + (v % 4);
                const int col = n0 + wn * 64 + j * 32 + lr;
                if (row < M && col < N) {
                    if (partial) {
                        out[(size_t)row * ldo + col] = acc[i][j][v];
                    } else {
                        float r = alpha * acc[i][j][v];
                        if (beta != 0.0f) r += beta * out[(size_t)row * ldo + col];
                        out[(size_t)row * ldo + col] = r;
                    }
                }
            }
}

// C = alpha * sum_z partial[z] + beta * C.  A work-group of 256 lanes owns 32 consecutive outputs; lane (o, g) adds the
// partials z = g, g + 8, ... of output o (eight independent loads in flight), and the eight sums of an output are added
// in g order - a fixed order, so the result is repeatable.  (One lane per output adding all the splits in turn took
// 31 ... 108 us for 227 ... 512 splits of a few thousand outputs: a chain of dependent round trips on a few dozen CUs.)
constexpr int kReduceOutputs = 32, kReduceGroups = 8;
__global__ __launch_bounds__(kReduceOutputs * kReduceGroups) void sgemm_reduce_kernel(
    int M, int N, int splits, const float *__restrict__ partial, float alpha, float beta, float *__restrict__ C, int ldc)
{
    __shared__ float s_sum[kReduceGroups][kReduceOutputs];
    const int64_t total = (int64_t)M * N;
    const int o = threadIdx.x % kReduceOutputs, g = threadIdx.x / kReduceOutputs;
    for (int64_t base = (int64_t)blockIdx.x * kReduceOutputs; base < total; base += (int64_t)gridDim.x * kReduceOutputs) {
        const int64_t idx = base + o;
        float s = 0.0f;
        if (idx < total) {
            int z = g;
            for (; z + 7 * kReduceGroups < splits; z += 8 * kReduceGroups) {
                float v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = partial[(size_t)(z + u * kReduceGroups) * total + idx];
#pragma unroll
                for (int u = 0; u < 8; ++u) s += v[u];
            }
            for (; z < splits; z += kReduceGroups) s += partial[(size_t)z * total + idx];
        }
        s_sum[g][o] = s;
        __syncthreads();
        if (g == 0 && idx < total) {
            float sum = s_sum[0][o];
#pragma unroll
            for (int k = 1; k < kReduceGroups; ++k) sum += s_sum[k][o];
            const int row = (int)(idx / N), col = (int)(idx % N);
            float r = alpha * sum;
            if (beta != 0.0f) r += beta * C[(size_t)row * ldc + col];
            C[(size_t)row * ldc + col] = r;
        }
        __syncthreads();
    }
}

// C (M x N) = alpha * A (M x K) * op(B) + beta * C for a tall A with short rows (K <= 128) and a small op(B)
// (N <= 128): the layer products H * W and dZ * W^T of the model, 700 bytes of A and C per row for 10 K multiply-adds.
// A wavefront owns a run of consecutive rows and takes them 16 at a time: it fetches the 16 rows with whole-line loads
// (consecutive lanes, consecutive 16-byte pieces of a row), parks them in its own strip of LDS, and reads them back in
// the layout v_mfma_f32_16x16x4_f32 wants (lane = row + 16 kk holds k = 16 q + 4 kk + j in component j of its q-th
// 16-byte read; a row pitch of K + 4 floats keeps these reads free of bank conflicts).  The next 16 rows are in flight
// in registers meanwhile, op(B) sits in LDS in the order the lanes read it, and the 16 x N result goes through the
// strip once more so that it leaves in 16-byte pieces of consecutive lanes.  A strip belongs to one wavefront, whose
// LDS accesses execute in order, so the loop has no barrier.  Values of A past K are replaced by zeros, whatever the
// padding of the rows holds.
// Measured on 232,965 rows (us; the general kernel / this one): 128 -> 41 columns 65 / 40, 41 -> 128 columns 74 / 37
// (the matrix instructions and LDS traffic alone take 30, the loads alone 19, the stores alone 20 - 25).
// What did not work: loading the operand layout straight from memory, every lane its own row, costs a cache lookup
// per lane (64 per instruction): 19 us for the 119 MB of H even when all of it hits L1, 48 - 56 us in all; storing the
// accumulators as they lie (64-byte pieces of four rows per instruction) 41 / 46.
constexpr int kTallRows = 16, kTallGroups = 256;
// Wavefronts per work-group: 12 where op(B) and 12 strips fit the 160 KB of LDS, else 8.
constexpr int tall_waves(int kq, int nt)
{
    const int pitch = 16 * kq + 4, cp = 16 * nt + 4;
    return kq * nt * 1024 + 12 * kTallRows * (pitch > cp ? pitch : cp) * 4 <= 160 * 1024 ? 12 : 8;
}
template <int KQ, int NT, bool TB>
__global__ __launch_bounds__(tall_waves(KQ, NT) * kWave) void sgemm_tall_kernel(int M, int N, int K, float alpha,
                                                                        const float *__restrict__ A, int lda,
                                                                        const float *__restrict__ B, int ldb, float beta,
                                                                        float *__restrict__ C, int ldc)
{
    constexpr int kTallWaves = tall_waves(KQ, NT);
    constexpr int KP = 16 * KQ, PITCH = KP + 4, PIECES = KP / 4;  // a row of A in the strip
    constexpr int CP = 16 * NT + 4, CPIECES = 4 * NT;              // a row of C in the strip
    constexpr int kStrip = kTallRows * (PITCH > CP ? PITCH : CP) / 4;
    __shared__ floatx4 s_b[KQ * NT * kWave];
    __shared__ floatx4 s_strip[kTallWaves][kStrip];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int lr = lane & 15, kk = lane >> 4;
    // the 16-row steps of the matrix are dealt out evenly: wavefront w of W takes steps [w S / W, (w + 1) S / W)
    const int64_t all_steps = ((int64_t)M + kTallRows - 1) / kTallRows, waves = (int64_t)gridDim.x * kTallWaves;
    const int64_t w = (int64_t)blockIdx.x * kTallWaves + wave;
    const int step0 = (int)(w * all_steps / waves), steps = (int)((w + 1) * all_steps / waves) - step0;
    float *mine = reinterpret_cast<float *>(s_strip[wave]);
    // load c of a step: this lane's piece is 16-byte piece number 64 c + lane of the 16 rows
    int piece_row[KQ], piece_k[KQ];
#pragma unroll
    for (int c = 0; c < KQ; ++c) {
        piece_row[c] = (kWave * c + lane) / PIECES;
        piece_k[c] = 4 * ((kWave * c + lane) % PIECES);
    }
    // store c of a step: 16-byte piece number 64 c + lane of the 16 rows of C
    int out_row[NT], out_col[NT];
#pragma unroll
    for (int c = 0; c < NT; ++c) {
        out_row[c] = (kWave * c + lane) / CPIECES;
        out_col[c] = 4 * ((kWave * c + lane) % CPIECES);
    }
    floatx4 pre[KQ];
    auto fetch = [&](int step) {
#pragma unroll
        for (int c = 0; c < KQ; ++c) {
            int row = (step0 + step) * kTallRows + piece_row[c];
            row = row < M ? row : M - 1;
            pre[c] = *reinterpret_cast<const floatx4 *>(A + (size_t)row * lda + piece_k[c]);
        }
    };
    if (steps > 0) fetch(0);  // in flight while op(B) is staged
    // op(B)(k, n) with k = 16 q + 4 kk + j, n = 16 tile + lr  ->  s_b[(q NT + tile) 64 + 16 kk + lr][j]
    for (int e = threadIdx.x; e < KQ * NT * kWave; e += kTallWaves * kWave) {
        const int l = e % kWave, tile = (e / kWave) % NT, q = e / (kWave * NT);
        const int n = 16 * tile + (l & 15), k0 = 16 * q + 4 * (l >> 4);
        floatx4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int k = k0 + j;
            v[j] = (k < K && n < N) ? (TB ? B[(size_t)n * ldb + k] : B[(size_t)k * ldb + n]) : 0.0f;
        }
        s_b[e] = v;
    }
    __syncthreads();
    for (int step = 0; step < steps; ++step) {
#pragma unroll
        for (int c = 0; c < KQ; ++c) {
            floatx4 v = pre[c];
            if (KP != K) {
#pragma unroll
                for (int j = 0; j < 4; ++j) v[j] = piece_k[c] + j < K ? v[j] : 0.0f;
            }
            *reinterpret_cast<floatx4 *>(mine + piece_row[c] * PITCH + piece_k[c]) = v;
        }
        if (step + 1 < steps) fetch(step + 1);
        floatx4 acc[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        // the wavefronts that have matrix instructions to issue go first: those fetching or storing wait anyway
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int q = 0; q < KQ; ++q) {
            const floatx4 a = *reinterpret_cast<const floatx4 *>(mine + lr * PITCH + 16 * q + 4 * kk);
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const floatx4 b = s_b[(q * NT + t) * kWave + lane];
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[j], acc[t], 0, 0, 0);
            }
        }
        __builtin_amdgcn_s_setprio(0);
        // Through the strip again, so that C is written in whole 16-byte pieces of consecutive lanes: the lane holds
        // C(row = 4 kk + i, column = lr) of every 16 x 16 tile.
        const int row_base = (step0 + step) * kTallRows;
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) mine[(4 * kk + i) * CP + 16 * t + lr] = alpha * acc[t][i];
        floatx4 out[NT];
#pragma unroll
        for (int c = 0; c < NT; ++c) out[c] = *reinterpret_cast<const floatx4 *>(mine + out_row[c] * CP + out_col[c]);
        if (beta != 0.0f) {
#pragma unroll
            for (int c = 0; c < NT; ++c) {
                const int row = row_base + out_row[c];
                if (row >= M) continue;
                const float *old = C + (size_t)row * ldc + out_col[c];
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (out_col[c] + j < N) out[c][j] += beta * old[j];
            }
        }
#pragma unroll
        for (int c = 0; c < NT; ++c) {
            const int row = row_base + out_row[c];
            if (row < M && out_col[c] + 4 <= N) *reinterpret_cast<floatx4 *>(C + (size_t)row * ldc + out_col[c]) = out[c];
        }
        if (N % 4 != 0) {
#pragma unroll
            for (int c = 0; c < NT; ++c) {
                const int row = row_base + out_row[c];
                if (row < M && out_col[c] < N && out_col[c] + 4 > N) {
                    float *dst = C + (size_t)row * ldc + out_col[c];
#pragma unroll
                    for (int j = 0; j < 3; ++j)
                        if (out_col[c] + j < N) dst[j] = out[c][j];
                }
            }
        }
    }
}

// Grow-only scratch for split-K partials, one per (device, stream): calls on one stream are ordered, so they can
// share a buffer; calls on different streams may overlap and get their own.  It grows under stream capture too: there nothing may be waited
// for, so what earlier calls may still read stays allocated, and a buffer that a graph was given stays for the graph's replays.  Such growth at least
// doubles, so what stays is less than what is in use.
struct SplitScratch {
    float *ptr = nullptr;
    size_t bytes = 0;
    bool recorded = false;  // allocated under capture
};
std::mutex g_ws_mutex;
std::map<std::pair<int, hipStream_t>, SplitScratch> g_ws;

int workspace(size_t bytes, hipStream_t s, float **out)
{
    int dev = 0;
    DRONE_HIP_TRY(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lock(g_ws_mutex);
    SplitScratch &w = g_ws[std::make_pair(dev, s)];
    if (w.bytes < bytes) {
        hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(s, &status) != hipSuccess) (void)hipGetLastError();  // the null stream beside another's capture: not recorded itself
        const bool capturing = status != hipStreamCaptureStatusNone;
        if (capturing || w.recorded) {
            bytes = std::max(bytes, 2 * w.bytes);
        } else if (w.ptr) {
            DRONE_HIP_TRY(hipStreamSynchronize(s));  // earlier calls on this stream may still read it
            (void)hipFree(w.ptr);
            w = SplitScratch{};
        }
        float *p = nullptr;
        // an allocation is no part of the graph: the thread's mode lets it through while others record in theirs
        hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
        if (capturing) DRONE_HIP_TRY(hipThreadExchangeStreamCaptureMode(&mode));
        const hipError_t allocated = hipMalloc(&p, bytes);
        if (capturing) DRONE_HIP_TRY(hipThreadExchangeStreamCaptureMode(&mode));
        DRONE_HIP_TRY(allocated);
        w = SplitScratch{p, bytes, capturing};
    }
    *out = w.ptr;
    return DRONE_OK;
}

template <int BM, int BN>
void launch(bool ta, bool tb, dim3 grid, hipStream_t s, int M, int N, int K, float alpha, const float *A, int lda,
            const float *B, int ldb, float beta, float *C, int ldc, int k_chunk, float *partial)
{
    if (!ta && !tb) sgemm_mfma_kernel<BM, BN, false, false><<<grid, 512, 0, s>>>(M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, k_chunk, partial);
    else if (!ta && tb) sgemm_mfma_kernel<BM, BN, false, true><<<grid, 512, 0, s>>>(M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, k_chunk, partial);
    else if (ta && !tb) sgemm_mfma_kernel<BM, BN, true, false><<<grid, 512, 0, s>>>(M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, k_chunk, partial);
    else sgemm_mfma_kernel<BM, BN, true, true><<<grid, 512, 0, s>>>(M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, k_chunk, partial);
}

}  // namespace
}  // namespace drone

using namespace drone;

// Split-K partials of the entry point that may not allocate: one fixed array per GPU, held by the library's code
// object until the process ends.  In host code this name is only a handle for hipGetSymbolAddress; the address a
// kernel can use is looked up once per device (static_scratch) and passed on as an ordinary pointer.
constexpr size_t kStaticScratchFloats = (size_t)8 << 20;  // 32 MiB
static __device__ __align__(256) float scratch[kStaticScratchFloats];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_static_mutex;
float *g_static_scratch[kMaxDevices] = {};

// Device address of this GPU's copy of `scratch` (every device holds its own copy at its own address).
int static_scratch(float **out)
{
    int dev = 0;
    DRONE_HIP_TRY(hipGetDevice(&dev));
    DRONE_REQUIRE(dev >= 0 && dev < kMaxDevices, "device ordinal out of range");
    std::lock_guard<std::mutex> lock(g_static_mutex);
    if (!g_static_scratch[dev]) {
        void *p = nullptr;
        DRONE_HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        DRONE_REQUIRE(p != nullptr, "no device address for the static scratch array");
        g_static_scratch[dev] = static_cast<float *>(p);
    }
    *out = g_static_scratch[dev];
    return DRONE_OK;
}

void launch_reduce(int M, int N, int splits, const float *partial, float alpha, float beta, float *C, int ldc, hipStream_t s)
{
    int blocks = (int)ceil_div((int64_t)M * N, kReduceOutputs);
    if (blocks > 8192) blocks = 8192;
    sgemm_reduce_kernel<<<blocks, kReduceOutputs * kReduceGroups, 0, s>>>(M, N, splits, partial, alpha, beta, C, ldc);
}

// Where a caller that adds the sums of a split reduction up by itself wants them.  splits: 0 until they are left there.
struct KeptSums {
    float *sums;
    int64_t floats;
    int splits = 0;
};

// Scratch for `floats` partial sums: the caller's, the stream's grow-only buffer, or the fixed array of the entry point that may not
// allocate.
int split_scratch(bool may_allocate, KeptSums *kept, size_t floats, hipStream_t s, int M, int N, int K, int splits, float **partial)
{
    if (kept && kept->sums && (int64_t)floats <= kept->floats) {
        kept->splits = splits;
        *partial = kept->sums;
        return DRONE_OK;
    }
    if (may_allocate) return workspace(sizeof(float) * floats, s, partial);
    if (floats > kStaticScratchFloats) {
        set_error(DRONE_ERR_INVALID,
                  "drone_sgemm_rm_f32_noalloc: %d x %d x %d splits the reduction %d ways and needs %zu bytes of "
                  "partial sums, the fixed scratch holds %zu; use drone_sgemm_rm_f32",
                  M, N, K, splits, floats * sizeof(float), kStaticScratchFloats * sizeof(float));
        return DRONE_ERR_INVALID;
    }
    return static_scratch(partial);
}

// C = alpha * A * op(B) + beta * C for a tall A with rows of at most 128 values (see sgemm_tall_kernel); false when no
// instance of the kernel covers the shape.
template <int KQ, int NT, bool TB>
void launch_tall(int M, int N, int K, float alpha, const float *A, int lda, const float *B, int ldb, float beta, float *C,
                 int ldc, hipStream_t s)
{
    // one work-group per CU, as many as there are 16-row steps for every wavefront
    const int64_t all_steps = ceil_div(M, kTallRows);
    constexpr int kTallWaves = tall_waves(KQ, NT);
    const unsigned grid = (unsigned)std::min<int64_t>(kTallGroups, ceil_div(all_steps, kTallWaves));
    sgemm_tall_kernel<KQ, NT, TB><<<grid, kTallWaves * kWave, 0, s>>>(M, N, K, alpha, A, lda, B, ldb, beta, C, ldc);
}
// Whether an instance of sgemm_tall_kernel covers the product.
bool tall_covers(int transB, int M, int N, int K, const float *A, int lda, const float *C, int ldc)
{
    const int kq = (K + 15) / 16;
    // Enough rows for its 256 x 12 wavefronts: 41 columns x 128 take 12.0 us (10.5 by sgemm_direct_kernel) at 30,000 rows, 15.1
    // (16.1) at 50,000.  The lanes read whole 16-byte pieces of A's rows up to column 16 kq, and write C's in such pieces.
    if (M < 32768 || K < 1 || N > 128 || lda < 16 * kq || lda % 4 != 0 || (reinterpret_cast<uintptr_t>(A) & 15) != 0 ||
        ldc % 4 != 0 || (reinterpret_cast<uintptr_t>(C) & 15) != 0)
        return false;
    return transB ? (kq == 3 || kq == 4 || kq == 8) && N > 48 : kq == 4 || kq == 8;
}
void sgemm_tall(int transB, int M, int N, int K, float alpha, const float *A, int lda, const float *B, int ldb, float beta,
                float *C, int ldc, hipStream_t s)
{
    const int kq = (K + 15) / 16, nt = N <= 48 ? 3 : N <= 64 ? 4 : 8;
#define DRONE_TALL(KQ_, NT_, TB_)                                                            \
    if (kq == KQ_ && nt == NT_ && (transB != 0) == TB_) {                                    \
        launch_tall<KQ_, NT_, TB_>(M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, s);         \
        return;                                                                              \
    }
    DRONE_TALL(8, 3, false)
    DRONE_TALL(8, 4, false)
    DRONE_TALL(4, 3, false)
    DRONE_TALL(4, 4, false)
    DRONE_TALL(8, 8, false)
    DRONE_TALL(4, 8, false)
    DRONE_TALL(8, 8, true)
    DRONE_TALL(8, 4, true)
    DRONE_TALL(3, 8, true)
    DRONE_TALL(4, 8, true)
    DRONE_TALL(3, 4, true)
    DRONE_TALL(4, 4, true)
#undef DRONE_TALL
}

// Whether 128-column tiles have 64 rows instead of 128: two of their work-groups on a CU work while one waits at its barrier
// (matrix cores busy 53 % of the time with one), and half as many CUs idle at the end.  us 128 / 64 rows: 30,011 x 301 x 100 34.6 /
// 32.0, 45,000 x 300 x 128 51.3 / 43.7, 5,000 x 1,000 x 1,000 146 / 119, 1,000 x 1,001 x 3,000 82 / 76.  Not where 128-row tiles come
// two to a CU anyway, 60,000 x 400 x 100 67.6 / 70.6, and not with A transposed, whose tiles are read in shorter runs.
bool half_rows(bool transA, int tiles) { return !transA && tiles <= 384; }

// How many ways the tiled kernel splits the reduction: when the output has too few tiles to fill 256 CUs and K is long.
int tiled_splits(int tiles, int K)
{
    if (tiles >= 256 || K < 4096) return 1;
    // two work-groups per CU in one round, and at least 1024 reduction steps per work-group (ms for outputs of 128 x 41 / 602 x 128
    // over 232,965 steps: 1024 work-groups of at least 512 steps 0.153 / 0.443; 512 and 512: 0.153 / 0.414; 256 and 1024:
    // 0.106 / 0.516; 512 and 1024: 0.106 / 0.411; 512 and 2048: 0.123 / 0.414)
    return std::max(1, std::min(512 / tiles, (int)ceil_div(K, 1024)));
}

// Which products sgemm_direct_kernel takes, and in which shape (ks = 0: the tiled kernel).  The shapes were chosen by
// timing all instances on some 150 layer products (2 ... 128 columns, inner dimensions 2 ... 700, 1,000 ... 233,000 rows);
// the choice between the kernels compares two estimates that were fitted to the same runs.
struct DirectShape {
    int mt = 0, nt = 0, ks = 0;
};
DirectShape direct_shape(int M, int N, int K)
{
    DirectShape d;
    if (K < 1) return d;
    const auto blocks = [&]() { return ceil_div(M, 16 * d.mt) * ceil_div(N, 16 * d.nt); };
    const int n16 = (int)ceil_div(N, 16);
    d.mt = 1;
    d.nt = n16 <= 4 ? n16 : n16 <= 6 ? 3 : n16 == 7 ? 7 : 4;
    const int64_t waves = blocks();
    if (K >= 384 && d.nt != 7) {
        // the wavefronts of a work-group share a row block: less of op(B) is read per product
        d.ks = 8;
        if (waves >= 1024 && d.nt != 3) d.mt = 2;
    } else if (waves >= 1024) {
        d.ks = 1;
        if (waves >= 4096) d.mt = 2;
    } else {
        if (d.nt == 7) d.nt = 4;
        if (K < 256 && d.nt > 2 && waves < 512) d.nt = 2;
        d.ks = K >= 384 ? 8 : K >= 64 ? 4 : 1;
    }
    // half of the CUs at least (1,884 x 137 x 25 4.1 -> 3.3 us, its transposed B 1,927 x 218 x 28 3.9 -> 3.4)
    while (d.ks == 4 && d.nt > 1 && blocks() < 128) d.nt = (d.nt + 1) / 2;
    // Deep reductions (384 steps and more) bring the tiled kernel's streams up to speed - 2.8 instead of 2.0 TB/s, and two of
    // its work-groups on a CU take 0.85 of two rounds -, and the direct kernel, whose row blocks each read all of op(B), reaches
    // 60 instead of 75 TFLOP/s there.  us direct / tiled: dense rectangles of an SpMM plan, 4,096 x 32,768 x 41 336 / 196 and
    // 16,384 x 32,768 x 64 834 / 688; layers of 53,965 x 527 x 59 60 / 49, 128,580 x 582 x 63 151 / 118, 11,824 x 619 x 94
    // 28 / 55.  With one set of rates for all depths an SpMM of 229 M entries and 41 columns under an ordinary plan took
    // 2.46 ms (2.26).
    const bool deep = K >= 384;
    // us: matrix instructions at the rate the kernel reaches on padded blocks, or its memory traffic
    const double in = 4.0 * ((double)M * K + (double)K * N), out = 4.0 * M * N;
    const double padded = 2.0 * blocks() * (16 * d.mt) * (16 * d.nt) * K;
    const double direct_us = std::max(padded / (deep ? 60e6 : 75e6), in / 4.5e6 + out / 1.9e6);
    // us: rounds of work-groups over the CUs times depth-32 tiles (1.6 us for a 64-wide tile, 2.25 for a 128-wide one)
    const int tiles = (int)(ceil_div(M, kTileRows) * ceil_div(N, N <= 64 ? 64 : 128)), splits = tiled_splits(tiles, K);
    const int64_t groups = (int64_t)tiles * splits;
    const double rounds = ceil_div(groups, 256) * (deep && groups > 256 ? 0.85 : N > 64 && half_rows(false, tiles) ? 0.9 : 1.0);
    const double tiled_us = std::max(rounds * ceil_div(ceil_div(K, splits), BK) * (N <= 64 ? 1.6 : 2.25),
                                     in / (deep ? 2.8e6 : 2.0e6) + out / 2.4e6) + (splits > 1 ? 5 : 0);
    if (tiled_us < direct_us) d.ks = 0;
    return d;
}

template <int MT, int NT, bool BK, int KS>
void launch_direct(int M, int N, int K, float alpha, const float *A, int lda, const float *B, int ldb, float beta, float *C, int ldc, hipStream_t s)
{
    constexpr int kWaves = KS > 4 ? KS : 4;
    const unsigned grid = (unsigned)(ceil_div(N, 16 * NT) * ceil_div(M, 16 * MT * (kWaves / KS)));
    const size_t lds = KS > 1 ? sizeof(float) * kWaves * MT * NT * 4 * kWave : 0;
    sgemm_direct_kernel<MT, NT, BK, KS><<<grid, kWaves * kWave, lds, s>>>(M, N, K, alpha, A, lda, B, ldb, beta, C, ldc);
}

// Tiles a block of sgemm_twin_kernel, or 0 to leave the product to sgemm_direct_kernel<., ., ., 8>: as few as leave no CU a second block, whose
// wavefronts would have to share its SIMDs (us by that kernel / this: 1,726 x 1,440 x 25 8.8 / 5.9, 1,052 x 972 x 100 9.5 / 8.1 and with more
// blocks than CUs 10.6, 5,000 x 1,400 x 128 32.4 / 33.0, 16,227 x 667 x 61 23.4 / 26.1).  Eight tiles want a long reduction (2,748 x 1,452 x 117 23.5 / 18.8,
// 2,640 x 508 x 113 10.7 / 11.1), and B transposed, which takes a quarter of the loads, gains by the smaller blocks alone (1,233 x 591 x 21 4.9 / 4.2, but
// 2,708 x 1,440 x 64 16.0 / 16.5 and 3,977 x 514 x 29 5.3 / 6.0).
int twin_width(const DirectShape &d, bool tb, int M, int N, int K)
{
    if (d.ks != 8 || d.mt != 1) return 0;
    for (const int nt : {1, 2, 3, 4, 5, 6, 8})
        if (ceil_div(M, 16) * ceil_div(N, 16 * nt) <= kTwinBlocks) return (nt == 8 && K < 768) || (tb && nt == d.nt) ? 0 : nt;
    return 0;
}

template <int NT>
void launch_twin(bool tb, int M, int N, int K, float alpha, const float *A, int lda, const float *B, int ldb, float beta, float *C, int ldc, hipStream_t s)
{
    const unsigned grid = (unsigned)(ceil_div(N, 16 * NT) * ceil_div(M, 16));
    const size_t lds = sizeof(float) * kTwinShares * NT * 4 * kWave;
    if (tb) sgemm_twin_kernel<NT, true><<<grid, kTwinWaves * kWave, lds, s>>>(M, N, K, alpha, A, lda, B, ldb, beta, C, ldc);
    else sgemm_twin_kernel<NT, false><<<grid, kTwinWaves * kWave, lds, s>>>(M, N, K, alpha, A, lda, B, ldb, beta, C, ldc);
}

int sgemm_direct(const DirectShape &d, bool tb, int M, int N, int K, float alpha, const float *A, int lda, const float *B, int ldb, float beta,
                 float *C, int ldc, hipStream_t s)
{
    bool done = false;
    const int twin = twin_width(d, tb, M, N, K);
#define DRONE_TWIN(NT_)                                                                    \
    if (twin == NT_) {                                                                     \
        launch_twin<NT_>(tb, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, s);             \
        done = true;                                                                       \
    }
    DRONE_TWIN(1)
    DRONE_TWIN(2)
    DRONE_TWIN(3)
    DRONE_TWIN(4)
    DRONE_TWIN(5)
    DRONE_TWIN(6)
    DRONE_TWIN(8)
#undef DRONE_TWIN
#define DRONE_DIRECT(MT_, NT_, KS_)                                                                   \
    if (!twin && d.mt == MT_ && d.nt == NT_ && d.ks == KS_) {                                         \
        if (tb) launch_direct<MT_, NT_, true, KS_>(M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, s);  \
        else launch_direct<MT_, NT_, false, KS_>(M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, s);    \
        done = true;                                                                                  \
    }
    DRONE_DIRECT(1, 1, 1)
    DRONE_DIRECT(1, 2, 1)
    DRONE_DIRECT(1, 3, 1)
    DRONE_DIRECT(1, 4, 1)
    DRONE_DIRECT(1, 7, 1)
    DRONE_DIRECT(2, 1, 1)
    DRONE_DIRECT(2, 2, 1)
    DRONE_DIRECT(2, 3, 1)
    DRONE_DIRECT(2, 4, 1)
    DRONE_DIRECT(2, 7, 1)
    DRONE_DIRECT(1, 1, 4)
    DRONE_DIRECT(1, 2, 4)
    DRONE_DIRECT(1, 3, 4)
    DRONE_DIRECT(1, 4, 4)
    DRONE_DIRECT(1, 1, 8)
    DRONE_DIRECT(1, 2, 8)
    DRONE_DIRECT(1, 3, 8)
    DRONE_DIRECT(1, 4, 8)
    DRONE_DIRECT(2, 1, 8)
    DRONE_DIRECT(2, 2, 8)
    DRONE_DIRECT(2, 4, 8)
#undef DRONE_DIRECT
    DRONE_REQUIRE(done, "no instance of the direct kernel for this shape");
    DRONE_HIP_TRY(hipGetLastError());
    return DRONE_OK;
}

int tiled_chunk(int tiles, int K, int *k_chunk)
{
    *k_chunk = (int)ceil_div(ceil_div(K > 0 ? K : 1, tiled_splits(tiles, K)), BK) * BK;
    return (int)ceil_div(K > 0 ? K : 1, *k_chunk);
}
int tiles_of(int M, int N) { return (int)(ceil_div(M, kTileRows) * ceil_div(N, N <= 64 ? 64 : 128)); }

// Outputs of 128 tiles and more keep the tiled kernel busy without a split, and its tiles are read once per 128 rows (us tiled /
// sgemm_grad_kernel: 4,096 x 4,096 over 1,024 rows 271 / 352, 1,000 x 3,000 over 1,001 86 / 84, 4,096 x 512 over 65,536 2,064 / 2,105, 1,000 x
// 1,000, 64 tiles, over 5,000 104 / 94).
bool grad_covers(int M, int N, int K) { return K > 0 && tiles_of(M, N) < 128; }

int sgemm_entry(bool may_allocate, KeptSums *kept, int transA, int transB, int M, int N, int K, float alpha, const float *A, int lda,
                const float *B, int ldb, float beta, float *C, int ldc, drone_stream_t stream)
{
    clear_error();
    DRONE_REQUIRE(M >= 0 && N >= 0 && K >= 0, "negative dimension");
    DRONE_REQUIRE(ldc >= N, "ldc < N");
    DRONE_REQUIRE(lda >= (transA ? M : K) && ldb >= (transB ? K : N), "leading dimension too small");
    if (M == 0 || N == 0) return DRONE_OK;
    DRONE_REQUIRE(C != nullptr && (K == 0 || (A && B)), "null operand");
    hipStream_t s = as_stream(stream);
    if (!transA && K <= 128 && tall_covers(transB, M, N, K, A, lda, C, ldc)) {
        sgemm_tall(transB, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, s);
        DRONE_HIP_TRY(hipGetLastError());
        return DRONE_OK;
    }
    if (transA && !transB && grad_covers(M, N, K)) {
        const GradShape grad = grad_shape(M, N, K);
        float *partial = nullptr;
        if (grad.splits > 1) {
            const int rc = split_scratch(may_allocate, kept, (size_t)grad.splits * M * N, s, M, N, K, grad.splits, &partial);
            if (rc != DRONE_OK) return rc;
        }
        sgemm_grad(grad, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, partial, s);
        if (partial && !(kept && kept->splits > 0)) launch_reduce(M, N, grad.splits, partial, alpha, beta, C, ldc, s);
        DRONE_HIP_TRY(hipGetLastError());
        return DRONE_OK;
    }
    if (!transA) {
        const DirectShape direct = direct_shape(M, N, K);
        if (direct.ks <= 1 && beta == 0.0f && flat_covers(direct.ks == 0, M, N, K)) {
            sgemm_flat(transB != 0, direct.ks == 0, M, N, K, alpha, A, lda, B, ldb, C, ldc, s);
            DRONE_HIP_TRY(hipGetLastError());
            return DRONE_OK;
        }
        if (direct.ks <= 1 && strip_covers(M, N, K)) {
            sgemm_strip(transB != 0, direct.ks == 0, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, s);
            DRONE_HIP_TRY(hipGetLastError());
            return DRONE_OK;
        }
        if (direct.ks > 0) return sgemm_direct(direct, transB != 0, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, s);
    }
    const bool narrow = N <= 64;
    const int bn = narrow ? 64 : 128;
    const int tiles = tiles_of(M, N);
    const int bm = !narrow && half_rows(transA != 0, tiles) ? kTileRows / 2 : kTileRows;
    int k_chunk = 0;
    const int splits = tiled_chunk(tiles, K, &k_chunk);
    float *partial = nullptr;
    if (splits > 1) {
        // every (tile, split) work-group stores its whole tile, so the partials need no clearing
        const size_t floats = (size_t)splits * M * N;
        const int rc = split_scratch(may_allocate, kept, floats, s, M, N, K, splits, &partial);
        if (rc != DRONE_OK) return rc;
    }
    dim3 grid((unsigned)ceil_div(N, bn), (unsigned)ceil_div(M, bm), (unsigned)splits);
    DRONE_REQUIRE(grid.y <= 65535u * 32u, "M too large for the launch grid");
    if (narrow) launch<kTileRows, 64>(transA != 0, transB != 0, grid, s, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, k_chunk, partial);
    else if (bm < kTileRows) launch<kTileRows / 2, 128>(transA != 0, transB != 0, grid, s, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, k_chunk, partial);
    else launch<kTileRows, 128>(transA != 0, transB != 0, grid, s, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, k_chunk, partial);
    if (splits > 1 && !(kept && kept->splits > 0)) launch_reduce(M, N, splits, partial, alpha, beta, C, ldc, s);
    DRONE_HIP_TRY(hipGetLastError());
    return DRONE_OK;
}
}  // namespace

extern "C" int drone_sgemm_rm_f32(int transA, int transB, int M, int N, int K, float alpha, const float *A, int lda,
                                  const float *B, int ldb, float beta, float *C, int ldc, drone_stream_t stream)
{
    return sgemm_entry(true, nullptr, transA, transB, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, stream);
}

extern "C" int drone_sgemm_rm_f32_noalloc(int transA, int transB, int M, int N, int K, float alpha, const float *A,
                                          int lda, const float *B, int ldb, float beta, float *C, int ldc,
                                          drone_stream_t stream)
{
    return sgemm_entry(false, nullptr, transA, transB, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, stream);
}

extern "C" int64_t drone_sgemm_tn_sums_floats(int M, int N, int K, int lda, int ldb)
{
    if (M < 1 || N < 1 || K < 1) return 0;
    int k_chunk = 0;
    const int splits = grad_covers(M, N, K) ? grad_shape(M, N, K).splits : tiled_chunk(tiles_of(M, N), K, &k_chunk);
    return splits > 1 ? (int64_t)splits * M * N : 0;
}

extern "C" int drone_sgemm_tn_sums_f32(int M, int N, int K, const float *A, int lda, const float *B, int ldb, float *C, int ldc,
                                       float *sums, int64_t floats, int *splits, drone_stream_t stream)
{
    KeptSums kept{sums, floats};
    const int rc = sgemm_entry(true, &kept, 1, 0, M, N, K, 1.0f, A, lda, B, ldb, 0.0f, C, ldc, stream);
    if (splits) *splits = rc == DRONE_OK ? kept.splits : 0;
    return rc;
}

// Also resolves (and caches) the current device's address of the array, so that a caller who asks for the size before
// entering a capture or a serving loop leaves nothing but kernel launches to drone_sgemm_rm_f32_noalloc.
extern "C" int64_t drone_sgemm_noalloc_scratch_bytes(void)
{
    float *ignored = nullptr;
    (void)static_scratch(&ignored);  // a failure here is reported by the first product that needs the array
    return (int64_t)(kStaticScratchFloats * sizeof(float));
}

extern "C" int64_t drone_sgemm_flops(int M, int N, int K) { return 2ll * M * N * K; }
