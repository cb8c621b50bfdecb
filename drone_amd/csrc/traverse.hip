// CC_PEVal / CC_IncEVal and SSSP_PEVal / SSSP_IncEVal on the Go worker's boundary.
//
// Reference: DRONE/src/cuda/algorithm/cc.cu:10-46, :340-447 and sssp.cu:11-73, :398-539.  There a superstep
// repeats a push kernel over the vertices activated in the previous round (one thread walks a vertex's out-edges
// and atomicMin's its label / distance into the targets) until nothing changes, with a device synchronise per
// round.
//
// Here a dense round of distances is one sweep of the merge-path aggregation over the IN-edge CSR with min as the combining
// operator: value[v] <- min(value[v], min over in-edges u->v of value[u] + length).  No atomics, hub rows are spread over tiles, and the sweep updates in place,
// so a change can travel several hops in one sweep.  Both iterations descend monotonically towards the least
// fixed point below the starting state.  Labels, and distances over unit or integer lengths, are identical to the
// reference's.  With real-valued lengths both can stop short of the fixed point: every lower distance is stored, but a
// vertex propagates only when the improvement exceeds 1e-6 (sssp.cu:62-68).  That rule is the same in every kind of
// round here: a vertex goes on the next list, and gets its mark, if the round lowered it past the tolerance.  A sweep
// looks at all in-edges, so it takes a smaller improvement along where the reference leaves it; results lie at most
// 1e-6 per hop below the reference's value.  g->active keeps the
// reference's three classes (> 0 lowered by propagation in this call, 0 activated by a message or initial,
// -1 untouched), which is all the exchange and countActive (common.cu:17-31) look at.  The round number
// stored in g->active by the reference depends on its thread schedule and is not reproduced.
//
// A full sweep costs E however few vertices changed, so a round with a sparse frontier runs the other way round: the
// frontier is a list of vertices, the list's out-edges are dealt out evenly whatever vertices they belong to, the targets
// are lowered, and each newly lowered vertex goes once into the next list.  Which kernel takes a round depends on the
// number of out-edges of the list: up to kSmallEdges one work-group in LDS, which stays for the following rounds
// (push_rounds_small_kernel), up to E / kPullShare the whole GPU (push_round_kernel), above that a sweep - over the open
// vertices only where it is known which these are (pull_open_kernel).  All move towards the same fixed point, so
// switching between them does not change the result.  Every kernel leaves the list's size in device memory for the next
// (TraverseState), so the host enqueues several rounds per wait.
#include <algorithm>
#include <chrono>
#include <rocprim/device/device_radix_sort.hpp>

#include "exchange.h"

using namespace drone;

namespace {

constexpr int kIpt = 8;  // the tiling ensure_aggregation_ready() builds
constexpr float kUnreached = 1e8f;  // sssp.cu:33
constexpr float kRelaxEps = 1e-6f;  // sssp.cu:64

struct SsspEpi {
    float *dist;  // updated in place, as above
    const float *__restrict__ in_len;
    int *active;
    int mark;

    __device__ __forceinline__ MinF32 load(int c, int64_t e) const { return MinF32{dist[c] + in_len[e]}; }
    __device__ __forceinline__ void lower(int r, float v, double &stat) const
    {
        const float old = dist[r];
        if (v < old) {  // sssp.cu:62-68: the minimum is always stored, the vertex is activated past the tolerance
            dist[r] = v;
            if (old > v + kRelaxEps) {
                active[r] = mark;
                stat += 1.0;
            }
        }
    }
    __device__ __forceinline__ void row(int r, MinF32 s, double &stat) const { lower(r, s.v, stat); }
    __device__ __forceinline__ void fix(int r, MinF32 s, double &stat) const { lower(r, s.v, stat); }
};

// The same over lengths that are all 1.0, as build_graph leaves them: 4 bytes per edge less.
struct SsspUnitEpi : SsspEpi {
    __device__ __forceinline__ MinF32 load(int c, int64_t) const { return MinF32{dist[c] + 1.0f}; }
};

constexpr double kNegative = 0x1p32, kNotWhole = 0x1p64;  // more than there are edges, more than kNegative times that

// Where a traversal stands.  Its launches hand it on in device memory, so that several rounds can be enqueued before the host
// has to know how the first of them went: every kernel that runs rounds looks at `listed` and leaves lists that are not for
// it alone.
struct TraverseState {
    unsigned long long listed;  // vertices that still have to propagate << 32 | their out-edges
    int mark;                   // of the next round, cc.cu:37 `active[v] = step + 1`: positive, and different in every round
    int rounds;                 // rounds completed
    int which;                  // which of the two list buffers holds the list
    double not_one;             // lengths other than 1.0, and kNotWhole for each that is no whole number, kNegative for each below zero
    int hold;                   // rounds before n + 2 at which push_rounds_small_kernel stops, for near_rounds_kernel to look at the list
    // All lengths are whole numbers, some not 1.0: every improvement is past the tolerance.
    __host__ __device__ bool other_whole() const { return not_one > 0.0 && not_one < kNotWhole; }
    // ... and none is below zero.
    __host__ __device__ bool other_natural() const { return not_one > 0.0 && not_one < kNegative; }
};
// Pinned memory; `state` is as the last launch before the wait left it.
struct Report {
    TraverseState state;
    double visited;  // vertices with active != 0, if the list is empty
    int again;       // labels: whether edges between trees are left
};
// Two lists of vertices, and where each listed vertex's out-edges start in the list's concatenated out-edges.
struct Lists {
    int *vertex[2], *offset[2];
};
// A list of no vertices that no round may take for its own: all of them still have to propagate.
__host__ __device__ __forceinline__ unsigned long long everything() { return (1ull << 32) + 0xFFFFFFFFull; }

// Ends a counting kernel: the last work-group adds the work-groups' counts and hands the sum to `finish` (thread 0).
template <typename Finish>
__device__ __forceinline__ void publish_sum(double mine, double *s_red, double *block_part, unsigned int *ticket, Finish finish)
{
    const double total = block_sum_256(mine, s_red);
    unsigned int one = 0;
    if (threadIdx.x == 0) one = publish_part(block_part + blockIdx.x, total);
    if (!last_block_done(ticket, one)) return;
    const double all = block_sum_of_parts(block_part, (int)gridDim.x, s_red);
    if (threadIdx.x == 0) finish(all);
}
__device__ __forceinline__ void publish_sum(double mine, double *s_red, double *block_part, unsigned int *ticket, double *out)
{
    publish_sum(mine, s_red, block_part, ticket, [out](double all) { *out = all; });
}

// ---- labels by joining trees -------------------------------------------------------------------------------
// Where every edge has its reverse, a vertex's label is the least vertex of its component, and it need not travel there hop by
// hop: the vertices are kept as trees in cc[] itself (cc[v] = v's parent, at most v; a root is its own), an edge between two
// trees makes the larger root a child of the smaller, and at the end every vertex takes its root's number.  (Joining by
// compare-and-swap on the roots, rows dealt out by length, and leaving out the tree that a sample finds largest are known from ECL-CC -
// Jaiganesh and Burtscher, 2018 - and Afforest - Sutton, Ben-Nun and Barak, 2018.)  Along edges whose reverse is missing only
// rounds of the kernels below can tell, so no property of the graph is assumed: a tree is joined along edges that lead both ways,
// and every edge inside it is looked up in the other direction, which is how the label of the tree above comes to all of it.
// The tree of vertex 0 is the exception: it is never joined to another, its label is the least there is, and the edges it is made of
// bring that label down.  By then it holds most of the graph where there are hubs, and its vertices are spared a line of memory each.
//   cc_begin    parent = least in-neighbour if that is smaller (rows are in ascending order: the first)
//   cc_flatten  parent = root, the edges to the parents looked up
//   cc_link     joins the trees that edges lead between
//   cc_finish   label = root, flags, and the report
// Four launches and one wait whatever the graph's diameter; us of a call, by rounds / with every parent looked up / this: 500,009
// vertices and 11.6 M edges 124 / 57 / 51, 1.2 M and 33 M 175 / 89 / 81, 2.4 M and 107 M 215 / 128 / 107, R-MAT numbered as generated, 2.4 M
// and 128 M 85 / 100 / 71, a path of 12,000 7,630 / 51 / 51, a 1,000 x 1,000 grid 17,200 / 220 / 218.  They are bound by a line of memory per
// vertex, their chains of dependent loads (row bounds, neighbour, its row, ...) and the launches.
constexpr int kCcSamples = kWave;
constexpr int kCcSteps = 64;  // along one edge, of one cc_link: past them it is left to the next
struct CcTrees {
    int directed;            // number of the last call that found an edge without its reverse
    int again;               // number of the last pass that left an edge undone
    int sample[kCcSamples];  // roots of vertices from all over the graph
};

// Whether the edge u -> v, entry i of v's in-row, has its reverse v -> u.  It usually is entry i of v's out-row (edge files that name
// an edge in both directions are often sorted); short out-rows are looked through, otherwise v is searched in u's in-row.
struct Rows {
    const int *__restrict__ in_index;
    const int *__restrict__ in_src;
    const int *__restrict__ index;
    const int *__restrict__ dst;

    __device__ __forceinline__ bool leads_back(int u, int v, unsigned int i) const
    {
        const unsigned int d0 = index[v], d1 = index[v + 1];
        if (d0 + i < d1 && dst[d0 + i] == u) return true;
        if (d1 - d0 <= 8) {
            bool found = false;
            for (unsigned int d = d0; d < d1; d += 4)
#pragma unroll
                for (int k = 0; k < 4; ++k) found |= dst[d + k < d1 ? d + k : d1 - 1] == u;
            return found;
        }
        return in_row(v, in_index[u], in_index[u + 1]);
    }
    // The same for the edge v -> u, entry i of v's out-row, of a v whose in-row is at [e0, e1).
    __device__ __forceinline__ bool comes_back(int u, unsigned int i, unsigned int e0, unsigned int e1) const
    {
        return (e0 + i < e1 && in_src[e0 + i] == u) || in_row(u, e0, e1);
    }
    __device__ __forceinline__ bool in_row(int u, unsigned int lo, unsigned int hi) const
    {
        const unsigned int end = hi;
        while (lo < hi) {
            const unsigned int mid = (lo + hi) >> 1;
            if (in_src[mid] < u) lo = mid + 1; else hi = mid;
        }
        return lo < end && in_src[lo] == u;
    }
};
// Parents only ever move to smaller numbers of the same tree, so an old one still leads to the root.
__device__ __forceinline__ int parent_of(const int *cc, int v) { return __hip_atomic_load(cc + v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); }

// cc.cu:10-20
__global__ __launch_bounds__(kSpmvBlock) void cc_begin_kernel(int n, Rows rows, int *__restrict__ cc, int *__restrict__ ubm,
                                                              TraverseState *__restrict__ state)
{
    for (int v = blockIdx.x * kSpmvBlock + threadIdx.x; v < n; v += gridDim.x * kSpmvBlock) {
        const int e0 = rows.in_index[v], e1 = rows.in_index[v + 1];
        cc[v] = e0 < e1 ? min(rows.in_src[e0], v) : v;
        ubm[v] = 0;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) *state = TraverseState{everything(), 2, 1, 0, 0.0};
}

// The start of the rounds on a graph that is known to have edges without their reverse: a vertex follows its first in-neighbour,
// that one's first, and so on for as long as the numbers fall and for at most kCcHops hops, and takes the number it arrives at.
// It arrives there against the edges' direction, so the label is one that propagation would bring; all vertices still have to
// propagate.  One launch and no look-ups of reverses, where cc_begin, cc_flatten and cc_finish stood before: us of a whole call with
// those / with this, 1 M vertices and 16.5 M directed edges 104 / 83, R-MAT numbered as generated, 2.4 M vertices and 65 M directed
// edges 157 / 100, what a random cut of 500,009 vertices into two / four leaves one worker 93 / 79 and 89 / 77, a quarter of the edges of a
// 1,000 x 1,000 grid 216 / 203.
constexpr int kCcHops = 32;
__global__ __launch_bounds__(kSpmvBlock) void cc_follow_kernel(int n, const int *__restrict__ in_index, const int *__restrict__ in_src,
                                                               int *__restrict__ active, int *__restrict__ cc, int *__restrict__ ubm,
                                                               TraverseState *__restrict__ state)
{
    for (int v = blockIdx.x * kSpmvBlock + threadIdx.x; v < n; v += gridDim.x * kSpmvBlock) {
        int label = v;
        for (int hop = 0; hop < kCcHops && label > 0; ++hop) {
            const int e0 = in_index[label], e1 = in_index[label + 1];
            if (e0 == e1) break;
            const int u = in_src[e0];
            if (u >= label) break;
            label = u;
        }
        active[v] = label < v;
        cc[v] = label;
        ubm[v] = 0;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) *state = TraverseState{everything(), 2, 1, 0, 0.0};
}

// *one_way = whether one of kCcSampled edges, the middle ones of the in-rows of vertices from all over the graph, has no reverse.
constexpr int kCcSampled = 256;
__global__ __launch_bounds__(kCcSampled) void cc_sample_kernel(int n, Rows rows, int *one_way)
{
    const int64_t v = (int64_t)threadIdx.x * (n > kCcSampled ? n / kCcSampled : 1);
    if (v >= n) return;
    const unsigned int e0 = rows.in_index[v], e1 = rows.in_index[v + 1], i = (e1 - e0) / 2;
    if (e0 < e1 && !rows.leads_back(rows.in_src[e0 + i], (int)v, i)) *one_way = 1;
}

// The root of v, which hands on how far it has come: walkers below take it from there, so a chain of d parents takes about
// log2(d) steps.  Where a walk is long, what the other XCDs have stored counts, so loads and stores go past the L2.
__device__ __forceinline__ int walk_to_root(int *cc, int v)
{
    int p = parent_of(cc, v);
    for (int step = 0;; ++step) {
        const bool far = step >= 8;
        const int up = far ? __hip_atomic_load(cc + p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : parent_of(cc, p);
        if (up == p) return p;
        p = up;
        if (far) __hip_atomic_store(cc + v, p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        else __hip_atomic_store(cc + v, p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
}

__host__ __device__ __forceinline__ int sample_stride(int n) { return n / kCcSamples > 0 ? n / kCcSamples : 1; }

// look_up: cc_begin has just made the parents, so that they are the first entries of the in-rows.
__global__ __launch_bounds__(kSpmvBlock) void cc_flatten_kernel(int n, Rows rows, int *cc, CcTrees *trees, int call, bool look_up)
{
    const int stride = sample_stride(n);
    for (int v = blockIdx.x * kSpmvBlock + threadIdx.x; v < n; v += gridDim.x * kSpmvBlock) {
        const int parent = parent_of(cc, v), root = walk_to_root(cc, v);  // nobody else writes cc[v]
        if (v % stride == 0 && v / stride < kCcSamples) trees->sample[v / stride] = root;
        if (look_up && root != 0 && parent != v && parent_of(&trees->directed, 0) != call && !rows.leads_back(parent, v, 0))
            trees->directed = call;
    }
}

// Joins the trees of a and b.  The larger of the two goes up its tree until it is the other one or a root, which becomes a child of
// the other: each step lowers the larger, so it ends; whether a is still a root is for the compare-and-swap at the memory
// side to say.
__device__ __forceinline__ bool join_trees(int *cc, int a, int b)
{
    for (int step = 0; step < kCcSteps; ++step) {
        if (a == b) return true;
        const int high = a > b ? a : b, low = a > b ? b : a;
        int up = parent_of(cc, high);
        if (up == high) {
            up = atomicCAS(cc + high, high, low);
            if (up == high) return true;
        }
        a = up;
        b = low;
    }
    return false;
}

// Rows are dealt out by length, as in pull_open_kernel.  Vertices of the tree that most samples lie in - after cc_begin usually
// most of a component with hubs - are left out: an edge from it to a vertex of another tree is in that vertex's in-row, an edge from
// there to it in that vertex's out-row, which is looked through for those that do not come back.  A root that has been made a
// child of that tree meanwhile is left out too, so this holds for edges between any two trees: whichever of an edge's ends is looked
// at sees it, and if neither is, both are in that tree.
constexpr int kLinkThreads = 256, kLinkBlocks = 2048;
constexpr int kLinkLane = 8, kLinkWave = 2048;  // entries up to which a row gets a lane, a wavefront
__global__ __launch_bounds__(kLinkThreads) void cc_link_kernel(int n, Rows rows, int *cc, CcTrees *trees, int call, int pass)
{
    constexpr int kWaves = kLinkThreads / kWave;
    __shared__ int s_wave[kLinkThreads], s_block[kLinkThreads];
    __shared__ int s_waves, s_blocks, s_over;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    if (tid == 0) s_over = trees->directed == call;  // read once: other work-groups may set it meanwhile
    const int stride = sample_stride(n), samples = (n - 1) / stride + 1 < kCcSamples ? (n - 1) / stride + 1 : kCcSamples;
    const int mine = lane < samples ? trees->sample[lane] : -1;
    int left_out = -1, most = 0;
    for (int k = 0; k < samples; ++k) {
        const int root = __builtin_amdgcn_readlane(mine, k), count = __popcll(__ballot(mine == root));
        if (count > most) {
            most = count;
            left_out = root;
        }
    }
    const auto edge = [&](int v, unsigned int i, int a, int u, int b) {  // entry i of v's row; roots a, b
        if (a == b) return;
        if (!rows.leads_back(u, v, i)) trees->directed = call;
        else if (!join_trees(cc, a, b)) trees->again = pass;
    };
    const auto leaves = [&](int a, unsigned int i, int u, int b, unsigned int e0, unsigned int e1) {  // entry i of an out-row
        if (b != a && !rows.comes_back(u, i, e0, e1)) trees->directed = call;
    };
    const auto walk = [&](int row, int first, int lanes) {
        const unsigned int e0 = rows.in_index[row], e1 = rows.in_index[row + 1];
        const int a = parent_of(cc, row);
        for (unsigned int e = e0 + first; e < e1; e += 2 * lanes) {
            const bool two = e + lanes < e1;
            const int u0 = rows.in_src[e], u1 = rows.in_src[two ? e + lanes : e];
            const int b0 = parent_of(cc, u0), b1 = parent_of(cc, u1);
            edge(row, e - e0, a, u0, b0);
            if (two) edge(row, e + lanes - e0, a, u1, b1);
        }
        const unsigned int d0 = rows.index[row], d1 = rows.index[row + 1];
        for (unsigned int d = d0 + first; d < d1; d += 2 * lanes) {
            const bool two = d + lanes < d1;
            const int u0 = rows.dst[d], u1 = rows.dst[two ? d + lanes : d];
            const int b0 = parent_of(cc, u0), b1 = parent_of(cc, u1);
            leaves(a, d - d0, u0, b0, e0, e1);
            if (two) leaves(a, d + lanes - d0, u1, b1, e0, e1);
        }
    };
    __syncthreads();
    if (s_over) return;
    const int64_t pieces = ((int64_t)n + kWave - 1) / kWave, per_pass = (int64_t)kWaves * gridDim.x;
    for (int64_t at = 0; at < pieces; at += per_pass) {
        if (tid == 0) s_waves = s_blocks = 0;
        __syncthreads();
        const int64_t r64 = (at + (int64_t)wave * gridDim.x + blockIdx.x) * kWave + lane;
        if (r64 < n) {
            const int r = (int)r64;
            const int a = parent_of(cc, r);
            if (a != left_out) {
                const unsigned int e0 = rows.in_index[r], e1 = rows.in_index[r + 1], d0 = rows.index[r], d1 = rows.index[r + 1];
                const unsigned int longer = max(e1 - e0, d1 - d0);
                if (longer <= kLinkLane) {
                    for (unsigned int i = 0; i < longer; i += 4) {
                        int u[4], b[4], to[4], c[4];
#pragma unroll
                        for (int k = 0; k < 4; ++k) {
                            u[k] = e0 + i + k < e1 ? rows.in_src[e0 + i + k] : r;
                            to[k] = d0 + i + k < d1 ? rows.dst[d0 + i + k] : r;
                        }
#pragma unroll
                        for (int k = 0; k < 4; ++k) {
                            b[k] = u[k] == r ? a : parent_of(cc, u[k]);
                            c[k] = to[k] == r || to[k] == u[k] ? a : parent_of(cc, to[k]);  // in the second case it comes back
                        }
                        for (int k = 0; k < 4; ++k) {
                            edge(r, i + k, a, u[k], b[k]);
                            leaves(a, i + k, to[k], c[k], e0, e1);
                        }
                    }
                } else if (longer <= kLinkWave) {
                    s_wave[atomicAdd(&s_waves, 1)] = r;
                } else {
                    s_block[atomicAdd(&s_blocks, 1)] = r;
                }
            }
        }
        __syncthreads();
        const int waves = s_waves, blocks = s_blocks;
        for (int i = wave; i < waves; i += kWaves) walk(s_wave[i], lane, kWave);
        for (int i = 0; i < blocks; ++i) walk(s_block[i], tid, kLinkThreads);
        __syncthreads();  // the lists have been read
    }
}

// Labels, cc.cu:16's flags (lowered or not; common.cu:17-31 counts the lowered) and where that leaves the traversal: at its end,
// or with everything still to propagate.
__global__ __launch_bounds__(kSpmvBlock) void cc_finish_kernel(int n, int *cc, int *__restrict__ active, const CcTrees *trees, int call, int pass,
                                                               double *block_part, unsigned int *ticket, Report *report)
{
    __shared__ double s_red[kSpmvBlock / kWave];
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        report->state = TraverseState{trees->directed == call ? everything() : 0ull, 2, 1, 0, 0.0};
        report->again = trees->again == pass;
    }
    double lowered = 0.0;
    for (int v = blockIdx.x * kSpmvBlock + threadIdx.x; v < n; v += gridDim.x * kSpmvBlock) {
        const bool falls = walk_to_root(cc, v) < v;
        active[v] = falls;
        lowered += falls;
    }
    publish_sum(lowered, s_red, block_part, ticket, &report->visited);
}

}  // namespace

#include "traverse_chains.h"

namespace {

// cc.cu:391-404 / sssp.cu:483-496
__global__ __launch_bounds__(kSpmvBlock) void process_messages_kernel(int n, int *__restrict__ active, int *__restrict__ ubm)
{
    for (int i = blockIdx.x * kSpmvBlock + threadIdx.x; i < n; i += gridDim.x * kSpmvBlock) {
        if (ubm[i] != 0) {
            active[i] = 0;
            ubm[i] = 0;
        } else {
            active[i] = -1;
        }
    }
}

// Ends what the host enqueues before it waits: tells it where the traversal stands and, if nothing is left to propagate or
// `always`, counts the vertices with active != 0 (common.cu:17-31, without atomics on one address).
__global__ __launch_bounds__(kSpmvBlock) void report_kernel(int n, bool always, const int *__restrict__ active, const TraverseState *state,
                                                            double *block_part, unsigned int *ticket, Report *report)
{
    __shared__ double s_red[kSpmvBlock / kWave];
    if (blockIdx.x == 0 && threadIdx.x == 0) report->state = *state;
    if (!always && state->listed != 0) return;
    double cnt = 0.0;
    for (int i = blockIdx.x * kSpmvBlock + threadIdx.x; i < n; i += gridDim.x * kSpmvBlock) cnt += active[i] != 0;
    publish_sum(cnt, s_red, block_part, ticket, &report->visited);
}

__global__ void iota_kernel(int *out, int n)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) out[i] = i;
}

// Lengths other than 1.0, and kNotWhole or kNegative for some: this lane's share of TraverseState::not_one (len is 16-byte aligned).
__device__ __forceinline__ double count_other_lengths(int n, const float *__restrict__ len)
{
    constexpr int kInFlight = 2;  // more, or more work-groups: the same within 2 %
    double cnt = 0.0;
    const auto other = [](float v) { return v == 1.0f ? 0.0 : !(v == rintf(v) && fabsf(v) < 0x1p24f) ? 1.0 + kNotWhole : v < 0.0f ? 1.0 + kNegative : 1.0; };
    const float4 *len4 = reinterpret_cast<const float4 *>(len);
    const int quads = n / 4, stride = gridDim.x * kSpmvBlock;
    for (int64_t i = blockIdx.x * kSpmvBlock + threadIdx.x; i < quads; i += (int64_t)kInFlight * stride) {
        float4 v[kInFlight];
#pragma unroll
        for (int k = 0; k < kInFlight; ++k) v[k] = i + (int64_t)k * stride < quads ? len4[i + (int64_t)k * stride] : make_float4(1.0f, 1.0f, 1.0f, 1.0f);
#pragma unroll
        for (int k = 0; k < kInFlight; ++k)
            if (v[k].x != 1.0f || v[k].y != 1.0f || v[k].z != 1.0f || v[k].w != 1.0f) cnt += (other(v[k].x) + other(v[k].y)) + (other(v[k].z) + other(v[k].w));
    }
    if (blockIdx.x == 0 && (int)threadIdx.x < n - 4 * quads) cnt += other(len[4 * quads + threadIdx.x]);
    return cnt;
}
__global__ __launch_bounds__(kSpmvBlock) void count_not_one_kernel(int n, const float *__restrict__ len, double *block_part,
                                                                   unsigned int *ticket, double *out)
{
    __shared__ double s_red[kSpmvBlock / kWave];
    publish_sum(count_other_lengths(n, len), s_red, block_part, ticket, out);
}

// sssp.cu:23-38, the list of the first round - the start vertex if this subgraph holds it (sssp.cu:30) and it has out-edges -, and the
// count of the lengths, which the stores do not wait for.  Distances of 1 M vertices and
// 13 M edges 129 us with two launches, 121 with one; 20,000 vertices 77 and 69.  (The arguments and the launch's size take two lines of 64 bytes, the numbers
// side by side: a third, which every work-group's last steps read, took 0.2 us of 4.7.)
__global__ __launch_bounds__(kSpmvBlock) void sssp_begin_kernel(int n, int hold, const int *__restrict__ global_to_local, int start_id, int edges,
                                                                int *__restrict__ active, float *__restrict__ dist, int *__restrict__ ubm,
                                                                const int *__restrict__ index, int *__restrict__ list, int *__restrict__ offset,
                                                                const float *__restrict__ len, double *block_part, unsigned int *ticket,
                                                                TraverseState *state)
{
    __shared__ double s_red[kSpmvBlock / kWave];
    const int start = global_to_local[start_id];
    for (int i = blockIdx.x * kSpmvBlock + threadIdx.x; i < n; i += gridDim.x * kSpmvBlock) {
        active[i] = i == start ? 0 : -1;
        dist[i] = i == start ? 0.0f : kUnreached;
        ubm[i] = 0;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        const int degree = start >= 0 ? index[start + 1] - index[start] : 0;
        list[0] = start;
        offset[0] = 0;
        state->listed = degree > 0 ? (1ull << 32) + (unsigned long long)degree : 0ull;
        state->mark = 1;
        state->rounds = state->which = 0;
    }
    publish_sum(count_other_lengths(edges, len), s_red, block_part, ticket, [&](double all) {
        state->not_one = all;
        state->hold = state->other_natural() ? hold : 0;
    });
}

__global__ void gather_len_kernel(int n, const int *__restrict__ eid, const float *__restrict__ len,
                                  float *__restrict__ out)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) out[i] = len[eid[i]];
}

constexpr int kListBlocks = 2048;  // most work-groups of the kernels that build a list
constexpr int kSumBlocks = 512;   // most work-groups of the counting kernels

// Per-call scratch of the traversals, hung off CCValues::ext / SSSPValues::ext.
struct TraverseExt {
    double *stat = nullptr;        // device scalar
    double *block_part = nullptr;  // device [kSumBlocks]: parts of the counting kernels
    int blocks = 0;                // work-groups of the passes over the vertices
    Lists lists{};                 // device [n] each; vertices with out-edges only
    unsigned long long *counters = nullptr; // device: vertices << 32 | out-edges of the list being built; zero between launches
    unsigned int *ticket = nullptr;         // device [ticket_words(kListBlocks)]: counters of last_block_done, zero between launches
    TraverseState *state = nullptr;         // device
    CcTrees *trees = nullptr;               // device
    int call = 0, pass = 0;                 // of the tree kernels, counted: what *trees names them by
    Report *report = nullptr;               // pinned
};

double seconds_since(std::chrono::steady_clock::time_point t0)
{
    return std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
}

void die(const char *what)
{
    printf("Failed: %s: %s\n", what, drone_last_error_string());
    exit(EXIT_FAILURE);
}

void allow_small_lds();  // of push_rounds_small_kernel, on the current device

// sampled: rows of which report->again says, for a start, whether some edges have no reverse.  A graph with many of them is so spared the
// launches and the wait in which its first call would find out; the sample is taken while the arrays are allocated.  us of the first
// call on a new graph without / with it (by rounds alone): 300,007 vertices and 3 M directed edges 240 / 210 (214), 1 M and 16.5 M
// 343 / 318 (346), one worker of a cut of 500,009 into two 271 / 236 (234), into four 248 / 220 (217); both ways 217 / 219 (288).
TraverseExt *traverse_ext_create(int n, const Rows *sampled = nullptr)
{
    allow_small_lds();
    TraverseExt *t = new TraverseExt();
    t->blocks = (int)ceil_div(n > 0 ? n : 1, kSpmvBlock * 4);
    if (t->blocks > 4096) t->blocks = 4096;
    DRONE_HIP_OR_DIE(hipHostMalloc(&t->report, sizeof(Report)));
    *t->report = Report{};
    if (sampled && n > 0) cc_sample_kernel<<<1, kCcSampled>>>(n, *sampled, &t->report->again);
    DRONE_HIP_OR_DIE(hipMalloc(&t->stat, sizeof(double)));
    DRONE_HIP_OR_DIE(hipMalloc(&t->block_part, sizeof(double) * (size_t)kSumBlocks));
    const size_t cnt = ((size_t)(n > 0 ? n : 1) + 63) & ~(size_t)63;
    DRONE_HIP_OR_DIE(hipMalloc(&t->lists.vertex[0], sizeof(int) * 4 * cnt));  // one allocation
    t->lists.vertex[1] = t->lists.vertex[0] + cnt;
    t->lists.offset[0] = t->lists.vertex[1] + cnt;
    t->lists.offset[1] = t->lists.offset[0] + cnt;
    DRONE_HIP_OR_DIE(hipMalloc(&t->counters, sizeof(unsigned long long)));
    DRONE_HIP_OR_DIE(hipMemset(t->counters, 0, sizeof(unsigned long long)));
    DRONE_HIP_OR_DIE(hipMalloc(&t->state, sizeof(TraverseState)));
    DRONE_HIP_OR_DIE(hipMalloc(&t->trees, sizeof(CcTrees)));
    DRONE_HIP_OR_DIE(hipMemset(t->trees, 0, sizeof(CcTrees)));
    DRONE_HIP_OR_DIE(hipMalloc(&t->ticket, sizeof(unsigned int) * ticket_words(kListBlocks)));
    DRONE_HIP_OR_DIE(hipMemset(t->ticket, 0, sizeof(unsigned int) * ticket_words(kListBlocks)));
    DRONE_HIP_OR_DIE(hipStreamSynchronize(nullptr));  // the kernels that count may run on any stream
    return t;
}

void traverse_ext_destroy(void *ext)
{
    TraverseExt *t = static_cast<TraverseExt *>(ext);
    if (!t) return;
    (void)hipFree(t->stat);
    (void)hipFree(t->block_part);
    (void)hipFree(t->lists.vertex[0]);
    (void)hipFree(t->counters);
    (void)hipFree(t->ticket);
    (void)hipFree(t->state);
    (void)hipFree(t->trees);
    (void)hipHostFree(t->report);
    delete t;
}

int sum_blocks(int64_t n, int per_lane = 4) { return (int)std::min<int64_t>(std::max<int64_t>(ceil_div(n, (int64_t)kSpmvBlock * per_lane), 1), kSumBlocks); }

void launch_report(Graph *g, TraverseExt *t, bool always, hipStream_t s)
{
    const int n = getLocalVertexSize(g);
    report_kernel<<<sum_blocks(n), kSpmvBlock, 0, s>>>(n, always, g->active, t->state, t->block_part, t->ticket, t->report);
}

int count_active(Graph *g, TraverseExt *t, hipStream_t s)
{
    launch_report(g, t, true, s);
    DRONE_HIP_OR_DIE(hipStreamSynchronize(s));
    return (int)t->report->visited;
}

// ---- push direction ---------------------------------------------------------------------------------------
// A value's place in the integers' order: what LDS atomics compare.
__device__ __forceinline__ int order_of(int v) { return v; }
__device__ __forceinline__ int order_of(float v)
{
    const int b = __float_as_int(v);
    return b ^ ((b >> 31) & 0x7FFFFFFF);
}

__device__ __forceinline__ int value_of_order(int o, int) { return o; }
__device__ __forceinline__ float value_of_order(int o, float) { return __int_as_float(o ^ ((o >> 31) & 0x7FFFFFFF)); }

struct CcPush {
    using Value = int;
    int *cc;
    __device__ __forceinline__ int load(int v) const { return __atomic_load_n(cc + v, __ATOMIC_RELAXED); }
    __device__ __forceinline__ int at(int v) const { return cc[v]; }
    __device__ __forceinline__ void store(int v, int x) const { cc[v] = x; }
    __device__ __forceinline__ int relax(int val, int) const { return val; }
    __device__ __forceinline__ int lower(int t, int nv) const { return atomicMin(cc + t, nv); }  // cc.cu:35-36
    static constexpr bool kTolerance = false;  // every lowered label propagates
    static __device__ __forceinline__ bool activates(int old, int nv) { return old > nv; }
};

struct SsspPush {
    using Value = float;
    float *dist;
    const float *__restrict__ len;  // out-edge order (g->edgeLen)
    __device__ __forceinline__ float load(int v) const
    {
        return __uint_as_float(__atomic_load_n(reinterpret_cast<unsigned int *>(dist + v), __ATOMIC_RELAXED));
    }
    __device__ __forceinline__ float at(int v) const { return dist[v]; }
    __device__ __forceinline__ void store(int v, float x) const { dist[v] = x; }
    __device__ __forceinline__ float relax(float val, int e) const { return val + len[e]; }
    // sssp.cu:11-21 fatomicMin without its compare-and-swap loop: floats of one sign order like their bits, a negative
    // float's bits are the larger the smaller it is.  Returns the value found.
    __device__ __forceinline__ float lower(int t, float nv) const
    {
        if (__float_as_int(nv) >= 0) return __int_as_float(atomicMin(reinterpret_cast<int *>(dist + t), __float_as_int(nv)));
        return __uint_as_float(atomicMax(reinterpret_cast<unsigned int *>(dist + t), __float_as_uint(nv)));
    }
    // The target counts as updated past the tolerance (sssp.cu:64).
    static constexpr bool kTolerance = true;
    static __device__ __forceinline__ bool activates(float old, float nv) { return old > nv + kRelaxEps; }
};

// Ends a round: the last work-group of a launch that built list `which` leaves the state for the next launch and clears the
// counter.  The counter is all it reads of the other work-groups' work, and it is only ever updated by returning
// agent-scope atomics (see publish_part in spmv_merge.h); the list itself is plain stores, read by the next launch.
// Every work-group has read *state by the time the last one gets here.
__device__ __forceinline__ void end_round(TraverseState *state, int mark, int rounds, int which, unsigned long long *counters,
                                          unsigned int *ticket, int hold = -1)
{
    __syncthreads();  // every wavefront of the work-group has issued its appends (their atomics return before they go on)
    if (!last_block_done(ticket, 1u) || threadIdx.x != 0) return;
    state->listed = __hip_atomic_exchange(counters, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    state->mark = mark;
    state->rounds = rounds;
    state->which = which;
    if (hold >= 0) state->hold = hold;
}

// A work-group's part of the next list: vertices and their out-degrees gathered in LDS, appended with ONE atomic on the
// shared counter.  (One atomic per wavefront with something to append cost 9 ns each, all on one address: 150 us for a
// million frontier edges.)
template <int CAP>
struct ListBuffer {
    int vertex[CAP], degree_before[CAP];
    unsigned long long held;  // vertices << 32 | out-edges
    unsigned long long base;

    __device__ __forceinline__ void add(int v, int degree)
    {
        const unsigned long long p = atomicAdd(&held, (1ull << 32) + (unsigned long long)degree);
        vertex[p >> 32] = v;
        degree_before[p >> 32] = (int)(p & 0xFFFFFFFFull);
    }
    // by all threads, between barriers; leaves the buffer empty
    __device__ __forceinline__ void flush(int *__restrict__ list, int *__restrict__ offset, unsigned long long *counters)
    {
        if (threadIdx.x == 0) {
            unsigned long long at = 0;
            if (held) {
                at = atomicAdd(counters, held);
                asm volatile("" ::"v"((unsigned int)at));  // waited for: end_round counts on it
            }
            base = at;
        }
        __syncthreads();
        const int count = (int)(held >> 32);
        const int v0 = (int)(base >> 32), e0 = (int)(base & 0xFFFFFFFFull);
        for (int i = threadIdx.x; i < count; i += blockDim.x) {
            list[v0 + i] = vertex[i];
            offset[v0 + i] = e0 + degree_before[i];
        }
        __syncthreads();
        if (threadIdx.x == 0) held = 0ull;
        __syncthreads();
    }
};

// List 0 <- vertices with out-edges whose active flag equals `value`; every work-group takes a contiguous range.
constexpr int kCollectBuffer = 2048, kCollectStep = 4 * kSpmvBlock;
__global__ __launch_bounds__(kSpmvBlock) void collect_frontier_kernel(int n, const int *__restrict__ active, int value,
                                                                      const int *__restrict__ index, Lists lists,
                                                                      unsigned long long *counters, unsigned int *ticket,
                                                                      TraverseState *state, int next_mark, int rounds)
{
    __shared__ ListBuffer<kCollectBuffer> s_buf;
    if (threadIdx.x == 0) s_buf.held = 0ull;
    __syncthreads();
    const int per_block = (int)(((int64_t)n + gridDim.x - 1) / gridDim.x);
    const int begin = blockIdx.x * per_block, end = begin + per_block < n ? begin + per_block : n;
    for (int64_t base = begin; base < end; base += kCollectStep) {
        bool take[kCollectStep / kSpmvBlock];
#pragma unroll
        for (int k = 0; k < kCollectStep / kSpmvBlock; ++k) {
            const int64_t v = base + k * kSpmvBlock + threadIdx.x;
            take[k] = v < end && active[v] == value;
        }
#pragma unroll
        for (int k = 0; k < kCollectStep / kSpmvBlock; ++k)
            if (take[k]) {
                const int v = (int)base + k * kSpmvBlock + (int)threadIdx.x;
                const int degree = index[v + 1] - index[v];
                if (degree > 0) s_buf.add(v, degree);
            }
        __syncthreads();
        const bool full = (int)(s_buf.held >> 32) > kCollectBuffer - kCollectStep || base + kCollectStep >= end;
        __syncthreads();  // everyone has read it before anyone adds again
        if (full) s_buf.flush(lists.vertex[0], lists.offset[0], counters);
    }
    end_round(state, next_mark, rounds, 0, counters, ticket, 0);
}

// One push round over a list: a work-group takes kChunk consecutive edges of the list's concatenated out-edges at a time,
// whatever vertices they belong to (hubs are spread, short rows packed).  A target is first looked at with a plain load:
// a value that is not above the new one there never will be (values only fall), whatever the load's age, so only real
// improvements pay for atomics, which are carried out at the memory side.  A target lowered in this round is appended to
// `next` once: its active flag is swapped to this round's mark, and only the lane that changes it appends.
// Lists of at most `above` edges are push_rounds_small_kernel's, of more than `limit` (over whole lengths other than 1.0
// limit_whole) a sweep's: left alone.
// (One wavefront per vertex and 1,024-edge piece, pieces along grid.y, launched 400,000 work-groups for a list of 50,000
// vertices with one hub of 39,000 edges: 70 us per round on the 11.5 M-edge graph, 9 us this way.)
constexpr int kPushThreads = 256;
constexpr int kPushBlocks = 1024;

template <typename Value, int PER>
struct PushShared {
    int start[kPushThreads * PER], edge[kPushThreads * PER];
    Value val[kPushThreads * PER];
    ListBuffer<kPushThreads * PER> buf;
    int first, entries;
};

template <typename Push, int PER>
__device__ __forceinline__ void push_chunks(PushShared<typename Push::Value, PER> &sh, int count, int edges, int mark,
                                            const int *__restrict__ list, const int *__restrict__ offset,
                                            const int *__restrict__ index, const int *__restrict__ dst, const Push &push,
                                            int *__restrict__ active, int *__restrict__ next, int *__restrict__ next_offset,
                                            unsigned long long *counters)
{
    using Value = typename Push::Value;
    constexpr int kChunk = kPushThreads * PER;
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int64_t chunks = ((int64_t)edges + kChunk - 1) / kChunk;
    for (int64_t chunk = blockIdx.x; chunk < chunks; chunk += gridDim.x) {
        const int j0 = (int)(chunk * kChunk), j1 = edges - j0 < kChunk ? edges : j0 + kChunk;
        if (tid < kWave) {  // the listed vertex that holds edge j0, 64 probes at a time
            int lo = 0, hi = count;  // offset[lo] <= j0, and offset[hi] > j0 (offset[count] would be `edges`)
            while (hi - lo > 1) {
                const int step = (hi - lo + kWave - 1) / kWave, at = lo + (lane + 1) * step;
                const unsigned long long below = __ballot(at < hi && offset[at < hi ? at : lo] <= j0);
                lo += __popcll(below) * step;
                hi = lo + step < hi ? lo + step : hi;
            }
            if (lane == 0) {
                sh.first = lo;
                sh.entries = 0;
                sh.buf.held = 0ull;
            }
        }
        __syncthreads();
        const int first = sh.first;
        int mine = 0;
#pragma unroll
        for (int k = 0; k < PER; ++k) {  // every listed vertex has an edge: at most kChunk of them
            const int i = tid + k * kPushThreads;
            if (first + i < count) {
                const int start = offset[first + i] - j0;
                if (start < j1 - j0) {
                    const int v = list[first + i];
                    sh.start[i] = start;
                    sh.edge[i] = index[v] - start;
                    sh.val[i] = push.load(v);
                    mine = i + 1;
                }
            }
        }
        if (mine) atomicMax(&sh.entries, mine);
        __syncthreads();
        const int entries = sh.entries;
        int t[PER], e[PER];
        Value nv[PER], old[PER];
        bool live[PER];
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const int j = tid + k * kPushThreads;
            int lo = 0, hi = entries;
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (sh.start[mid] <= j) lo = mid; else hi = mid;
            }
            live[k] = j < j1 - j0;
            if (!live[k]) lo = 0;
            e[k] = sh.edge[lo] + (live[k] ? j : 0);  // past the list's end: its edge j0 once more
            nv[k] = sh.val[lo];
        }
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            t[k] = dst[e[k]];
            nv[k] = push.relax(nv[k], e[k]);
        }
#pragma unroll
        for (int k = 0; k < PER; ++k) old[k] = push.at(t[k]);
#pragma unroll
        for (int k = 0; k < PER; ++k) live[k] = live[k] && nv[k] < old[k];
#pragma unroll
        for (int k = 0; k < PER; ++k)
            if (live[k]) old[k] = push.lower(t[k], nv[k]);
#pragma unroll
        for (int k = 0; k < PER; ++k)
            if (live[k]) live[k] = Push::activates(old[k], nv[k]) && atomicExch(active + t[k], mark) != mark;
#pragma unroll
        for (int k = 0; k < PER; ++k)
            if (live[k]) {
                const int degree = index[t[k] + 1] - index[t[k]];
                if (degree > 0) sh.buf.add(t[k], degree);
            }
        __syncthreads();
        sh.buf.flush(next, next_offset, counters);
    }
}

template <typename Push>
__global__ __launch_bounds__(kPushThreads) void push_round_kernel(TraverseState *state, unsigned long long above, unsigned long long limit,
                                                                  unsigned long long limit_whole, Lists lists, const int *__restrict__ index,
                                                                  const int *__restrict__ dst, Push push, int *__restrict__ active,
                                                                  unsigned long long *counters, unsigned int *ticket)
{
    using Value = typename Push::Value;
    __shared__ union Shared {
        PushShared<Value, 8> wide;
        PushShared<Value, 1> narrow;
    } s_push;
    const TraverseState now = *state;
    const unsigned long long edges = now.listed & 0xFFFFFFFFull;
    if (edges <= above || edges > (now.other_whole() ? limit_whole : limit)) return;
    const int count = (int)(now.listed >> 32), w = now.which & 1;
    // more than two chunks a work-group: eight edges a lane in flight instead of one (the launch may have been sized for a shorter list)
    if (edges >= 2ull * kPushThreads * gridDim.x)
        push_chunks<Push, 8>(s_push.wide, count, (int)edges, now.mark, lists.vertex[w], lists.offset[w], index, dst, push, active,
                             lists.vertex[w ^ 1], lists.offset[w ^ 1], counters);
    else
        push_chunks<Push, 1>(s_push.narrow, count, (int)edges, now.mark, lists.vertex[w], lists.offset[w], index, dst, push, active,
                             lists.vertex[w ^ 1], lists.offset[w ^ 1], counters);
    end_round(state, now.mark + 1, now.rounds + 1, w ^ 1, counters, ticket);
}

// One sweep over the in-edges of the vertices that can still fall (the "open" ones): a vertex's in-neighbours are looked
// at until one settles it.  Most of a sweep over all edges is spent on vertices that have their final value; and of those
// that have not, most find a settling neighbour in a few steps (the bottom-up step of breadth-first search).  It is bound
// by the chains of dependent loads (value, row bounds, neighbour, its value), so rows are spread: a work-group takes
// 64-row pieces from all over the graph (vertices of high degree often sit side by side), rows of up to kPullLane entries
// get a lane, of up to kPullGroup 16 lanes, of up to kPullWave a wavefront, longer ones the work-group.  Lowered vertices are
// listed for the next round on the way.  1 M vertices, 11.5 M edges: 26 us for either of the two sweeps of a shortest-path
// run, 91 for the sweep over all edges; 72 with rows side by side in one work-group and wavefronts for all rows above 16
// entries.
struct CcPull {  // no label is below 0
    using Value = int;
    int *cc;
    __device__ __forceinline__ bool begin(const TraverseState &) { return true; }
    __device__ __forceinline__ int at(int v) const { return cc[v]; }
    __device__ __forceinline__ void store(int v, int x) const { cc[v] = x; }
    __device__ __forceinline__ bool open(int v) const { return v > 0; }
    __device__ __forceinline__ int offer(int u, int) const { return cc[u]; }  // what in-neighbour u offers
    __device__ __forceinline__ bool settles(int x) const { return x <= 0; }
};
struct LevelPull {  // rounds of unit lengths from one start vertex: round k reaches the vertices at distance k, for good
    using Value = float;
    float *dist;
    float level = 0.0f;
    // beyond 2^24 levels are no longer exact
    static constexpr int kMostRounds = (1 << 24) - 1;
    __device__ __forceinline__ bool begin(const TraverseState &s)
    {
        level = (float)(s.rounds + 1);
        return s.not_one == 0.0 && s.rounds < kMostRounds;
    }
    __device__ __forceinline__ float at(int v) const { return dist[v]; }
    __device__ __forceinline__ void store(int v, float x) const { dist[v] = x; }
    __device__ __forceinline__ bool open(float v) const { return v >= kUnreached; }
    __device__ __forceinline__ float offer(int u, float otherwise) const { return dist[u] == level - 1.0f ? level : otherwise; }
    __device__ __forceinline__ bool settles(float x) const { return x == level; }
};
constexpr int kPullThreads = 1024, kPullBlocks = 512;  // all resident at once: an append to the shared counter each
constexpr int kPullList = 2048;
constexpr int kPullLane = 8, kPullGroup = 256, kPullWave = 4096;

// A row that waits for more lanes than one, and what is known of it.
struct OpenRow {
    int vertex;
    unsigned int e0, e1;
    int was;  // order_of
};

template <typename Pull>
__global__ __launch_bounds__(kPullThreads) void pull_open_kernel(TraverseState *state, unsigned long long limit, int n,
                                                                 const int *__restrict__ in_index,
                                                                 const int *__restrict__ in_src, Pull pull,
                                                                 int *__restrict__ active, const int *__restrict__ index,
                                                                 Lists lists, unsigned long long *counters, unsigned int *ticket)
{
    using Value = typename Pull::Value;
    constexpr int kWaves = kPullThreads / kWave;
    __shared__ ListBuffer<kPullList> s_buf;
    __shared__ OpenRow s_group[kPullThreads], s_wave[kPullThreads], s_block[kPullThreads];
    __shared__ int s_groups, s_waves, s_blocks, s_best;
    const TraverseState now = *state;
    if ((now.listed & 0xFFFFFFFFull) <= limit || !pull.begin(now)) return;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    if (tid == 0) s_buf.held = 0ull;
    const auto lower = [&](int r, Value was, Value to) {
        if (!(to < was)) return;
        pull.store(r, to);
        active[r] = now.mark;
        const int degree = index[r + 1] - index[r];
        if (degree > 0) s_buf.add(r, degree);
    };
    // G lanes a row
    const auto walk = [&](auto lanes, const OpenRow *rows, int count) {
        constexpr int G = decltype(lanes)::value;
        const int l = tid & (G - 1);
        for (int i = tid / G; i < count; i += kPullThreads / G) {
            const int row = rows[i].vertex;
            const unsigned int e0 = rows[i].e0, e1 = rows[i].e1;
            const Value was = value_of_order(rows[i].was, Value{});
            Value best = was;
            for (unsigned int base = e0; base < e1; base += 2 * G) {
                int u[2];
                Value x[2];
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const unsigned int e = base + k * G + l;
                    u[k] = in_src[e < e1 ? e : e1 - 1];
                }
#pragma unroll
                for (int k = 0; k < 2; ++k) x[k] = pull.offer(u[k], was);
#pragma unroll
                for (int k = 0; k < 2; ++k) best = x[k] < best ? x[k] : best;
                const unsigned long long settled = __ballot(pull.settles(best));
                if (G == kWave ? settled != 0 : ((settled >> (lane & ~(G - 1))) & ((1ull << (G & 63)) - 1)) != 0) break;
            }
#pragma unroll
            for (int m = G / 2; m > 0; m >>= 1) {
                const Value o = __shfl_xor(best, m, kWave);
                best = o < best ? o : best;
            }
            if (l == 0) lower(row, was, best);
        }
    };
    const int64_t pieces = ((int64_t)n + kWave - 1) / kWave, per_pass = (int64_t)kWaves * gridDim.x;
    for (int64_t pass = 0; pass < pieces; pass += per_pass) {
        if (tid == 0) s_groups = s_waves = s_blocks = 0;
        __syncthreads();
        const int64_t r64 = (pass + (int64_t)wave * gridDim.x + blockIdx.x) * kWave + lane;
        if (r64 < n) {
            const int r = (int)r64;
            const Value was = pull.at(r);
            if (pull.open(was)) {
                const unsigned int e0 = in_index[r], e1 = in_index[r + 1];
                if (e1 - e0 <= kPullLane) {
                    Value best = was;
                    for (unsigned int e = e0; e < e1 && !pull.settles(best); e += 4) {
                        int u[4];
                        Value x[4];
#pragma unroll
                        for (int k = 0; k < 4; ++k) u[k] = in_src[e + k < e1 ? e + k : e1 - 1];
#pragma unroll
                        for (int k = 0; k < 4; ++k) x[k] = pull.offer(u[k], was);
#pragma unroll
                        for (int k = 0; k < 4; ++k) best = x[k] < best ? x[k] : best;
                    }
                    lower(r, was, best);
                } else if (e1 - e0 <= kPullGroup) {
                    s_group[atomicAdd(&s_groups, 1)] = OpenRow{r, e0, e1, order_of(was)};
                } else if (e1 - e0 <= kPullWave) {
                    s_wave[atomicAdd(&s_waves, 1)] = OpenRow{r, e0, e1, order_of(was)};
                } else {
                    s_block[atomicAdd(&s_blocks, 1)] = OpenRow{r, e0, e1, order_of(was)};
                }
            }
        }
        __syncthreads();
        walk(std::integral_constant<int, kWave>{}, s_wave, s_waves);
        walk(std::integral_constant<int, 16>{}, s_group, s_groups);
        for (int i = 0; i < s_blocks; ++i) {  // the same count for all: s_blocks is settled
            const int row = s_block[i].vertex;
            const unsigned int e0 = s_block[i].e0, e1 = s_block[i].e1;
            const Value was = value_of_order(s_block[i].was, Value{});
            if (tid == 0) s_best = order_of(was);
            __syncthreads();
            Value best = was;
            for (unsigned int base = e0; base < e1; base += 4 * kPullThreads) {
                int u[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const unsigned int e = base + k * kPullThreads + tid;
                    u[k] = in_src[e < e1 ? e : e1 - 1];
                }
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const Value x = pull.offer(u[k], was);
                    best = x < best ? x : best;
                }
                if (__syncthreads_or(pull.settles(best))) break;
            }
            if (best < was) atomicMin(&s_best, order_of(best));
            __syncthreads();
            if (tid == 0) lower(row, was, value_of_order(s_best, was));
            __syncthreads();
        }
        __syncthreads();
        const bool full = (int)(s_buf.held >> 32) > kPullList - kPullThreads;
        __syncthreads();  // everyone has read it before anyone adds again
        if (full) s_buf.flush(lists.vertex[0], lists.offset[0], counters);
    }
    __syncthreads();
    s_buf.flush(lists.vertex[0], lists.offset[0], counters);
    end_round(state, now.mark + 1, now.rounds + 1, 0, counters, ticket);
}

// Index and head of a vertex's out-edges, for the rounds of a lone wavefront: one access gives what a hop needs to go on from
// the vertex, where row bounds and then targets are two that wait for each other.
__global__ void first_edges_kernel(int n, const int *__restrict__ index, const int *__restrict__ dst, FirstEdges *__restrict__ first)
{
    for (int v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += gridDim.x * blockDim.x) {
        FirstEdges f{index[v], index[v + 1] - index[v], {-1, -1, -1, -1}, {0, 0}};
#pragma unroll
        for (int k = 0; k < kFirstEdges; ++k)
            if (k < f.degree) f.dst[k] = dst[f.begin + k];
        first[v] = f;
    }
}

// Push rounds of a short list inside ONE launch: a single work-group keeps the list in LDS, builds the next one there and
// goes on with it for as long as it has at most kSmallEdges out-edges and is not empty, up to max_rounds rounds.
// What bounds it is a hop's chain of dependent loads - the edge's target, then the target's value and its row's bounds - so
// everything else stays out of the chain: the lists and the round's new values live in LDS (a hash table finds a target that
// several edges lower), no global atomics (only this work-group writes), and a round's values are stored beside the next
// round's first loads.  Edges are dealt out one per lane across the listed vertices.  While a list has no more edges than a
// wavefront has lanes, the first wavefront goes on alone, without barriers (run_lone).  A hop of a 20,000-vertex path
// 2.0 -> 0.40 us, a round of a 593 x 130 grid 50 -> 2.6 us (lists in global memory, atomics, a wavefront per listed vertex before).
// Ordering: a value or flag is stored by a plain store before a point that waits for it (a barrier, or the lone
// wavefront's own wait), and read behind that point by the same work-group, i.e. through the same L1.
// Longer lists are left alone.  It runs rounds until n + 2 of the call are done.
constexpr int kSmallEdges = 4096, kSmallThreads = 1024;
constexpr int kSmallSlots = 2 * kSmallEdges;  // of the hash table: at most half full
constexpr size_t kSmallLds = sizeof(int) * (5 * kSmallEdges + 2 * kSmallSlots);
constexpr int kNearEdges = 2048, kNearFrom = 64;  // of NearRounds
static_assert(sizeof(int) * (8 * kNearEdges + 2 * kSmallSlots + kNearEdges / 2) <= kSmallLds, "NearRounds' arrays lie where SmallRounds' do");

constexpr int kWarmBytes = 3 << 20;  // of the 4 MB of an XCD's L2
constexpr int64_t kNearBytes = 3 << 20;
constexpr int kFirstEdgesPer = 8;  // see ensure_first_edges

// Inclusive sum over the wavefront's lanes, all of them active.
__device__ __forceinline__ int wave_scan(int v)
{
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // from 1, 2, 4, 8 lanes below in the row of 16
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // lane 15 of the row below to rows 1 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // lane 31 to rows 2 and 3
    return v;
}
// A place in a list in LDS for each lane that wants one, with one addition per wavefront: those of a round's lanes on one address are carried out one
// after the other, which took most of the time of a round of some hundred edges.  All lanes take part.
__device__ __forceinline__ int lanes_take(int *count, bool wants)
{
    const unsigned long long who = __ballot(wants);
    if (who == 0) return 0;
    int base = 0;
    if ((threadIdx.x & (kWave - 1)) == 0) base = atomicAdd(count, __popcll(who));
    base = __builtin_amdgcn_readfirstlane(base);
    return base + __builtin_amdgcn_mbcnt_hi((unsigned)(who >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)who, 0u));
}
// ... and for `degree` > 0 edges of it: place << 32 | first edge
__device__ __forceinline__ unsigned long long lanes_take_edges(unsigned long long *listed, bool wants, int degree)
{
    const unsigned long long who = __ballot(wants);
    if (who == 0) return 0;
    const int mine = wants ? degree : 0, upto = wave_scan(mine);
    unsigned long long base = 0;
    if ((threadIdx.x & (kWave - 1)) == kWave - 1) base = atomicAdd(listed, ((unsigned long long)__popcll(who) << 32) + (unsigned long long)(unsigned)upto);
    const unsigned lo = __builtin_amdgcn_readlane((unsigned)base, kWave - 1), hi = __builtin_amdgcn_readlane((unsigned)(base >> 32), kWave - 1);
    const unsigned place = hi + __builtin_amdgcn_mbcnt_hi((unsigned)(who >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)who, 0u));
    return ((unsigned long long)place << 32) + lo + (unsigned)(upto - mine);
}

struct LoneShared {
    int4 edge[kWave];  // {target or -1, edge, place of the value it starts from, -} of the next round's lanes
    int least[kWave];
    int tag[256];
};

template <typename Push>
struct SmallRounds {
    using Value = typename Push::Value;
    int *s_start, *s_edge, *s_vertex, *s_val, *s_slot_vertex, *s_slot_val;
    Value *s_old;
    unsigned long long *s_counters;  // [2]: of the current list and of the one being built, by turns
    int *s_ends;                     // [2]: lowered vertices that do not propagate (no out-edges, or within the tolerance): kept from the list's far end
    int *s_slight;                   // whether an edge of the round lowers its target within the tolerance
    LoneShared *s_lone;
    const FirstEdges *__restrict__ first;  // null where the graph has none
    const int *__restrict__ index;
    const int *__restrict__ dst;
    Push push;
    int *active;
    int first_mark;

    __device__ __forceinline__ void store(int i, int mark) const
    {
        const int v = s_vertex[i];
        const Value nv = value_of_order(s_val[i], Value{});
        push.store(v, nv);
        if (Push::activates(s_old[i], nv)) active[v] = mark;
    }

    // The work-group runs rounds until the list is too long for it or fits a wavefront; rounds / pending: how many ran,
    // whether the list's values are still to be stored.  Starts and ends behind a barrier.
    __device__ __forceinline__ void run(int max_rounds, int &rounds, bool &pending) const
    {
        constexpr int T = kSmallThreads, PER = kSmallEdges / T;
        const int tid = threadIdx.x;
        for (;;) {
            const int now = rounds & 1, n = (int)(s_counters[now] >> 32), m = (int)(s_counters[now] & 0xFFFFFFFFull), ends = s_ends[now];
            if (n + ends == 0 || m > kSmallEdges || rounds >= max_rounds) break;
            if (m <= kWave && ends <= kWave && m > 0) break;  // a wavefront's work
            int t[PER], e[PER];
            Value nv[PER];
            // the edges' targets, and beside them the stores of the last round's values
#pragma unroll
            for (int k = 0; k < PER; ++k) {
                const int j = tid + k * T;
                if (j < m) {
                    int lo = 0, hi = n;
                    while (hi - lo > 1) {
                        const int mid = (lo + hi) >> 1;
                        if (s_start[mid] <= j) lo = mid; else hi = mid;
                    }
                    e[k] = s_edge[lo] + (j - s_start[lo]);
                    t[k] = dst[e[k]];
                    nv[k] = push.relax(value_of_order(s_val[lo], Value{}), e[k]);
                }
            }
            if (pending) {
                for (int i = tid; i < n; i += T) store(i, first_mark + rounds - 1);
                for (int i = tid; i < ends; i += T) store(kSmallEdges - 1 - i, first_mark + rounds - 1);
            }
            __syncthreads();  // the list has been read and its values are stored
            Value old[PER];
            int r0[PER], r1[PER];
#pragma unroll
            for (int k = 0; k < PER; ++k)
                if (tid + k * T < m) {
                    old[k] = push.at(t[k]);
                    r0[k] = index[t[k]];
                    r1[k] = index[t[k] + 1];
                }
            const auto keep = [&](int k, bool goes) {
                unsigned int slot = ((unsigned int)t[k] * 0x9E3779B1u) >> 19;
                static_assert(kSmallSlots == 1 << 13, "the hash keeps 13 bits");
                int found;
                while ((found = atomicCAS(&s_slot_vertex[slot], -1, t[k])) != -1 && found != t[k]) slot = (slot + 1) & (kSmallSlots - 1);
                if (found == -1) {  // first edge to lower it
                    int i;
                    if (goes && r1[k] > r0[k]) {
                        const unsigned long long p = atomicAdd(&s_counters[now ^ 1], (1ull << 32) + (unsigned long long)(r1[k] - r0[k]));
                        i = (int)(p >> 32);
                        s_start[i] = (int)(p & 0xFFFFFFFFull);
                        s_edge[i] = r0[k];
                    } else {
                        i = kSmallEdges - 1 - atomicAdd(&s_ends[now ^ 1], 1);
                    }
                    s_vertex[i] = t[k];
                    s_old[i] = old[k];
                    s_val[i] = (int)slot;
                }
                atomicMin(&s_slot_val[slot], order_of(nv[k]));
            };
#pragma unroll
            for (int k = 0; k < PER; ++k)
                if (tid + k * T < m && nv[k] < old[k]) {
                    if (Push::activates(old[k], nv[k])) keep(k, true);
                    else *s_slight = 1;
                }
            __syncthreads();  // the next list is complete
            const int n2 = (int)(s_counters[now ^ 1] >> 32);
            int ends2 = s_ends[now ^ 1];
            // (a word of LDS and not __syncthreads_or: that took a 40 x 1,000 grid from 2.31 to 2.74 ms)
            if (Push::kTolerance && *s_slight) {
                // Targets that no edge lowers past the tolerance: their value is stored and goes no further.  After the
                // others, so that a target that one edge lowers a little and another by more is on the list.
                __syncthreads();
#pragma unroll
                for (int k = 0; k < PER; ++k)
                    if (tid + k * T < m && nv[k] < old[k] && !Push::activates(old[k], nv[k])) keep(k, false);
                if (tid == 0) *s_slight = 0;
                __syncthreads();
                ends2 = s_ends[now ^ 1];
            }
            const auto settle = [&](int i) {  // the vertex's value out of its slot, which is emptied
                const int slot = s_val[i];
                s_val[i] = s_slot_val[slot];
                s_slot_val[slot] = INT_MAX;
                s_slot_vertex[slot] = -1;
            };
            for (int i = tid; i < n2; i += T) settle(i);
            for (int i = tid; i < ends2; i += T) settle(kSmallEdges - 1 - i);
            if (tid == 0) {
                s_counters[now] = 0ull;
                s_ends[now] = 0;
            }
            pending = true;
            ++rounds;
            __syncthreads();
        }
    }

    // Orders the lanes' accesses to LDS and memory, which the hardware carries out in a wavefront's program order.
    static __device__ __forceinline__ void lanes_meet()
    {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }

    // The first wavefront runs rounds alone, an edge per lane, while they have at most 64 edges.  A round is a chain: the
    // targets' values and first edges come from memory in one access, lanes with the same target agree on the least value
    // (not if only one lane lowers anything), and each lowered vertex hands its edges to the lanes of the next round through
    // LDS.  Against a list in LDS, searched, hashed and settled like the work-group's, and row bounds and targets fetched one
    // after the other: a hop of a 20,000-vertex path 0.95 -> 0.57 us, 0.40 with the single lowering lane's edges passed on
    // in registers and the L2 warm.  (Four edges per lane, up to 256: a 40 x 1,000 grid took 3.0 ms instead of 2.3.)
    // warm(), run by the other wavefronts beside it, brings the vertices' first edges into this XCD's L2 if they fit: a
    // launch finds it cold.  (Only what nobody writes.)  A branch that is taken costs the lone wavefront a refill of its
    // instructions, so a path's case is the one that falls through: without the hints a hop of distances takes 0.41 us (grids two
    // and five wide 1 % less than with them).  Labels are faster without.
#define DRONE_LONE_EXPECT(condition, value) (Push::kTolerance ? __builtin_expect((condition), (value)) : (condition))
    // Ends with the list in LDS and all values stored.
    __device__ __forceinline__ void run_lone(int max_rounds, int &rounds, bool &pending) const
    {
        const int lane = threadIdx.x, now = rounds & 1;
        const int n = (int)(s_counters[now] >> 32), ends = s_ends[now];
        int m = (int)(s_counters[now] & 0xFFFFFFFFull), t = 0, e = 0, count = 0;
        Value from{}, nv{};
        if (lane < m) {
            int lo = 0, hi = n;
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (s_start[mid] <= lane) lo = mid; else hi = mid;
            }
            e = s_edge[lo] + (lane - s_start[lo]);
            t = dst[e];
            from = value_of_order(s_val[lo], Value{});
        }
        if (pending) {
            if (lane < n) store(lane, first_mark + rounds - 1);
            if (lane < ends) store(kSmallEdges - 1 - lane, first_mark + rounds - 1);
            pending = false;
        }
        lanes_meet();
        // Where the loop's branches lie within 32 bytes decides 3 % of a hop (a 5 x 2,000 grid 1.84 ms at an offset of 0 or 4 bytes, 1.85 at 20, 1.89 at the others).
        asm volatile(".p2align 6");
        for (;;) {
            Value old{};
            FirstEdges f{0, 0, {-1, -1, -1, -1}, {0, 0}};
            if (lane < m) {
                old = push.at(t);
                if (first) {
                    f = first[t];
                } else {
                    f.begin = index[t];
                    f.degree = index[t + 1] - f.begin;
                }
                nv = push.relax(from, e);
            }
            bool lowers = lane < m && nv < old;
            const int mark = first_mark + rounds++;
            const unsigned long long lowering = __ballot(lowers);
            if (DRONE_LONE_EXPECT(__popcll(lowering) > 1, 0)) {
                int leader = lane;
                bool open = lowers;
                int *tag = s_lone->tag + (((unsigned int)t * 0x9E3779B1u) >> 24);
                static_assert(sizeof(s_lone->tag) == sizeof(int) << 8, "the hash keeps 8 bits");
                while (__ballot(open)) {  // one lane of each tag's is settled, and with it all that have its target
                    if (open) __hip_atomic_store(tag, lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    lanes_meet();
                    const int who = open ? __hip_atomic_load(tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) : lane;
                    lanes_meet();
                    if (__shfl(t, who, kWave) == t && open) {
                        leader = who;
                        open = false;
                    }
                }
                if (__ballot(leader != lane)) {
                    s_lone->least[lane] = INT_MAX;
                    lanes_meet();
                    if (lowers) atomicMin(&s_lone->least[leader], order_of(nv));
                    lanes_meet();
                    if (lowers) nv = value_of_order(s_lone->least[leader], Value{});
                    lowers = lowers && leader == lane;
                    lanes_meet();
                }
            }
            const bool goes = Push::kTolerance ? lowers && Push::activates(old, nv) : lowers;
            if (lowers) {
                push.store(t, nv);
                if (!Push::kTolerance) active[t] = mark;
            }
            if (Push::kTolerance && goes) active[t] = mark;
            if (DRONE_LONE_EXPECT(__popcll(lowering) == 1 && rounds < max_rounds, 1)) {  // its edges go to the first lanes, out of registers
                const int who = __ffsll(lowering) - 1, degree = __builtin_amdgcn_readlane(goes ? f.degree : 0, who);
                if (DRONE_LONE_EXPECT(degree <= kWave, 1)) {
                    count = degree > 0;
                    m = degree;
                    if (DRONE_LONE_EXPECT(m == 0, 0)) break;
                    e = __builtin_amdgcn_readlane(f.begin, who) + lane;
                    from = value_of_order(__builtin_amdgcn_readlane(order_of(nv), who), Value{});
                    t = -1;
#pragma unroll
                    for (int k = 0; k < kFirstEdges; ++k) {
                        const int d = __builtin_amdgcn_readlane(f.dst[k], who);
                        if (lane == k) t = d;
                    }
                    if (t < 0 && lane < m) t = dst[e];
                    lanes_meet();
                    continue;
                }
            }
            const int take = goes ? f.degree : 0;
            const int upto = wave_scan(take), before = upto - take;
            m = __builtin_amdgcn_readlane(upto, kWave - 1);
            const unsigned long long taking = __ballot(take > 0);
            count = __popcll(taking);
            if (m == 0 || m > kWave || rounds >= max_rounds) {  // over, or not for this wavefront: the list goes back to LDS
                if (take > 0) {
                    const int i = __popcll(taking & ((1ull << lane) - 1));
                    s_start[i] = before;
                    s_edge[i] = f.begin;
                    s_vertex[i] = t;
                    s_val[i] = order_of(nv);
                }
                break;
            }
#pragma unroll
            for (int k = 0; k < kFirstEdges; ++k)
                if (k < take) s_lone->edge[before + k] = make_int4(f.dst[k], f.begin + k, order_of(nv), 0);
            for (int k = kFirstEdges; __ballot(k < take); ++k)
                if (k < take) s_lone->edge[before + k] = make_int4(-1, f.begin + k, order_of(nv), 0);
            lanes_meet();
            const int4 mine = s_lone->edge[lane];
            lanes_meet();
            if (lane < m) {
                e = mine.y;
                t = mine.x >= 0 ? mine.x : dst[e];
                from = value_of_order(mine.z, Value{});
            }
        }
        if (lane == 0) {
            s_counters[rounds & 1] = ((unsigned long long)count << 32) + (unsigned long long)(unsigned int)m;
            s_counters[(rounds & 1) ^ 1] = 0ull;
            s_ends[0] = s_ends[1] = 0;
        }
    }
#undef DRONE_LONE_EXPECT

    // Touches the lines of the vertices' first edges, until *stop.
    __device__ __forceinline__ void warm(int n, const int *stop) const
    {
        constexpr int kPerLine = 128 / sizeof(FirstEdges);
        if (!first || (int64_t)n * (int)sizeof(FirstEdges) > kWarmBytes) return;
        for (int v = ((int)threadIdx.x - kWave) * kPerLine; v < n; v += (kSmallThreads - kWave) * kPerLine) {
            if (__hip_atomic_load(stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) return;
            asm volatile("" ::"v"(first[v].begin));  // the load stays
        }
    }
};

// Rounds of distances over natural lengths, inside one launch as SmallRounds', but nearest vertices first.  Rounds over all that was lowered lower
// most vertices many times over: on a 23 x 846 grid with lengths 1 ... 16 they relax every edge 51 times, 3,600 a round.  Here a lowered vertex whose
// distance is below a threshold goes on the list, the others wait; when the list is empty the threshold moves past the nearest of them (near and far
// piles, as Davidson, Baxter, Garland and Owens, 2014, split delta-stepping's buckets), by a step that is doubled while lists are shorter than a quarter of the
// lanes and halved when one is longer than the lanes: 1.4 times every edge, 100 a round.  Sums of whole numbers have the same least fixed point in any order, so the distances
// are the same bits.  Every move of the threshold settles the nearest waiting vertex, as no length is negative: it ends.
// A list that would be too long is cut, and what it leaves waits too.  A vertex with more edges than a list may have waits until no other goes on the list in
// front of it, which ends it, and so do n rounds: all go back on the call's list, and the launch ends.  What bounds a round (2 us) is its chain of loads - target and length, then value, row bounds and flag - and two
// barriers.  ms by rounds over all / this, lengths 1 ... 16: a 23 x 846 grid 9.8 / 2.4, 50 x 900 12.0 / 3.1, 100 x 500 7.1 / 2.5, 5 x 2,000 14.3 / 4.6, 12 x 200
// 0.78 / 0.58, 200 x 300 4.7 / 3.6; where a lone wavefront suffices it stays with it (a path of 10,000 3.96 / 4.03).
struct NearRounds {
    int *s_start, *s_edge, *s_vertex, *s_val;           // the list
    int *s_low, *s_slot, *s_low_edge, *s_low_degree;    // lowered vertices, and 2 * out-edges + whether they wait already
    int *s_slot_vertex, *s_slot_val;                    // hash table of the round's targets, kSmallSlots
    unsigned short *s_owner;                            // list entry of an edge of the list, if that entry's edges are few
    unsigned long long *s_list;                         // [2] vertices << 32 | out-edges, of the current list and of the one being built, by turns
    unsigned long long *s_cut;                          // [2] the first entry that found no room: its place << 32 | its first edge, or ~0
    int *s_lows;                                        // [2]
    int *s_fars, *s_fars_kept, *s_least, *s_most;       // s_fars: entries of `far`
    const int *__restrict__ index;
    const int *__restrict__ dst;
    SsspPush push;
    int *active;
    int *far, *waits;                                   // device [n] each: waiting vertices, some no longer or again; waits[v]: v's valid place there + 1, or 0
    int first_mark, n_all;

    static __device__ __forceinline__ unsigned int hash(int v) { return ((unsigned int)v * 0x9E3779B1u) >> 19; }

    // On the list that is being built, if there is room.  All lanes of the wavefront take part.
    __device__ __forceinline__ bool append(int which, bool wants, int v, int edge, int degree, float value) const
    {
        const unsigned long long p = lanes_take_edges(&s_list[which], wants, degree);
        if (!wants) return false;
        const int i = (int)(p >> 32), start = (int)(p & 0xFFFFFFFFull);
        if (i >= kNearEdges || start + degree > kNearEdges) {
            atomicMin(&s_cut[which], p);
            return false;
        }
        s_start[i] = start;
        s_edge[i] = edge;
        s_vertex[i] = v;
        s_val[i] = order_of(value);
        constexpr int kFew = 16;
        if (degree <= kFew)
            for (int k = 0; k < degree; ++k) s_owner[start + k] = (unsigned short)i;
        return true;
    }
    __device__ __forceinline__ unsigned long long listed(int which) const { return s_cut[which] != ~0ull ? s_cut[which] : s_list[which]; }

    // Of the first `fars` waiting places those that are valid: on the list that is being built if their distance is below the threshold and there is room, the others
    // move down to the first *s_fars_kept places.  Begins and ends behind a barrier.
    __device__ __forceinline__ void sift(int fars, int which, float threshold) const
    {
        for (int base = 0; base < fars; base += kSmallThreads) {
            const int i = base + (int)threadIdx.x;
            bool there = i < fars;
            int v = 0, edge = 0, degree = 0;
            float d = 0.0f;
            if (there) {
                v = far[i];
                there = waits[v] == i + 1;
                d = push.at(v);
                edge = index[v];
                degree = index[v + 1] - edge;
            }
            __syncthreads();  // these have been read: places below them may be written
            const bool goes = append(which, there && d < threshold, v, edge, degree, d);
            const int place = lanes_take(s_fars_kept, there && !goes);
            if (there && !goes) far[place] = v;
            if (there) waits[v] = goes ? 0 : place + 1;
        }
        __syncthreads();
    }

    // From a list in s_start ... s_val, s_list[0].  Returns the rounds done; the list and the waiting vertices are left in list, offset and *out.
    __device__ __forceinline__ int run(int *list, int *offset, unsigned long long *out) const
    {
        constexpr int T = kSmallThreads, PER = kNearEdges / T;
        const int tid = threadIdx.x;
        float threshold = -1.0f, step = 0.0f;
        int rounds = 0, flips = 0, longest = 0;  // flips: lists built
        for (;;) {
            const int now = flips & 1, next = now ^ 1;
            const unsigned long long all = listed(now);
            const int n = (int)(all >> 32), m = (int)(all & 0xFFFFFFFFull), fars = *s_fars;
            if ((n == 0 && fars == 0) || rounds >= n_all) break;
            if (n > 0 && fars + m > n_all) {
                // A place for each vertex that may come to wait: those that no longer hold are taken out, and what is left and comes are different vertices.
                if (tid == 0) *s_fars_kept = 0;
                __syncthreads();
                sift(fars, next, -1.0f);
                if (tid == 0) *s_fars = *s_fars_kept;
                __syncthreads();
            }
            if (n > 0) {
                longest = max(longest, m);
                int t[PER], e[PER], r0[PER], r1[PER], waiting[PER];
                float nv[PER], old[PER];
#pragma unroll
                for (int k = 0; k < PER; ++k) {
                    const int j = tid + k * T;
                    if (j < m) {
                        int lo = s_owner[j] < n ? s_owner[j] : 0;
                        if (!(s_start[lo] <= j && (lo + 1 < n ? s_start[lo + 1] : m) > j)) {  // the entry has many edges
                            lo = 0;
                            int hi = n;
                            while (hi - lo > 1) {
                                const int mid = (lo + hi) >> 1;
                                if (s_start[mid] <= j) lo = mid; else hi = mid;
                            }
                        }
                        e[k] = s_edge[lo] + (j - s_start[lo]);
                        t[k] = dst[e[k]];
                        nv[k] = push.relax(value_of_order(s_val[lo], 0.0f), e[k]);
                    }
                }
                if (tid == 0) s_lows[next] = 0;
#pragma unroll
                for (int k = 0; k < PER; ++k)
                    if (tid + k * T < m) {
                        old[k] = push.at(t[k]);
                        r0[k] = index[t[k]];
                        r1[k] = index[t[k] + 1];
                        waiting[k] = waits[t[k]];
                    }
#pragma unroll
                for (int k = 0; k < PER; ++k) {
                    if (k * T >= m) break;
                    unsigned int slot = 0;
                    bool first = false;  // edge to lower its target
                    if (tid + k * T < m && nv[k] < old[k]) {
                        slot = hash(t[k]);
                        int found;
                        while ((found = atomicCAS(&s_slot_vertex[slot], -1, t[k])) != -1 && found != t[k]) slot = (slot + 1) & (kSmallSlots - 1);
                        first = found == -1;
                        atomicMin(&s_slot_val[slot], order_of(nv[k]));
                    }
                    const int i = lanes_take(&s_lows[now], first);
                    if (first) {
                        s_low[i] = t[k];
                        s_slot[i] = (int)slot;
                        s_low_edge[i] = r0[k];
                        s_low_degree[i] = 2 * (r1[k] - r0[k]) + (waiting[k] != 0);
                    }
                }
                __syncthreads();  // the list has been read, the lowered vertices are complete
                const int lows = s_lows[now];
                if (tid == 0) {
                    s_list[now] = 0ull;
                    s_cut[now] = ~0ull;
                }
                for (int base = 0; base < lows; base += T) {
                    const int i = base + tid;
                    int v = 0, degree = 0, edge = 0;
                    bool waited = false;
                    float value = 0.0f;
                    if (i < lows) {
                        const int slot = s_slot[i];
                        v = s_low[i];
                        edge = s_low_edge[i];
                        degree = s_low_degree[i] >> 1;
                        waited = s_low_degree[i] & 1;
                        value = value_of_order(s_slot_val[slot], 0.0f);
                        s_slot_val[slot] = INT_MAX;
                        s_slot_vertex[slot] = -1;
                        push.store(v, value);
                        active[v] = first_mark + rounds;
                    }
                    const bool goes = append(next, degree > 0 && value < threshold, v, edge, degree, value);
                    if (goes && waited) waits[v] = 0;
                    const bool stays = degree > 0 && !goes && !waited;
                    const int place = lanes_take(s_fars, stays);
                    if (stays) {
                        waits[v] = place + 1;
                        far[place] = v;
                    }
                }
                ++rounds;
                ++flips;
                __syncthreads();
                continue;
            }
            // The threshold moves on.
            if (tid == 0) {
                *s_least = INT_MAX;
                *s_most = INT_MIN;
                *s_fars_kept = 0;
                s_list[next] = 0ull;
                s_cut[next] = ~0ull;
                s_lows[next] = 0;
            }
            __syncthreads();
            if (tid == 0) {  // the empty list too (everyone has seen that it is): one that is cut before its first entry has counted what found no room
                s_list[now] = 0ull;
                s_cut[now] = ~0ull;
            }
            for (int i = tid; i < fars; i += T) {
                const int v = far[i];
                if (waits[v] != i + 1) continue;
                const int d = order_of(push.at(v));
                atomicMin(s_least, d);
                atomicMax(s_most, d);
            }
            __syncthreads();
            const float least = value_of_order(*s_least, 0.0f), most = value_of_order(*s_most, 0.0f);
            step = step == 0.0f ? most - least : longest * 4 < T ? 2.0f * step : longest > T ? 0.5f * step : step;
            step = fmaxf(step, 1.0f);
            longest = 0;
            threshold = least + step;
            if (!(threshold > least)) threshold = nextafterf(least, INFINITY);
            sift(fars, next, threshold);
            const bool stuck = (listed(next) >> 32) == 0 && *s_fars_kept > 0;
            if (tid == 0) *s_fars = *s_fars_kept;
            ++flips;
            __syncthreads();
            if (stuck) break;
        }
        // What is left goes back.
        const unsigned long long all = listed(flips & 1);
        const int n = (int)(all >> 32), fars = *s_fars;
        if (tid == 0) *out = all;
        __syncthreads();
        for (int i = tid; i < n; i += T) {
            list[i] = s_vertex[i];
            offset[i] = s_start[i];
        }
        for (int i = tid; i < fars; i += T) {
            const int v = far[i];
            if (waits[v] != i + 1) continue;
            const unsigned long long p = atomicAdd(out, (1ull << 32) + (unsigned long long)(unsigned int)(index[v + 1] - index[v]));
            list[p >> 32] = v;
            offset[p >> 32] = (int)(p & 0xFFFFFFFFull);
        }
        __syncthreads();
        return rounds;
    }
};

// A list of any length: all of it waits at first.  One work-group.
__global__ __launch_bounds__(kSmallThreads) void near_rounds_kernel(TraverseState *state, Lists lists, const int *__restrict__ index,
                                                                   const int *__restrict__ dst, SsspPush push, int *active, int n_all)
{
    extern __shared__ int s_small[];
    __shared__ unsigned long long s_list[2], s_cut[2], s_out;
    __shared__ int s_lows[2], s_fars, s_fars_kept, s_least, s_most;
    const TraverseState start = *state;
    const int tid = threadIdx.x;
    if (start.listed == 0 || start.hold <= 0 || start.rounds < n_all + 2 - start.hold) return;
    if ((start.listed & 0xFFFFFFFFull) <= (unsigned long long)kWave) {  // a lone wavefront's: to be looked at when four times as many rounds have run
        if (tid == 0) state->hold = max(n_all + 2 - 4 * start.rounds, 0);
        return;
    }
    int *list = lists.vertex[start.which & 1], *offset = lists.offset[start.which & 1];
    int *at = s_small;
    const auto take = [&](int words) { int *p = at; at += words; return p; };
    NearRounds nr;
    nr.s_start = take(kNearEdges);
    nr.s_edge = take(kNearEdges);
    nr.s_vertex = take(kNearEdges);
    nr.s_val = take(kNearEdges);
    nr.s_low = take(kNearEdges);
    nr.s_slot = take(kNearEdges);
    nr.s_low_edge = take(kNearEdges);
    nr.s_low_degree = take(kNearEdges);
    nr.s_slot_vertex = take(kSmallSlots);
    nr.s_slot_val = take(kSmallSlots);
    nr.s_owner = reinterpret_cast<unsigned short *>(take(kNearEdges / 2));
    nr.s_list = s_list;
    nr.s_cut = s_cut;
    nr.s_lows = s_lows;
    nr.s_fars = &s_fars;
    nr.s_fars_kept = &s_fars_kept;
    nr.s_least = &s_least;
    nr.s_most = &s_most;
    nr.index = index;
    nr.dst = dst;
    nr.push = push;
    nr.active = active;
    nr.far = lists.vertex[(start.which & 1) ^ 1];
    nr.waits = lists.offset[(start.which & 1) ^ 1];
    nr.first_mark = start.mark;
    nr.n_all = n_all;
    const int n = (int)(start.listed >> 32);
    for (int v = tid; v < n_all; v += kSmallThreads) nr.waits[v] = 0;
    for (int j = tid; j < kNearEdges; j += kSmallThreads) nr.s_owner[j] = 0xFFFF;
    for (int i = tid; i < kSmallSlots; i += kSmallThreads) {
        nr.s_slot_vertex[i] = -1;
        nr.s_slot_val[i] = INT_MAX;
    }
    if (tid == 0) {
        s_list[0] = s_list[1] = 0ull;
        s_cut[0] = s_cut[1] = ~0ull;
        s_lows[0] = s_lows[1] = 0;
        s_fars = n;
    }
    __syncthreads();
    for (int i = tid; i < n; i += kSmallThreads) {  // all of them wait
        const int v = list[i];
        nr.far[i] = v;
        nr.waits[v] = i + 1;
    }
    __syncthreads();
    const int rounds = nr.run(list, offset, &s_out);
    if (tid == 0) {
        state->listed = s_out;
        state->mark = start.mark + rounds;
        // Whatever is left is the other rounds', which have n to go from any distances: no length is negative, so a call may make more than n + 1 in all.
        state->rounds = s_out == 0ull ? min(start.rounds + rounds, n_all) : 0;
        state->hold = 0;
    }
}

template <typename Push>
__global__ __launch_bounds__(kSmallThreads) void push_rounds_small_kernel(TraverseState *state, Lists lists, const int *__restrict__ index,
                                                                         const int *__restrict__ dst, const FirstEdges *__restrict__ first,
                                                                         Push push, int *active, int n_all)
{
    extern __shared__ int s_small[];
    __shared__ LoneShared s_lone;
    __shared__ unsigned long long s_counters[2];
    __shared__ int s_ends[2], s_rounds, s_pending, s_done, s_slight;
    SmallRounds<Push> sr;
    sr.s_start = s_small;
    sr.s_edge = sr.s_start + kSmallEdges;
    sr.s_vertex = sr.s_edge + kSmallEdges;
    sr.s_val = sr.s_vertex + kSmallEdges;
    sr.s_old = reinterpret_cast<typename Push::Value *>(sr.s_val + kSmallEdges);
    sr.s_slot_vertex = sr.s_val + 2 * kSmallEdges;
    sr.s_slot_val = sr.s_slot_vertex + kSmallSlots;
    sr.s_counters = s_counters;
    sr.s_ends = s_ends;
    sr.s_slight = &s_slight;
    sr.s_lone = &s_lone;
    sr.first = first;
    sr.index = index;
    sr.dst = dst;
    sr.push = push;
    sr.active = active;
    const int tid = threadIdx.x;
    const TraverseState start = *state;
    if ((start.listed & 0xFFFFFFFFull) > (unsigned long long)kSmallEdges || start.listed == 0) return;
    const int count = (int)(start.listed >> 32), edges = (int)(start.listed & 0xFFFFFFFFull), mark = start.mark;
    const int max_rounds = n_all + 2 - start.hold - start.rounds;  // the host tells a cycle of negative length by n + 2
    int *list = lists.vertex[start.which & 1], *offset = lists.offset[start.which & 1];
    sr.first_mark = mark;
    for (int i = tid; i < kSmallSlots; i += kSmallThreads) {
        sr.s_slot_vertex[i] = -1;
        sr.s_slot_val[i] = INT_MAX;
    }
    for (int i = tid; i < count; i += kSmallThreads) {
        const int v = list[i];
        sr.s_start[i] = offset[i];
        sr.s_edge[i] = index[v];
        sr.s_val[i] = order_of(push.at(v));
    }
    if (tid == 0) {
        s_counters[0] = ((unsigned long long)count << 32) + (unsigned long long)edges;
        s_counters[1] = 0ull;
        s_ends[0] = s_ends[1] = 0;
        s_done = s_slight = 0;
    }
    __syncthreads();
    int rounds = 0;
    bool pending = false, warmed = false;
    for (;;) {
        const int now = rounds & 1, n = (int)(s_counters[now] >> 32), m = (int)(s_counters[now] & 0xFFFFFFFFull), ends = s_ends[now];
        if (n + ends == 0 || m > kSmallEdges || rounds >= max_rounds) break;
        if (m > 0 && m <= kWave && ends <= kWave) {
            if (tid < kWave) {
                sr.run_lone(max_rounds, rounds, pending);
                if (tid == 0) {
                    s_rounds = rounds;
                    s_pending = pending;
                    __hip_atomic_store(&s_done, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                }
            } else if (!warmed) {
                sr.warm(n_all, &s_done);
            }
            warmed = true;  // or found that it was not worth it
            __syncthreads();
            rounds = s_rounds;
            pending = s_pending != 0;
            __syncthreads();
        } else {
            sr.run(max_rounds, rounds, pending);
        }
    }
    const int now = rounds & 1, n = (int)(s_counters[now] >> 32), ends = s_ends[now];
    if (rounds > 0)
        for (int i = tid; i < n; i += kSmallThreads) {
            list[i] = sr.s_vertex[i];
            offset[i] = sr.s_start[i];
        }
    if (pending) {
        for (int i = tid; i < n; i += kSmallThreads) sr.store(i, mark + rounds - 1);
        for (int i = tid; i < ends; i += kSmallThreads) sr.store(kSmallEdges - 1 - i, mark + rounds - 1);
    }
    if (tid == 0) {
        state->listed = s_counters[now];
        state->mark = mark + rounds;
        state->rounds = start.rounds + rounds;
    }
}

void allow_small_lds()
{
    for (const void *kernel : {reinterpret_cast<const void *>(&push_rounds_small_kernel<CcPush>),
                               reinterpret_cast<const void *>(&push_rounds_small_kernel<SsspPush>), reinterpret_cast<const void *>(&near_rounds_kernel)})
        DRONE_HIP_OR_DIE(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kSmallLds));
}

// A list with at most this many out-edges is pushed along them; for a longer one a sweep costs less: a push costs
// the list's out-edges and two atomics per vertex it lowers, a sweep up to all edges but nothing per vertex.
constexpr unsigned kPullShare = 16;
unsigned long long push_limit(const GraphExt *x) { return std::max((unsigned long long)x->edges / kPullShare, (unsigned long long)kSmallEdges); }
// Over whole lengths other than 1.0, where there are no sweeps over the open vertices, a small graph's lists are all pushed: a sweep
// over all edges is two launches, and a third collects what it lowered.  10,000 vertices, 70,000 edges 200 -> 134 us, a 40 x 1,000
// grid 16.5 -> 13.2 ms; 100,000 vertices, 1.3 M edges 204 -> 228 us, where a list of most edges costs more in atomics.  (Over other
// lengths a sweep takes improvements along that a push leaves, so there what was swept stays swept.)
constexpr unsigned long long kPushAll = 1ull << 19;
// near_rounds_kernel may change the list and its mark behind the host's back, in front of rounds that the host has chosen by what it knew: pushes and the small rounds
// look for themselves, a sweep would run with a mark that has passed.  No list of a graph that near_hold() takes is too long to be pushed, so none is chosen.
static_assert(kNearBytes / 8 < (int64_t)kPushAll, "graphs whose nearest vertices go first have lists that are pushed");
unsigned long long push_limit_whole(const GraphExt *x) { return (unsigned long long)x->edges <= kPushAll ? kPushAll : push_limit(x); }

// List 0 <- the vertices with active == value.
void launch_collect(Graph *g, TraverseExt *t, int value, int next_mark, int rounds, hipStream_t s)
{
    const int n = getLocalVertexSize(g);
    collect_frontier_kernel<<<std::min(t->blocks, 512), kSpmvBlock, 0, s>>>(n, g->active, value, g->index, t->lists, t->counters,
                                                                           t->ticket, t->state, next_mark, rounds);
}

template <typename Pull>
void launch_pull(Graph *g, TraverseExt *t, Pull pull, hipStream_t s)
{
    GraphExt *x = static_cast<GraphExt *>(g->ext);
    pull_open_kernel<Pull><<<(unsigned)std::min<int64_t>(ceil_div(x->n, kPullThreads), kPullBlocks), kPullThreads, 0, s>>>(
        t->state, push_limit(x), x->n, x->in_index, x->in_src, pull, g->active, g->index, t->lists, t->counters, t->ticket);
}

// TraverseState::hold for natural lengths: where rounds of the nearest vertices pay.  For lists that reach a hundred edges or so at a time for hundreds of rounds, on roads
// and grids: at most kFirstEdgesPer edges a vertex, and kNearFrom rounds gone by (a graph with hubs is done after a few tens; 3,000 vertices and 18,000 edges
// 85 -> 221 us from the first round on).  And what a round's targets need - values, flags, row bounds, edges, lengths - within an XCD's L2: beyond,
// one CU waits for each of them (ms before / with them: 100 x 500 7.1 / 2.4, 200 x 300 4.7 / 3.6, but 300 x 400 7.3 / 8.1, 1,000 x 1,000 30 / 93).
int near_hold(const GraphExt *x)
{
    const bool pays = (int64_t)x->edges <= (int64_t)kFirstEdgesPer * x->n && 8ll * x->edges + 12ll * x->n <= kNearBytes;
    return pays ? std::max(x->n + 2 - kNearFrom, 0) : 0;
}

// Runs rounds until nothing changes, from what *t->state says is left to propagate (`now`, if known).  What it takes of `run`:
//   run.push                 the relaxation along out-edges
//   run.sweep(mark)          launches a sweep over all in-edges that marks what it lowers
//   run.speculates(state)    whether pull() may be launched before its round is known to come
//   Run::kSweeps             whether there are rounds that pull() cannot do:
//   run.can_pull(state)      whether it may do the next one
//   run.pull()               launches a sweep over the open vertices that lists what it lowers
// Returns the number of rounds, or -1 when the bound of n + 1 rounds is exceeded (a cycle of negative length).
//
// A wait for the GPU costs ~12 us and a launch that finds nothing to do ~3, so the host enqueues the kinds of rounds that
// usually follow each other - a list grows past what one work-group takes, then past what is worth pushing, and shrinks
// again - and only then waits.  Breadth-first distances over 1 M vertices and 11.5 M edges: 550 us with a wait per round and sweeps
// over all edges, 269 with the kernels here and a wait per round, 128 with the rounds enqueued together; labels of
// 500,009 vertices 880, 440, 244 (where every edge has its reverse, labels need no rounds: see cc_begin_kernel).
template <typename Run>
int run_to_fixed_point(Graph *g, TraverseExt *t, Run &run, TraverseState now, bool known, hipStream_t s)
{
    using Push = decltype(run.push);
    GraphExt *x = static_cast<GraphExt *>(g->ext);
    const int n = x->n;
    const unsigned long long limit = push_limit(x), limit_whole = push_limit_whole(x);
    const auto now_limit = [&] { return now.other_whole() ? limit_whole : limit; };
    const auto small = [&] {
        push_rounds_small_kernel<Push><<<1, kSmallThreads, kSmallLds, s>>>(t->state, t->lists, g->index, g->dst, x->first_edges, run.push,
                                                                            g->active, n);
    };
    const auto push = [&](int times) {  // there are such lists at all if limit > kSmallEdges
        const unsigned long long most = std::min(now_limit(), (unsigned long long)x->edges);
        unsigned blocks = (unsigned)std::min<int64_t>(ceil_div((int64_t)most, kPushThreads), kPushBlocks);
        // Before the lengths are known to the host: for lists of up to limit_whole edges as many work-groups as still draw their tickets from one counter.
        // (Sized by `limit` alone, lists of most of a graph's edges went through a sixteenth of the work-groups: distances over whole lengths, 6,746 vertices and 81,000
        // edges 182 -> 92 us, 17,900 and 160,000 192 -> 143.)
        if (!known) blocks = std::max(blocks, (unsigned)std::min<int64_t>(ceil_div((int64_t)std::min(limit_whole, (unsigned long long)x->edges), kPushThreads), kTicketDirect));
        for (int i = 0; i < times && most > (unsigned long long)kSmallEdges; ++i)
            push_round_kernel<Push><<<blocks, kPushThreads, 0, s>>>(t->state, kSmallEdges, limit, limit_whole, t->lists, g->index, g->dst, run.push,
                                                                  g->active, t->counters, t->ticket);
    };
    int sweeps = 1, pushes = 3;  // per wait: double while nothing else is to be done
    const auto pull_maybe = [&](int times) {
        for (int i = 0; i < times && run.speculates(now) && (unsigned long long)x->edges > limit; ++i) run.pull();
    };
    for (;;) {
        const unsigned long long edges = now.listed & 0xFFFFFFFFull;
        int sweeps_next = 1, pushes_next = 3;
        const auto can_pull = [&] {
            if constexpr (Run::kSweeps) return run.can_pull(now);
            else return true;
        };
        if constexpr (Run::kSweeps)
            if (known && now.hold > 0 && now.rounds >= n + 2 - now.hold) {
                for (int i = 0; i < 3; ++i) {  // they take turns while a lone wavefront suffices
                    if (i > 0) small();
                    near_rounds_kernel<<<1, kSmallThreads, kSmallLds, s>>>(t->state, t->lists, g->index, g->dst, run.push, g->active, n);
                }
            }
        if (!known || edges <= (unsigned long long)kSmallEdges) {
            small();
            push(1);
            pull_maybe(2);
            push(2);
            small();
        } else if (edges <= now_limit()) {
            push(pushes);
            small();
            pushes_next = std::min(2 * pushes, 24);
        } else if (can_pull()) {
            run.pull();
            pull_maybe(1);
            push(3);
            small();
        } else if constexpr (Run::kSweeps) {
            for (int i = 0; i < sweeps; ++i) run.sweep(now.mark + i);
            launch_collect(g, t, now.mark + sweeps - 1, now.mark + sweeps, now.rounds + sweeps, s);
            push(1);
            small();
            sweeps_next = std::min(2 * sweeps, 8);
        }
        sweeps = sweeps_next;
        pushes = pushes_next;
        launch_report(g, t, false, s);
        DRONE_HIP_OR_DIE(hipGetLastError());
        DRONE_HIP_OR_DIE(hipStreamSynchronize(s));
        now = t->report->state;
        known = true;
        if (now.listed == 0) return now.rounds;
        if (now.rounds > n + 1) return -1;
    }
}

void report_rounds(int rounds, const char *who)
{
    if (rounds >= 0) return;
    set_error(DRONE_ERR_INVALID, "%s: no fixed point after n + 1 rounds (a cycle of negative length); the values are "
              "not converged", who);
    printf("%s: no fixed point after n + 1 rounds (a cycle of negative length)\n", who);
}

// Position in the out-edge CSR of every in-edge: a stable sort of the edge numbers by target keeps the
// ascending-source order that the in-edge CSR has inside a row.
void ensure_in_edge_ids(Graph *g, hipStream_t s)
{
    GraphExt *x = static_cast<GraphExt *>(g->ext);
    if (x->in_eid) return;
    const int e = x->edges;
    const size_t cnt = (size_t)(e > 0 ? e : 1);
    int *keys_out = nullptr, *iota = nullptr;
    DRONE_HIP_OR_DIE(hipMalloc(&x->in_eid, sizeof(int) * cnt));
    DRONE_HIP_OR_DIE(hipMalloc(&x->in_len, sizeof(float) * cnt));
    if (e == 0) return;
    DRONE_HIP_OR_DIE(hipMalloc(&keys_out, sizeof(int) * cnt));
    DRONE_HIP_OR_DIE(hipMalloc(&iota, sizeof(int) * cnt));
    iota_kernel<<<1024, 256, 0, s>>>(iota, e);
    size_t tmp_bytes = 0;
    void *tmp = nullptr;
    int bits = 1;
    while (bits < 31 && (1 << bits) < (x->n > 1 ? x->n : 2)) ++bits;
    DRONE_HIP_OR_DIE(rocprim::radix_sort_pairs(nullptr, tmp_bytes, g->dst, keys_out, iota, x->in_eid, (size_t)e, 0,
                                               bits, s));
    DRONE_HIP_OR_DIE(hipMalloc(&tmp, tmp_bytes ? tmp_bytes : 1));
    DRONE_HIP_OR_DIE(rocprim::radix_sort_pairs(tmp, tmp_bytes, g->dst, keys_out, iota, x->in_eid, (size_t)e, 0, bits,
                                               s));
    DRONE_HIP_OR_DIE(hipStreamSynchronize(s));
    (void)hipFree(tmp);
    (void)hipFree(keys_out);
    (void)hipFree(iota);
}

struct CcRun {
    Graph *g;
    TraverseExt *t;
    int *cc;
    hipStream_t s;
    CcPush push{cc};
    bool speculates(const TraverseState &) const { return true; }
    static constexpr bool kSweeps = false;
    void pull() { launch_pull(g, t, CcPull{cc}, s); }
};

Rows rows_of(const Graph *g)
{
    const GraphExt *x = static_cast<const GraphExt *>(g->ext);
    return Rows{x->in_index, x->in_src, g->index, g->dst};
}

// Trees from the least in-neighbours, joined until no edge leads between two of them, or left to the rounds: returns where that
// leaves the traversal.  A pass that gives up on an edge has flattened what was in its way, so the next gets further.  A graph that
// has shown an edge without its reverse is not tried again.
TraverseState join_labels(Graph *g, TraverseExt *t, int *cc, hipStream_t s)
{
    GraphExt *x = static_cast<GraphExt *>(g->ext);
    const int n = x->n;
    const unsigned blocks = (unsigned)std::min<int64_t>(ceil_div(n, kSpmvBlock), 4096);
    if (x->one_way) {
        cc_follow_kernel<<<blocks, kSpmvBlock, 0, s>>>(n, x->in_index, x->in_src, g->active, cc, g->updateByMessage, t->state);
        DRONE_HIP_OR_DIE(hipGetLastError());
        return TraverseState{everything(), 2, 1, 0, 0.0};
    }
    const int call = ++t->call;
    const Rows rows = rows_of(g);
    cc_begin_kernel<<<blocks, kSpmvBlock, 0, s>>>(n, rows, cc, g->updateByMessage, t->state);
    for (bool first = true;; first = false) {
        const int pass = ++t->pass;
        cc_flatten_kernel<<<blocks, kSpmvBlock, 0, s>>>(n, rows, cc, t->trees, call, first);
        cc_link_kernel<<<(unsigned)std::min<int64_t>(ceil_div(n, kLinkThreads), kLinkBlocks), kLinkThreads, 0, s>>>(n, rows, cc, t->trees, call, pass);
        cc_finish_kernel<<<sum_blocks(n, 1), kSpmvBlock, 0, s>>>(n, cc, g->active, t->trees, call, pass, t->block_part, t->ticket, t->report);
        DRONE_HIP_OR_DIE(hipGetLastError());
        DRONE_HIP_OR_DIE(hipStreamSynchronize(s));
        x->one_way = t->report->state.listed != 0;
        if (x->one_way || !t->report->again) return t->report->state;
    }
}

// levels: the rounds start from one vertex, so over unit lengths round k reaches the vertices at distance k.  Whether all
// lengths are 1.0 (as build_graph leaves them) is counted on the device, at the start of such a call and otherwise when a
// sweep first needs to know it, as are the lengths in in-edge order, whose random gather costs more than a whole sweep.
struct SsspRun {
    Graph *g;
    TraverseExt *t;
    float *dist;
    hipStream_t s;
    bool levels;
    SsspPush push{dist, g->edgeLen};
    bool counted = false, gathered = false;
    static constexpr bool kSweeps = true;

    void count_lengths()
    {
        GraphExt *x = static_cast<GraphExt *>(g->ext);
        count_not_one_kernel<<<sum_blocks(x->edges, 16), kSpmvBlock, 0, s>>>(x->edges, g->edgeLen, t->block_part, t->ticket, &t->state->not_one);
        counted = true;
    }
    bool unit_lengths()  // between waits
    {
        if (!counted) {
            count_lengths();
            launch_report(g, t, false, s);
            DRONE_HIP_OR_DIE(hipStreamSynchronize(s));
        }
        return t->report->state.not_one == 0.0;
    }
    bool speculates(const TraverseState &now) const { return levels && now.not_one == 0.0; }
    bool can_pull(const TraverseState &now) { return levels && now.rounds < LevelPull::kMostRounds && unit_lengths(); }
    void pull() { launch_pull(g, t, LevelPull{dist}, s); }
    void sweep(int mark)
    {
        GraphExt *x = static_cast<GraphExt *>(g->ext);
        ensure_aggregation_ready(g);
        if (unit_lengths()) {
            spmv_merge_launch<MinF32, int, kIpt>(x->mt, x->ms, x->in_index, x->in_src, SsspUnitEpi{{dist, nullptr, g->active, mark}},
                                                 t->stat, s);
            return;
        }
        if (!gathered) {
            ensure_in_edge_ids(g, s);
            gather_len_kernel<<<1024, 256, 0, s>>>(x->edges, x->in_eid, g->edgeLen, x->in_len);
            gathered = true;
        }
        spmv_merge_launch<MinF32, int, kIpt>(x->mt, x->ms, x->in_index, x->in_src, SsspEpi{dist, x->in_len, g->active, mark},
                                             t->stat, s);
    }
};

template <typename Policy, typename T>
void exchange_values(Graph *g, T *vals, int **send_id, int **recv_id, T **send_val, T **recv_val, int workerId,
                     int workerNum, Comm *comm, Response *res)
{
    if (workerNum <= 1) return;  // one subgraph: the reference moves zero elements
    int rc = DRONE_OK;
    if (!*send_id)
        rc = exchange_buffers_create(g, workerNum, send_id, recv_id, reinterpret_cast<void **>(send_val),
                                     reinterpret_cast<void **>(recv_val));
    if (rc == DRONE_OK)
        rc = exchange_phase<Policy>(g, kMirrorToMaster, vals, *send_id, *recv_id, *send_val, *recv_val, workerId,
                                    workerNum, comm, &res->Mirror2MasterSendSize, &res->Mirror2MasterRecvSize);
    if (rc == DRONE_OK)
        rc = exchange_phase<Policy>(g, kMasterToMirror, vals, *send_id, *recv_id, *send_val, *recv_val, workerId,
                                    workerNum, comm, &res->Master2MirrorSendSize, &res->Master2MirrorRecvSize);
    if (rc != DRONE_OK) die("exchange");
}

// The vertices' first edges, for graphs of at most kFirstEdgesPer edges per vertex: there lists of few edges last for many rounds
// (roads, grids, chains); where vertices have more, a list outgrows a wavefront within a few rounds.  Without them
// (no memory, or more than kFirstEdgesMost of it) rounds take an access more: a hop along a path of 20 K / 0.5 M / 2 M vertices
// 0.49 / 0.72 / 0.78 us instead of 0.40 / 0.53 / 0.54; lists too long for a lone wavefront do not read them.  They are made
// before the first launch, which often runs all the rounds there are; 256 MB (8 Mi vertices) is the Infinity Cache, beyond
// which the one access goes to HBM.
constexpr int64_t kFirstEdgesMost = 256 << 20;
void ensure_first_edges(Graph *g, hipStream_t s)
{
    GraphExt *x = static_cast<GraphExt *>(g->ext);
    if (x->first_edges || x->n == 0 || (int64_t)x->edges > (int64_t)kFirstEdgesPer * x->n ||
        (int64_t)sizeof(FirstEdges) * x->n > kFirstEdgesMost)
        return;
    if (hipMalloc(&x->first_edges, sizeof(FirstEdges) * (size_t)x->n) != hipSuccess) {
        (void)hipGetLastError();
        x->first_edges = nullptr;
        return;
    }
    first_edges_kernel<<<(unsigned)std::min<int64_t>(ceil_div(x->n, 256), 2048), 256, 0, s>>>(x->n, g->index, g->dst, x->first_edges);
}

// The chains of a graph, if nearly all its vertices lie in some: distances over them are weighted, and a graph of ends that is not
// much smaller than the graph takes as many rounds as the graph.  A vertex that is not inner for each kChainsPer that
// are leaves at most 3 edges per vertex where it has few, which keeps denser graphs from being looked at at all; chains shorter
// than kChainsLeast hops cost less than looking for them.
constexpr int kChainsPer = 8, kChainsLeast = 256, kChainsEdgesPer = 3;
bool ensure_chains(Graph *g, TraverseExt *t, hipStream_t s)
{
    GraphExt *x = static_cast<GraphExt *>(g->ext);
    Chains &c = x->chains;
    if (c.tried) return c.ready;
    c.tried = true;
    const int n = x->n;
    if (n < kChainsLeast || (int64_t)x->edges > (int64_t)kChainsEdgesPer * n || (int64_t)sizeof(FirstEdges) * n > kFirstEdgesMost) return false;
    const Rows rows = rows_of(g);
    count_inner_kernel<<<sum_blocks(n), kSpmvBlock, 0, s>>>(n, rows, t->block_part, t->ticket, &t->report->visited);
    DRONE_HIP_OR_DIE(hipStreamSynchronize(s));
    const int64_t inner = (int64_t)t->report->visited;
    if ((n - inner) * kChainsPer > n) return false;
    c.most = x->edges - 2 * inner;  // (in a ring, which nothing else reaches, lists have up to two vertices)
    c.arena.want(&c.arc, 2 * (size_t)n);
    c.arena.want(&c.dst, (size_t)x->edges);
    c.arena.want(&c.len, (size_t)x->edges);
    c.arena.want(&c.first, (size_t)n);
    if (c.arena.commit() != hipSuccess) {
        (void)hipGetLastError();
        c.arena.release();
        return false;
    }
    const unsigned blocks = (unsigned)std::min<int64_t>(ceil_div(n, kSpmvBlock), 4096);
    chain_arcs_kernel<<<blocks, kSpmvBlock, 0, s>>>(n, rows, c.arc);
    for (int64_t reach = 1; reach < n; reach *= kChainJumps + 1) chain_jump_kernel<<<blocks, kSpmvBlock, 0, s>>>(n, c.arc);
    chain_edges_kernel<<<blocks, kSpmvBlock, 0, s>>>(n, rows, c.arc, c.dst, c.len, c.first);
    DRONE_HIP_OR_DIE(hipGetLastError());
    return c.ready = true;
}

// Rounds over the ends of the chains until nothing changes, and the inner vertices' distances; false if the lengths are not all 1.0,
// with nothing done.  sssp_begin_kernel has been launched.
bool run_chains(Graph *g, TraverseExt *t, float *dist, int start_id, hipStream_t s)
{
    GraphExt *x = static_cast<GraphExt *>(g->ext);
    Chains &c = x->chains;
    const int n = x->n;
    const Rows rows = rows_of(g);
    const SsspPush push{dist, c.len};
    const unsigned blocks = (unsigned)std::min<int64_t>(ceil_div(c.most, kPushThreads), kPushBlocks);
    const bool long_lists = c.most > kSmallEdges;
    chain_start_kernel<<<1, kWave, 0, s>>>(rows, g->Global2Local, start_id, c.arc, g->active, dist, t->lists.vertex[0], t->lists.offset[0], t->state);
    const auto small = [&] { push_rounds_small_kernel<SsspPush><<<1, kSmallThreads, kSmallLds, s>>>(t->state, t->lists, g->index, c.dst, c.first, push, g->active, n); };
    do {
        small();
        for (int k = 0; k < 3 && long_lists; ++k)
            push_round_kernel<SsspPush><<<blocks, kPushThreads, 0, s>>>(t->state, kSmallEdges, (unsigned long long)c.most, (unsigned long long)c.most, t->lists, g->index,
                                                                      c.dst, push, g->active, t->counters, t->ticket);
        if (long_lists) small();
        chain_fill_kernel<<<sum_blocks(n), kSpmvBlock, 0, s>>>(n, rows, g->Global2Local, start_id, c.arc, g->active, dist, t->state, t->block_part,
                                                              t->ticket, t->report);
        DRONE_HIP_OR_DIE(hipGetLastError());
        DRONE_HIP_OR_DIE(hipStreamSynchronize(s));
        c.other_lengths = t->report->state.not_one != 0.0;
    } while (!c.other_lengths && t->report->state.listed != 0);
    return !c.other_lengths;
}

void ensure_flags(Graph *g)
{
    const size_t cnt = (size_t)(getLocalVertexSize(g) > 0 ? getLocalVertexSize(g) : 1);
    if (!g->active) DRONE_HIP_OR_DIE(hipMalloc(&g->active, sizeof(int) * cnt));
    if (!g->updateByMessage) DRONE_HIP_OR_DIE(hipMalloc(&g->updateByMessage, sizeof(int) * cnt));
}

}  // namespace

// ---- connected components ---------------------------------------------------------------------------------
extern "C" Response CC_PEVal(Graph *g, CCValues *values, int workerId, int workerNum, Comm *comm)
{
    clear_error();
    const auto t0 = std::chrono::steady_clock::now();
    DRONE_HIP_OR_DIE(hipSetDevice(g->GID));
    hipStream_t s = comm ? static_cast<hipStream_t>(comm->s) : nullptr;
    Response res = {};
    const int n = getLocalVertexSize(g);
    ensure_flags(g);
    if (!values->ext) {  // cc.cu:349-351: the state is allocated by this call
        DRONE_HIP_OR_DIE(hipMalloc(&values->ccValue, sizeof(int) * (size_t)(n > 0 ? n : 1)));
        GraphExt *x = static_cast<GraphExt *>(g->ext);
        const Rows rows = rows_of(g);
        TraverseExt *t = traverse_ext_create(n, x->one_way ? nullptr : &rows);
        x->one_way |= t->report->again != 0;
        values->ext = t;
    }
    TraverseExt *t = static_cast<TraverseExt *>(values->ext);
    if (n > 0) {
        const TraverseState now = join_labels(g, t, values->ccValue, s);
        CcRun run{g, t, values->ccValue, s};
        if (now.listed != 0) {
            ensure_first_edges(g, s);
            run_to_fixed_point(g, t, run, now, true, s);
        }
    }
    res.LocalVertexSize = n;
    res.CalTime = (float)seconds_since(t0);
    const auto t1 = std::chrono::steady_clock::now();
    exchange_values<CcExchange>(g, values->ccValue, &values->sendID, &values->recvID, &values->sendCCValue,
                                &values->recvCCValue, workerId, workerNum, comm, &res);
    res.SendTime = (float)seconds_since(t1);
    res.VisitedSize = workerNum <= 1 && t->report->state.listed == 0 ? (int)t->report->visited : count_active(g, t, s);
    return res;
}

extern "C" Response CC_IncEVal(Graph *g, CCValues *values, int workerId, int workerNum, Comm *comm)
{
    clear_error();
    const auto t0 = std::chrono::steady_clock::now();
    DRONE_HIP_OR_DIE(hipSetDevice(g->GID));
    hipStream_t s = comm ? static_cast<hipStream_t>(comm->s) : nullptr;
    Response res = {};
    if (!values->ext) {
        set_error(DRONE_ERR_INVALID, "CC_IncEVal: CC_PEVal has not been called");
        die("CC_IncEVal");
    }
    TraverseExt *t = static_cast<TraverseExt *>(values->ext);
    const int n = getLocalVertexSize(g);
    ensure_first_edges(g, s);
    process_messages_kernel<<<sum_blocks(n), kSpmvBlock, 0, s>>>(n, g->active, g->updateByMessage);
    launch_collect(g, t, 0, 1, 0, s);  // cc.cu:425: the vertices a message activated propagate
    CcRun run{g, t, values->ccValue, s};
    run_to_fixed_point(g, t, run, TraverseState{}, false, s);
    res.LocalVertexSize = n;
    res.CalTime = (float)seconds_since(t0);
    const auto t1 = std::chrono::steady_clock::now();
    exchange_values<CcExchange>(g, values->ccValue, &values->sendID, &values->recvID, &values->sendCCValue,
                                &values->recvCCValue, workerId, workerNum, comm, &res);
    res.SendTime = (float)seconds_since(t1);
    res.VisitedSize = workerNum <= 1 && t->report->state.listed == 0 ? (int)t->report->visited : count_active(g, t, s);
    return res;
}

extern "C" void drone_cc_values_destroy(Graph *g, CCValues *values)
{
    if (!values) return;
    if (g) (void)hipSetDevice(g->GID);
    traverse_ext_destroy(values->ext);
    if (values->ccValue) (void)hipFree(values->ccValue);
    if (values->sendID) (void)hipFree(values->sendID);
    if (values->recvID) (void)hipFree(values->recvID);
    if (values->sendCCValue) (void)hipFree(values->sendCCValue);
    if (values->recvCCValue) (void)hipFree(values->recvCCValue);
    *values = CCValues{};
}

// ---- single-source shortest paths -------------------------------------------------------------------------
extern "C" Response SSSP_PEVal(Graph *g, SSSPValues *values, int startId, int workerId, int workerNum, Comm *comm)
{
    clear_error();
    const auto t0 = std::chrono::steady_clock::now();
    DRONE_HIP_OR_DIE(hipSetDevice(g->GID));
    hipStream_t s = comm ? static_cast<hipStream_t>(comm->s) : nullptr;
    Response res = {};
    const int n = getLocalVertexSize(g), nglobal = getGlobalVertexSize(g);
    if (startId < 0 || startId >= nglobal) {
        set_error(DRONE_ERR_INVALID, "SSSP_PEVal: startId %d is outside [0, %d)", startId, nglobal);
        die("SSSP_PEVal");
    }
    ensure_flags(g);
    if (!values->ext) {  // sssp.cu:408-411
        DRONE_HIP_OR_DIE(hipMalloc(&values->distance, sizeof(float) * (size_t)(n > 0 ? n : 1)));
        values->ext = traverse_ext_create(n);
    }
    TraverseExt *t = static_cast<TraverseExt *>(values->ext);
    GraphExt *x = static_cast<GraphExt *>(g->ext);
    SsspRun run{g, t, values->distance, s, true};
    const auto begin = [&] {
        sssp_begin_kernel<<<std::max(sum_blocks(n), sum_blocks(x->edges, 16)), kSpmvBlock, 0, s>>>(
            n, near_hold(x), g->Global2Local, startId, x->edges, g->active, values->distance, g->updateByMessage, g->index, t->lists.vertex[0],
            t->lists.offset[0], g->edgeLen, t->block_part, t->ticket, t->state);
        run.counted = true;
    };
    const bool chains = ensure_chains(g, t, s) && !x->chains.other_lengths;
    begin();
    if (!chains || !run_chains(g, t, values->distance, startId, s)) {
        if (chains) begin();
        ensure_first_edges(g, s);
        report_rounds(run_to_fixed_point(g, t, run, TraverseState{}, false, s), "SSSP_PEVal");
        x->chains.other_lengths = t->report->state.not_one != 0.0;
    }
    res.LocalVertexSize = n;
    res.CalTime = (float)seconds_since(t0);
    const auto t1 = std::chrono::steady_clock::now();
    exchange_values<SsspExchange>(g, values->distance, &values->sendID, &values->recvID, &values->sendDis,
                                  &values->recvDis, workerId, workerNum, comm, &res);
    res.SendTime = (float)seconds_since(t1);
    res.VisitedSize = workerNum <= 1 && t->report->state.listed == 0 ? (int)t->report->visited : count_active(g, t, s);
    return res;
}

extern "C" Response SSSP_IncEVal(Graph *g, SSSPValues *values, int workerId, int workerNum, Comm *comm)
{
    clear_error();
    const auto t0 = std::chrono::steady_clock::now();
    DRONE_HIP_OR_DIE(hipSetDevice(g->GID));
    hipStream_t s = comm ? static_cast<hipStream_t>(comm->s) : nullptr;
    Response res = {};
    if (!values->ext) {
        set_error(DRONE_ERR_INVALID, "SSSP_IncEVal: SSSP_PEVal has not been called");
        die("SSSP_IncEVal");
    }
    TraverseExt *t = static_cast<TraverseExt *>(values->ext);
    const int n = getLocalVertexSize(g);
    ensure_first_edges(g, s);
    process_messages_kernel<<<sum_blocks(n), kSpmvBlock, 0, s>>>(n, g->active, g->updateByMessage);
    launch_collect(g, t, 0, 1, 0, s);
    SsspRun run{g, t, values->distance, s, false};
    report_rounds(run_to_fixed_point(g, t, run, TraverseState{}, false, s), "SSSP_IncEVal");
    res.LocalVertexSize = n;
    res.CalTime = (float)seconds_since(t0);
    const auto t1 = std::chrono::steady_clock::now();
    exchange_values<SsspExchange>(g, values->distance, &values->sendID, &values->recvID, &values->sendDis,
                                  &values->recvDis, workerId, workerNum, comm, &res);
    res.SendTime = (float)seconds_since(t1);
    res.VisitedSize = workerNum <= 1 && t->report->state.listed == 0 ? (int)t->report->visited : count_active(g, t, s);
    return res;
}

extern "C" void drone_sssp_values_destroy(Graph *g, SSSPValues *values)
{
    if (!values) return;
    if (g) (void)hipSetDevice(g->GID);
    traverse_ext_destroy(values->ext);
    if (values->distance) (void)hipFree(values->distance);
    if (values->sendID) (void)hipFree(values->sendID);
    if (values->recvID) (void)hipFree(values->recvID);
    if (values->sendDis) (void)hipFree(values->sendDis);
    if (values->recvDis) (void)hipFree(values->recvDis);
    *values = SSSPValues{};
}
