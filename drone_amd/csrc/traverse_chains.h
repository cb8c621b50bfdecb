// Shortest paths over unit lengths on graphs that are mostly chains (paths, roads between crossings): a chain is taken in one
// step.  Part of traverse.hip.
//
// An inner vertex has edges to and from exactly two others, so a path through it comes in from one and leaves to the other.  A
// maximal run of inner vertices is a chain between two others, its ends, and an edge into it stands for one edge to the far
// end, as long as the chain.  Rounds then run over the ends alone, and every inner vertex has its distance from those of its
// two ends.  A hop costs a round trip to the L2 however it is done, so what counts is the number of hops one after the other:
// a path of 20,000 vertices took 7.9 ms at 0.39 us per hop, and takes 33 us as one edge.  Where the inner vertices are is found once per
// graph, by pointer doubling: 55 us of kernels for that path.
//
// arc 2 v + s: from inner vertex v to its out-neighbour s (0, 1).  Its successor leaves that neighbour on the other side.
#pragma once

namespace {

struct InnerVertex {
    int to[2];
    bool inner;
};
__device__ __forceinline__ InnerVertex inner_vertex(int v, const Rows &rows)
{
    const int d = rows.index[v], s = rows.in_index[v];
    if (rows.index[v + 1] - d != 2 || rows.in_index[v + 1] - s != 2) return InnerVertex{{-1, -1}, false};
    const int a = rows.dst[d], b = rows.dst[d + 1], low = a < b ? a : b, high = a < b ? b : a;
    return InnerVertex{{a, b}, a != b && a != v && b != v && rows.in_src[s] == low && rows.in_src[s + 1] == high};
}

__global__ __launch_bounds__(kSpmvBlock) void count_inner_kernel(int n, Rows rows, double *block_part, unsigned int *ticket, double *out)
{
    __shared__ double s_red[kSpmvBlock / kWave];
    double count = 0.0;
    for (int v = blockIdx.x * kSpmvBlock + threadIdx.x; v < n; v += gridDim.x * kSpmvBlock) count += inner_vertex(v, rows).inner;
    publish_sum(count, s_red, block_part, ticket, out);
}

// arc[a] = {an arc further along the chain, hops to it}; the chain's last arc has itself and 0.  -1 where v is not inner.
__global__ __launch_bounds__(kSpmvBlock) void chain_arcs_kernel(int n, Rows rows, int2 *__restrict__ arc)
{
    for (int v = blockIdx.x * kSpmvBlock + threadIdx.x; v < n; v += gridDim.x * kSpmvBlock) {
        const InnerVertex me = inner_vertex(v, rows);
#pragma unroll
        for (int side = 0; side < 2; ++side) {
            int2 a = make_int2(-1, 0);
            if (me.inner) {
                const InnerVertex next = inner_vertex(me.to[side], rows);
                a = next.inner ? make_int2(2 * me.to[side] + (next.to[0] == v), 1) : make_int2(2 * v + side, 0);
            }
            arc[2 * v + side] = a;
        }
    }
}

__device__ __forceinline__ int2 load_arc(const int2 *arc, int a)  // both words at once: other lanes move them on
{
    const unsigned long long w = __hip_atomic_load(reinterpret_cast<const unsigned long long *>(arc) + a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return make_int2((int)(w & 0xFFFFFFFFull), (int)(w >> 32));
}
__device__ __forceinline__ void store_arc(int2 *arc, int a, int2 x)
{
    __hip_atomic_store(reinterpret_cast<unsigned long long *>(arc) + a, (unsigned long long)(unsigned int)x.x | (unsigned long long)(unsigned int)x.y << 32,
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ bool is_last_arc(int2 there, int a) { return there.x == a && there.y == 0; }

// Every arc moves on kChainJumps times, each time as far as the arc it is at has come: at least kChainJumps + 1 times as far as
// before.  A ring of inner vertices has no last arc; its arcs stop once they are further than a chain can be long.
constexpr int kChainJumps = 15;
__global__ __launch_bounds__(kSpmvBlock) void chain_jump_kernel(int n, int2 *arc)
{
    for (int a = blockIdx.x * kSpmvBlock + threadIdx.x; a < 2 * n; a += gridDim.x * kSpmvBlock) {
        int2 at = load_arc(arc, a);
        if (at.x < 0 || is_last_arc(at, a)) continue;
        for (int k = 0; k < kChainJumps && at.y <= n; ++k) {
            const int2 there = load_arc(arc, at.x);
            if (is_last_arc(there, at.x)) break;
            at = make_int2(there.x, at.y + there.y);
        }
        store_arc(arc, a, at);
    }
}

// The edges of the graph of ends, at the places of the graph's own; vertices of rings stay as they are.
__global__ __launch_bounds__(kSpmvBlock) void chain_edges_kernel(int n, Rows rows, int2 *arc, int *__restrict__ to, float *__restrict__ len,
                                                                 FirstEdges *__restrict__ first)
{
    const auto whole = [&](int a) {  // of an inner vertex: its chain has an end
        const int2 at = load_arc(arc, a);
        return at.x >= 0 && is_last_arc(load_arc(arc, at.x), at.x);
    };
    for (int v = blockIdx.x * kSpmvBlock + threadIdx.x; v < n; v += gridDim.x * kSpmvBlock) {
        if (load_arc(arc, 2 * v).x >= 0) {
            if (whole(2 * v)) continue;
            store_arc(arc, 2 * v, make_int2(-1, 0));
            store_arc(arc, 2 * v + 1, make_int2(-1, 0));
        }
        FirstEdges f{rows.index[v], rows.index[v + 1] - rows.index[v], {-1, -1, -1, -1}, {0, 0}};
        for (int k = 0; k < f.degree; ++k) {
            int w = rows.dst[f.begin + k];
            float hops = 1.0f;
            if (load_arc(arc, 2 * w).x >= 0 && whole(2 * w)) {  // away from v
                const int2 at = load_arc(arc, 2 * w + (rows.dst[rows.index[w]] == v));
                hops = (float)(at.y + 2);
                w = rows.dst[rows.index[at.x >> 1] + (at.x & 1)];
            }
            to[f.begin + k] = w;
            len[f.begin + k] = hops;
            if (k < kFirstEdges) f.dst[k] = w;
        }
        first[v] = f;
    }
}

struct ChainEnd {
    int vertex, hops;
};
__device__ __forceinline__ ChainEnd chain_end(int2 at, const Rows &rows) { return ChainEnd{rows.dst[rows.index[at.x >> 1] + (at.x & 1)], at.y + 1}; }

// After sssp_begin_kernel: an inner start vertex has reached its chain's ends.  Over lengths other than
// 1.0 there is nothing to do here.
__global__ void chain_start_kernel(Rows rows, const int *__restrict__ global_to_local, int start_id, const int2 *__restrict__ arc,
                                   int *__restrict__ active, float *__restrict__ dist, int *__restrict__ list, int *__restrict__ offset,
                                   TraverseState *state)
{
    if (threadIdx.x != 0) return;
    const int start = global_to_local[start_id];
    if (state->not_one != 0.0) {
        state->listed = 0ull;
        return;
    }
    if (start < 0 || arc[2 * start].x < 0) return;
    const ChainEnd end[2] = {chain_end(arc[2 * start], rows), chain_end(arc[2 * start + 1], rows)};
    const bool one = end[0].vertex == end[1].vertex;
    unsigned long long listed = 0ull;
    for (int k = 0; k < (one ? 1 : 2); ++k) {
        const int v = end[k].vertex, hops = one && end[1].hops < end[0].hops ? end[1].hops : end[k].hops;
        dist[v] = (float)hops;
        active[v] = state->mark;
        list[k] = v;
        offset[k] = (int)(listed & 0xFFFFFFFFull);
        listed += (1ull << 32) + (unsigned long long)(rows.index[v + 1] - rows.index[v]);  // it has an edge back into the chain
    }
    state->listed = listed;
    state->mark += 1;
    state->rounds += 1;
}

// Ends what the host enqueues before it waits, like report_kernel.  If the ends have their distances, so do now the inner vertices:
// from either end, and in the start vertex's chain straight from there.
__global__ __launch_bounds__(kSpmvBlock) void chain_fill_kernel(int n, Rows rows, const int *__restrict__ global_to_local, int start_id,
                                                                const int2 *__restrict__ arc, int *__restrict__ active, float *dist,
                                                                const TraverseState *state, double *block_part, unsigned int *ticket,
                                                                Report *report)
{
    __shared__ double s_red[kSpmvBlock / kWave];
    if (blockIdx.x == 0 && threadIdx.x == 0) report->state = *state;
    if (state->listed != 0 || state->not_one != 0.0) return;
    const int start = global_to_local[start_id], mark = state->mark;
    const int2 from = start >= 0 ? arc[2 * start] : make_int2(-1, 0);
    double count = 0.0;
    for (int v = blockIdx.x * kSpmvBlock + threadIdx.x; v < n; v += gridDim.x * kSpmvBlock) {
        const int2 at[2] = {arc[2 * v], arc[2 * v + 1]};
        int flag = active[v];
        if (at[0].x >= 0 && v != start) {
            float least = kUnreached;
#pragma unroll
            for (int side = 0; side < 2; ++side) {
                const ChainEnd end = chain_end(at[side], rows);
                float d = dist[end.vertex] + (float)end.hops;
                if (from.x >= 0 && at[side].x == from.x) {
                    const float straight = (float)(at[side].y > from.y ? at[side].y - from.y : from.y - at[side].y);
                    d = straight < d ? straight : d;
                }
                least = d < least ? d : least;
            }
            if (least < kUnreached) {
                dist[v] = least;
                active[v] = flag = mark;
            }
        }
        count += flag != 0;
    }
    publish_sum(count, s_red, block_part, ticket, &report->visited);
}

}  // namespace
