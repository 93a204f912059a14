// coo.hip -- the COO radius graph of padded neighbour lists for callers that size its tensor
// by the edge count: swarp_edge_count (sums of the list counts, read by the host) and
// swarp_edge_fill (the edges).
//
// A tile is 2048 agents (more where that would give over 1024 tiles).  k_edge_sums leaves one
// sum per tile on the device and, by its own store, in pinned host memory, so the host has the
// edge count after one launch and one wait.  No prefix of single agents goes through memory: a
// workgroup of k_edge_fill adds the tiles before its own, the counts before it in its tile, and
// scans its counts, 512 at a time, from reads that wait for nothing else; a row of up to four
// neighbours is one 16-byte read.
//
// What bounds it: the wait, the launches and the gaps between them, then one line of the lists
// per agent with a neighbour.  Against a library prefix sum (counts widened to 64 bits, the
// scan's two launches, a copy of its last entry: 20 us of kernels and their gaps) and one agent
// per thread (11.8 us): 200 envs x 1000 agents, K = 16, build and edges 63.9 -> 53.2 us; 16000
// x 64, K = 16, 1.0 M counts, sums 3.5 us and edges 11.7 us, 16 builds of a rollout 240 us less.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "swarp_hip.h"

namespace swarp {
int set_error(const char *msg);  // swarp_hip.hip: the message swarp_last_error() returns
}

namespace {

constexpr int EDGE_BLOCK = 256;                    // threads of a workgroup
constexpr int EDGE_PART = 2 * EDGE_BLOCK;          // agents k_edge_fill scans at a time
constexpr int64_t EDGE_TILE = 2048, EDGE_TILES = 1024;

// Agents per tile (a multiple of EDGE_TILE) and how many tiles there are.
int64_t edge_per(int64_t n)
{
    const int64_t most = EDGE_TILE * EDGE_TILES;
    return EDGE_TILE * ((n + most - 1) / most);
}
int64_t edge_tiles(int64_t n) { return (n + edge_per(n) - 1) / edge_per(n); }

// A list count as the number of valid slots of its row (counts from the neighbour kernels
// already lie in [0, K]).
__device__ __forceinline__ int32_t slots_of(int32_t c, int32_t K) { return c < 0 ? 0 : (c > K ? K : c); }

// The thread's share of the sum of cnt[i0 .. i1), i0 a multiple of 4.
__device__ __forceinline__ int64_t share_of(const int32_t *cnt, int64_t i0, int64_t i1, int32_t K)
{
    int64_t v = 0, q1 = i0;
    if (((uintptr_t)cnt & 15u) == 0) {
        q1 = i0 + ((i1 - i0) & ~(int64_t)3);
        for (int64_t q = i0 + 4 * (int)threadIdx.x; q < q1; q += 4 * EDGE_BLOCK) {
            const int4 c = *(const int4 *)(cnt + q);
            v += (int64_t)slots_of(c.x, K) + slots_of(c.y, K) + slots_of(c.z, K) + slots_of(c.w, K);
        }
    }
    for (int64_t q = q1 + (int)threadIdx.x; q < i1; q += EDGE_BLOCK) v += slots_of(cnt[q], K);
    return v;
}

__global__ __launch_bounds__(EDGE_BLOCK) void k_edge_sums(int64_t n, int64_t per, int32_t K,
                                                          const int32_t *cnt, int64_t *sums,
                                                          int64_t *host)
{
    __shared__ int64_t red[EDGE_BLOCK / 64];
    const int64_t i0 = (int64_t)blockIdx.x * per, i1 = i0 + per < n ? i0 + per : n;
    int64_t v = share_of(cnt, i0, i1, K);
    for (int d = 32; d > 0; d >>= 1) v += __shfl_down(v, d, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x != 0) return;
    for (int w = 1; w < EDGE_BLOCK / 64; ++w) v += red[w];
    sums[blockIdx.x] = v;
    host[blockIdx.x] = v;
}

// The `c` edges of agent i of env e from edge o on.
__device__ __forceinline__ void edges_of(int64_t i, int64_t e, int32_t A, int32_t K, int32_t c,
                                         const int32_t *idx, bool rows16, int64_t o,
                                         int64_t n_edges, int64_t *out)
{
    const int32_t *row = idx + i * K;
    if (rows16) {
        for (int s = 0; s < c; s += 4) {
            const int4 j = *(const int4 *)(row + s);
            const int32_t id[4] = {j.x, j.y, j.z, j.w};
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                if (s + u >= c || o + s + u >= n_edges) break;
                out[o + s + u] = e * A + id[u];
                out[n_edges + o + s + u] = i;
            }
        }
        return;
    }
    for (int s = 0; s < c && o + s < n_edges; ++s) {
        out[o + s] = e * A + row[s];
        out[n_edges + o + s] = i;
    }
}

// A workgroup takes per / EDGE_TILE parts of EDGE_PART agents, a quarter of a tile whatever its
// size, so that what it reads again (the counts before it in its tile, the tiles before) stays
// below the counts themselves: of 64 M agents, 0.3 edges an agent, the graph took 1250 us with one
// part a workgroup (and 1037 us with a library's prefix sum), now 600.  ONE: one part, up to 2 M
// agents, compiled without the loop (1.0 M agents, count and fill 26.0 us, looping 27.5).
template <bool ONE>
__global__ __launch_bounds__(EDGE_BLOCK) void k_edge_fill(int64_t n, int64_t per, int32_t A,
                                                          int32_t K, const int32_t *idx,
                                                          const int32_t *cnt, const int64_t *sums,
                                                          int64_t n_edges, int64_t *out)
{
    __shared__ int64_t before[EDGE_BLOCK / 64];
    __shared__ int32_t wsum[2][EDGE_BLOCK / 64];  // by turns: one barrier a part
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int64_t parts = ONE ? 1 : per / EDGE_TILE;
    const int64_t start = (int64_t)blockIdx.x * parts * EDGE_PART, tile = start / per;
    const bool rows16 = (K & 3) == 0 && ((uintptr_t)idx & 15u) == 0;
    int64_t base = 0;  // edges before the part
    for (int64_t p = 0; p < parts; ++p) {
        const int64_t i0 = start + p * EDGE_PART;
        if (i0 >= n) return;
        const int64_t i = i0 + 2 * (int)threadIdx.x;
        const int32_t c0 = i < n ? slots_of(cnt[i], K) : 0;
        const int32_t c1 = i + 1 < n ? slots_of(cnt[i + 1], K) : 0;
        int32_t *const ws = wsum[p & 1];
        if (p == 0) {
            int64_t b = share_of(cnt, tile * per, start, K);
            for (int64_t t = threadIdx.x; t < tile; t += EDGE_BLOCK) b += sums[t];
            for (int d = 32; d > 0; d >>= 1) b += __shfl_down(b, d, 64);
            if (lane == 0) before[wv] = b;
        }
        int32_t v = c0 + c1;
        for (int d = 1; d < 64; d <<= 1) {
            const int32_t y = __shfl_up(v, d, 64);
            if (lane >= d) v += y;
        }
        if (lane == 63) ws[wv] = v;
        __syncthreads();
        if (p == 0)
            for (int w = 0; w < EDGE_BLOCK / 64; ++w) base += before[w];
        int64_t o = base + v - c0 - c1;
        for (int w = 0; w < EDGE_BLOCK / 64; ++w) {
            o += w < wv ? ws[w] : 0;
            base += ws[w];
        }
        if (i < n) {
            const int64_t e0 = i0 / A;  // one 64-bit division per part
            const uint32_t r = (uint32_t)(i - e0 * A);
            edges_of(i, e0 + r / (uint32_t)A, A, K, c0, idx, rows16, o, n_edges, out);
            edges_of(i + 1, e0 + (r + 1) / (uint32_t)A, A, K, c1, idx, rows16, o + c0, n_edges, out);
        }
    }
}

int fail(const char *msg) { return swarp::set_error(msg); }

}  // namespace

extern "C" {

int64_t swarp_edge_tiles(int32_t n_envs, int32_t n_agents)
{
    if (n_envs < 1 || n_agents < 1) return 0;
    return edge_tiles((int64_t)n_envs * n_agents);
}

int swarp_edge_count(int32_t n_envs, int32_t n_agents, int32_t max_neighbors, const int32_t *cnt,
                     int64_t *sums, int64_t *host_sums, int64_t *n_edges, void *stream)
{
    swarp::set_error("");
    if (n_envs < 1 || n_agents < 1 || max_neighbors < 1) return fail("bad sizes");
    if (!cnt || !sums || !host_sums || !n_edges) return fail("pointer arguments must be set");
    void *dev = nullptr;  // an error for memory that is not pinned
    hipError_t e = hipHostGetDevicePointer(&dev, host_sums, 0);
    if (e != hipSuccess || !dev) {
        (void)hipGetLastError();
        return fail("host_sums must be pinned host memory");
    }
    const int64_t n = (int64_t)n_envs * n_agents, tiles = edge_tiles(n);
    hipStream_t st = (hipStream_t)stream;
    hipLaunchKernelGGL(k_edge_sums, dim3((unsigned)tiles), dim3(EDGE_BLOCK), 0, st, n, edge_per(n),
                       max_neighbors, cnt, sums, (int64_t *)dev);
    e = hipGetLastError();
    if (e == hipSuccess) {
        e = hipStreamSynchronize(st);
        // (reported here: not left for the next launch's check to find)
        if (e != hipSuccess) (void)hipGetLastError();
    }
    if (e != hipSuccess) return fail(hipGetErrorString(e));
    int64_t total = 0;
    for (int64_t t = 0; t < tiles; ++t) total += host_sums[t];
    *n_edges = total;
    return 0;
}

int swarp_edge_fill(int32_t n_envs, int32_t n_agents, int32_t max_neighbors, const int32_t *idx,
                    const int32_t *cnt, const int64_t *sums, int64_t n_edges, int64_t *edge_index,
                    void *stream)
{
    swarp::set_error("");
    if (n_envs < 1 || n_agents < 1 || max_neighbors < 1) return fail("bad sizes");
    if (n_edges < 0) return fail("n_edges must be >= 0");
    if (n_edges == 0) return 0;
    if (!idx || !cnt || !sums || !edge_index) return fail("pointer arguments must be set");
    const int64_t n = (int64_t)n_envs * n_agents;
    const int64_t agents = edge_per(n) / EDGE_TILE * EDGE_PART;  // of a workgroup
    const int64_t blocks = (n + agents - 1) / agents;           // (at most 4 EDGE_TILES)
    const dim3 g((unsigned)blocks), b(EDGE_BLOCK);
    hipStream_t st = (hipStream_t)stream;
    if (agents == EDGE_PART)
        hipLaunchKernelGGL((k_edge_fill<true>), g, b, 0, st, n, edge_per(n), n_agents, max_neighbors,
                           idx, cnt, sums, n_edges, edge_index);
    else
        hipLaunchKernelGGL((k_edge_fill<false>), g, b, 0, st, n, edge_per(n), n_agents,
                           max_neighbors, idx, cnt, sums, n_edges, edge_index);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(hipGetErrorString(e));
    return 0;
}

}  // extern "C"
