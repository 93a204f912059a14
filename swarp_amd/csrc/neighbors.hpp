// neighbors.hpp -- padded radius-neighbour lists of one state and the COO radius graph.
#pragma once
#include "common.hpp"

namespace swarp {

// --------------------------------------------------------------- neighbour lists

// Rows of up to ROWS_WHOLE slots are staged in LDS slot by slot, longer ones packed (RowLds):
// a short row has little to save and its slots leave without being taken apart.  16000 envs x
// 64 agents, us, whole / packed: rows of less than one member, K = 8 16.0 / 16.8, K = 16 20.1 /
// 19.2, K = 32 30 / 23; full rows 16.9 / 18.3, 21.3 / 23.3, 33 / 31; 32000 x 30, K = 13, full
// 14.2 / 16.9.
constexpr int ROWS_WHOLE = 16;

inline size_t neighbors_lds_bytes(int PA, int K)
{
    return K <= ROWS_WHOLE ? (size_t)64 * K * sizeof(int32_t) : row_lds_bytes(PA, K);
}

// Padded lists of one state (NeighborGrid.query_into's brute-force order): each lane finds its
// list, the wave writes the rows of its envs, one contiguous block of idx.  Bound by that write
// and the scan: 16000 envs x 64 agents with K = 16 take 20 us for 82 MB.
template <typename T, int PA>
__global__ __launch_bounds__(64) void k_neighbors(const Cst<T> C, const T *pos, int32_t *idx,
                                                  int32_t *cnt, int32_t *tru)
{
    typedef typename MaskT<PA>::type M;
    constexpr int EPW = 64 / PA;
    __shared__ T lx[64], ly[64];
    extern __shared__ __align__(16) unsigned char smem[];
    const int lane = threadIdx.x, agent = lane % PA, base = lane - agent;
    const int e0 = blockIdx.x * EPW;
    const int env = e0 + lane / PA;
    const bool active = agent < C.A && env < C.E;
    const size_t i = active ? (size_t)env * C.A + agent : 0;
    const bool real = agent < C.A;
    const T px = real ? pos[2 * i] : (T)__builtin_nan(""), py = real ? pos[2 * i + 1] : (T)__builtin_nan("");
    lx[lane] = px;
    ly[lane] = py;
    wave_lds_sync();  // the workgroup is this one wave
    M cd;
    const M incl = scan_all<T, PA>(lx, ly, base, C.A, agent, px, py, C.t_nbr, C.t_nbr, cd);
    M m = cap_list(incl, C.K);
    const int n = m_popc(m), row = (lane / PA) * C.A + agent;
    if (active) {
        cnt[i] = n;
        if (tru) tru[i] = m_popc(incl);
    }
    const int rows = (C.E - e0 < EPW ? C.E - e0 : EPW) * C.A;
    int32_t *const dst = idx + (size_t)e0 * C.A * C.K;
    if (C.K > ROWS_WHOLE) {
        const RowLds R = row_lds(smem, PA, C.K);
        if (active) row_put(R, row, m);
        wave_lds_sync();
        rows_out(dst, R, 0, rows, C.K, lane);
        return;
    }
    int32_t *const slots = (int32_t *)smem;  // [EPW * A][K]
    if (active) {
        int32_t *const mine = slots + row * C.K;
        int k = 0;
        if ((C.K & 3) == 0) {
            // 16 bytes at a time: a quarter of the writes to the few banks the stride leaves
            for (; k < C.K; k += 4) {
                int v[4];
                for (int u = 0; u < 4; ++u) {
                    v[u] = 0;
                    if (k + u < n) {
                        v[u] = m_ctz(m);
                        m &= m - 1;
                    }
                }
                *(int4 *)(mine + k) = make_int4(v[0], v[1], v[2], v[3]);
            }
        }
        for (; k < C.K; ++k) {
            int v = 0;
            if (k < n) {
                v = m_ctz(m);
                m &= m - 1;
            }
            mine[k] = v;
        }
    }
    wave_lds_sync();
    const int total = rows * C.K;
    if (((uintptr_t)dst & 15u) == 0u && (total & 3) == 0) {
        for (int q = lane; q < total / 4; q += 64) ((int4 *)dst)[q] = ((const int4 *)slots)[q];
    } else {
        for (int q = lane; q < total; q += 64) dst[q] = slots[q];
    }
}

template <typename T>
void launch_neighbors(int PA, const Cst<T> &C, const T *p, int32_t *idx, int32_t *cnt,
                      int32_t *tru, hipStream_t st)
{
    const dim3 grid((C.E + (64 / PA) - 1) / (64 / PA));
    const size_t shm = neighbors_lds_bytes(PA, C.K);
    switch (PA) {
    case 4: hipLaunchKernelGGL((k_neighbors<T, 4>), grid, dim3(64), shm, st, C, p, idx, cnt, tru); break;
    case 8: hipLaunchKernelGGL((k_neighbors<T, 8>), grid, dim3(64), shm, st, C, p, idx, cnt, tru); break;
    case 16: hipLaunchKernelGGL((k_neighbors<T, 16>), grid, dim3(64), shm, st, C, p, idx, cnt, tru); break;
    case 32: hipLaunchKernelGGL((k_neighbors<T, 32>), grid, dim3(64), shm, st, C, p, idx, cnt, tru); break;
    default: hipLaunchKernelGGL((k_neighbors<T, 64>), grid, dim3(64), shm, st, C, p, idx, cnt, tru); break;
    }
}

void launch_edge_index(int E, int A, int K, const int32_t *idx, const int32_t *cnt,
                       const int64_t *off, int64_t n_edges, int64_t *out, hipStream_t st);

#ifdef SWARP_EDGE_INDEX_IMPL
__global__ void k_edge_index(int E, int A, int K, const int32_t *idx, const int32_t *cnt,
                             const int64_t *off, int64_t n_edges, int64_t *out)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)E * A) return;
    const int64_t e = (int64_t)(i / A);
    const int64_t n = cnt[i];
    const int64_t o = off[i];
    for (int64_t s = 0; s < n && o + s < n_edges; ++s) {
        out[o + s] = e * A + idx[i * K + s];
        out[n_edges + o + s] = (int64_t)i;
    }
}

void launch_edge_index(int E, int A, int K, const int32_t *idx, const int32_t *cnt,
                       const int64_t *off, int64_t n_edges, int64_t *out, hipStream_t st)
{
    const size_t n = (size_t)E * A;
    hipLaunchKernelGGL(k_edge_index, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, E, A,
                       K, idx, cnt, off, n_edges, out);
}
#endif

}  // namespace swarp
