// swarm.hpp -- the rollout kernels of disc fleets on the wide layout (one workgroup per env,
// wide.hpp): any model, obstacles, walls, clamp, integrator, index- or grid-ordered lists.
// Box worlds keep wide.hpp's own kernels.
//
// What a substep needs of its lists is little: an agent has a few neighbours, and only the
// touching ones exert a force.  The lists' order and cap decide which K members a crowded
// list keeps and the order its forces are added in.
//
// Forward.  Every agent keeps candidates: the agents within the skin radius where it was when
// they were found.  They stay complete until some agent of the env is half the skin away from
// that place, usually for a step or two, and a substep tests the candidates only.  They come
// from a counting sort of the env's agents into square cells at least as wide as the skin
// radius: an agent reads three runs of it, the rows of its 3x3 block.  Cells hold their
// agents in arrival order and candidates come as found, but a list is taken from them by key
// -- the index, or for the uniform grid (slot of the 3x3 block, index), which orders as (slot,
// rank in the cell) does -- so no result depends on it.  An env that overflows its candidate
// lists takes a quarter of the skin (where that pays, see NEAR_FULL) and else falls back, for the
// rest of the rollout, to wide.hpp's traversal of the whole list at every substep: a search in
// vain dearer than that traversal alone, which is 2 to 8 % of a crowded rollout.
//
// Tape.  The forward leaves each substep's total force and the agents it touched (up to
// NEAR_TOUCH ids); the backward then integrates to the substeps' inputs with the recorded
// forces and walks the touching pairs.  With no list truncated each pair acts both ways, so
// own and reverse side are known without the lists.  A record that overflowed, or a
// truncated list, sends the env's substep to the full traversal.  Same terms in the same
// order as without a tape: the same bits.
//
// What bounds it: the dependent chain of a substep between its barriers (4 to 16 waves share
// them), not bandwidth and not issue.  Measured (MI355X, holonomic agents between walls),
// forward / backward, before (every pair tested at every substep, the backward recomputing
// the lists of S (S + 1) / 2 substeps a step) and now: 500 envs x 200 agents, 8 steps of 4
// substeps 595 / 2326 -> 129 / 121 us; 48 x 2000, uniform grid, 8 steps of 2 substeps 519 /
// 1402 -> 213 / 169 us.  Candidates through chains of hashed cells instead of sorted runs
// took 310 and 465 us forward: a chain is a dependent LDS read per agent of the block.
#pragma once
#include "wide.hpp"

namespace swarp {

constexpr int NEAR_MAX = 16;   // candidates an agent keeps (fewer where the LDS is short)
constexpr int NEAR_TOUCH = 8;  // touching agents a tape record holds
constexpr uint32_t NEAR_NONE = 0xffffu, NEAR_SLOW = 0xfffeu;

// Index-ordered envs of up to this many agents whose candidates overflow take no quarter of the
// skin: their full traversal is short.  Forward without gradient, 16 substeps, 60 agents per unit
// area, us, a quarter / the full traversal: 857 envs x 70 agents 262 / 202, 461 x 130 304 / 290,
// and at 15 per unit area and more agents 300 x 200 152 / 352, 60 x 1000 171 / 1833.
constexpr int NEAR_FULL = 128;

// Most cells per axis of the search: about four cells per agent slot (fewer are used where
// the skin radius asks for wider ones; the scan covers those used).
__host__ __device__ inline int near_side(int AP) { return AP <= 128 ? 24 : (AP <= 512 ? 40 : 64); }

// LDS after the positions, velocities and radii (5 AP scalars): candidates, four 16-bit ids to
// a word and `cap / 4` words per agent slot; 16 + 16 + 16 vote words; cell starts; grid cells
// (GRID); the agents sorted by cell.
__host__ __device__ inline size_t near_fixed_bytes(int AP, bool grid)
{
    const int hm = near_side(AP);
    return (48 + (size_t)hm * hm + 1 + (grid ? AP : 0)) * sizeof(int32_t) +
           (size_t)AP * sizeof(uint16_t);
}

// Candidates per agent within the workgroup's LDS (less the static wsum[16]): a multiple of 4.
template <typename T> __host__ __device__ inline int near_cap(int AP, bool grid)
{
    const size_t used = (size_t)5 * AP * sizeof(T) + near_fixed_bytes(AP, grid) + 16 * sizeof(int32_t);
    if (used >= LDS_MAX) return 0;
    const size_t n = (LDS_MAX - used) / ((size_t)AP * sizeof(uint64_t)) * 4;
    return n < (size_t)NEAR_MAX ? (int)n : NEAR_MAX;
}

// Dynamic LDS of the forward: the candidate search and, in its place, the full traversal.
template <typename T> inline size_t swarm_fwd_lds(int AP, int NC)
{
    const bool grid = NC > 0;
    const size_t b = wide_lds_bytes<T>(AP, NC), cap = near_cap<T>(AP, grid);
    if (cap == 0) return b;  // the full traversal from the start
    const size_t a = (size_t)5 * AP * sizeof(T) + near_fixed_bytes(AP, grid) +
                     cap / 4 * AP * sizeof(uint64_t);
    return a > b ? a : b;
}

template <typename T> struct NearLds {
    uint64_t *cand;         // [cap / 4][AP]
    int32_t *moved, *over;  // votes, one word per wave
    int32_t *scan;          // [16] the sort's wave sums
    int32_t *start;         // [cells + 1] first sorted slot of each cell
    uint32_t *cell;         // grid cell of each agent: x | y << 16 (GRID)
    uint16_t *sorted;       // [AP] agents by cell
    int AP, cap;
};

template <typename T, bool GRID>
__device__ __forceinline__ NearLds<T> near_lds(unsigned char *smem, int AP)
{
    NearLds<T> N;
    N.AP = AP;
    N.cap = near_cap<T>(AP, GRID);
    N.cand = (uint64_t *)((T *)smem + 5 * AP);  // (AP a multiple of 64)
    int32_t *p = (int32_t *)(N.cand + N.cap / 4 * AP);
    N.moved = p;
    N.over = p + 16;
    N.scan = p + 32;
    N.start = p + 48;
    p += 48 + near_side(AP) * near_side(AP) + 1;
    N.cell = (uint32_t *)p;
    if (GRID) p += AP;
    N.sorted = (uint16_t *)p;
    return N;
}

// Whether any thread of the workgroup voted true: written before a barrier, read after it.
__device__ __forceinline__ void vote_put(int32_t *v, bool mine)
{
    const uint64_t b = __ballot(mine);
    if ((threadIdx.x & 63) == 0) v[threadIdx.x >> 6] = b != 0;
}
__device__ __forceinline__ bool vote_get(const int32_t *v)
{
    int32_t r = 0;
    for (int w = 0; w < (int)blockDim.x / 64; ++w) r |= v[w];
    return r != 0;
}

// The search's cells and skin.  A position's cell is clamped into the frame, so agents
// outside it are found too (in longer runs); the frame only has to fit where most are.
template <typename T> struct NearGrid {
    T ox, oy, ix, iy;  // origin, cells per unit length
    int nx, ny;
    T t_skin, half2;   // squared skin radius, squared displacement the candidates bear
};

// Cells for a skin of `part` (0 .. 1) of the launch's over a box.  The cells are wider than
// the skin radius by 1/16, far above the roundings of (p - o) * i below 64 cells, so agents
// within the skin radius of each other land at most one cell apart.
template <typename T>
__device__ __forceinline__ NearGrid<T> near_grid(const Cst<T> &C, const Box4<T> &box, T part, int AP)
{
    NearGrid<T> H;
    const T r = m_sqrt(C.t_nbr), skin = (m_sqrt(C.t_skin) - r) * part;
    const T rs = r + skin, w = rs * T(1.0625);
    H.t_skin = wmax(rs * rs, C.t_nbr);
    // (half the skin, less the roundings of r, rs and the squares)
    const T half = wmax(skin * T(0.499) - r * (sizeof(T) == 4 ? T(1e-6) : T(1e-14)), T(0));
    H.half2 = half * half;
    const int most = near_side(AP);
    const T ex = box.mxx - box.mnx, ey = box.mxy - box.mny;
    const T wx = wmax(w, ex / T(most)), wy = wmax(w, ey / T(most));
    H.ox = box.mnx;
    H.oy = box.mny;
    H.ix = T(1) / wx;
    H.iy = T(1) / wy;
    // (an empty box, or a radius or box that is not finite, takes one cell)
    const T qx = ex * H.ix, qy = ey * H.iy;
    const bool cells = w < T(1e30) && wx < T(1e30) && wy < T(1e30);
    H.nx = cells && qx >= T(1) ? (qx < T(most) ? (int)qx + 1 : most) : 1;
    H.ny = cells && qy >= T(1) ? (qy < T(most) ? (int)qy + 1 : most) : 1;
    return H;
}

template <typename T> __device__ __forceinline__ int near_axis(T p, T o, T i, int n)
{
    const T q = (p - o) * i;
    return q >= T(1) ? (q < T(n) ? (int)q : n - 1) : 0;  // (NaN: cell 0)
}

// The candidates of one agent once the sort is complete, as they come.  Returns how many
// there are; those past the list's room are not kept.  A started word is filled up with the
// agent's own id, which every reader skips.  A word is put together in a register and stored
// once: its ids stored one by one as 16-bit values would be accesses of another type than the
// word's, which the compiler may order as it likes.
template <typename T>
__device__ __forceinline__ int near_find(const WideLds<T> &W, const NearLds<T> &N,
                                         const NearGrid<T> &H, int i, T px, T py)
{
    const int cx = near_axis(px, H.ox, H.ix, H.nx), cy = near_axis(py, H.oy, H.iy, H.ny);
    const int x0 = cx > 0 ? cx - 1 : 0, x1 = (cx + 1 < H.nx ? cx + 1 : H.nx - 1) + 1;
    int q0[3], q1[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int y = cy + k - 1;
        const bool in = y >= 0 && y < H.ny;
        const int row = (in ? y : cy) * H.nx;
        q0[k] = N.start[row + x0];
        q1[k] = in ? N.start[row + x1] : q0[k];
    }
    int n = 0;
    const uint64_t own = (uint64_t)i * 0x0001000100010001ull;
    uint64_t word = own;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        for (int q = q0[k]; q < q1[k]; q += 4) {
            // four at a time, so that their reads are waited for together
            int j[4];
            bool hit[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) j[u] = q + u < q1[k] ? N.sorted[q + u] : i;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const T dx = W.px[j[u]] - px, dy = W.py[j[u]] - py;
                hit[u] = dx * dx + dy * dy <= H.t_skin && j[u] != i;
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                if (!hit[u]) continue;
                word ^= (uint64_t)(uint32_t)(j[u] ^ i) << (16 * (n & 3));
                if ((n & 3) == 3) {
                    if (n < N.cap) N.cand[(n >> 2) * N.AP + i] = word;
                    word = own;
                }
                ++n;
            }
            if (n > N.cap) return n;  // the env gives these up
        }
    }
    if ((n & 3) != 0 && n < N.cap) N.cand[(n >> 2) * N.AP + i] = word;
    return n;
}

// The agents one agent touched in a substep, in list order: 16-bit ids, four to a word, the
// rest NEAR_NONE.  `slow`: the list was truncated, or more agents touched it than fit.
struct NearRec {
    uint64_t w0 = ~0ull, w1 = ~0ull;
    int n = 0;
    bool slow = false;
    __device__ __forceinline__ void push(int j)
    {
        const uint64_t keep = (uint64_t)((uint32_t)j ^ NEAR_NONE) << (16 * (n & 3));
        if (n < 4) w0 ^= keep;
        else if (n < NEAR_TOUCH) w1 ^= keep;
        else slow = true;
        ++n;
    }
    // the first word as stored: its last id says whether a second word is there (an id) or
    // the record does not hold the substep (NEAR_SLOW)
    __device__ __forceinline__ uint64_t first() const
    {
        return slow ? (w0 & 0x0000ffffffffffffull) | (uint64_t)NEAR_SLOW << 48 : w0;
    }
    __device__ __forceinline__ bool second() const { return !slow && n >= 4; }
};

// Contact force of agent j on the lane's agent, added and (`keep`: there is a tape) recorded.
template <typename T>
__device__ __forceinline__ void near_pair(const Cst<T> &C, const WideLds<T> &W, const WLane<T> &L,
                                          const St<T> &st, int j, T &fx, T &fy, NearRec &rec,
                                          bool keep)
{
    T gx, gy;
    if (pair_force(C, st.px - W.px[j], st.py - W.py[j], st.vx - W.vx[j], st.vy - W.vy[j],
                   L.pr.radius + W.rad[j] + C.margin, L.ddv, gx, gy)) {
        fx += gx;  // apart, a pair adds exactly +0
        fy += gy;
        if (keep) rec.push(j);
    }
}

// Whether candidate j is listed for the lane's agent, and its key in list order (GRID: outside
// the 3x3 block of grid cells it is within the radius by rounding only, and not visited).
template <typename T, bool GRID>
__device__ __forceinline__ bool near_key(const Cst<T> &C, const WideLds<T> &W, const NearLds<T> &N,
                                         int i, uint32_t me, int j, T dx, T dy, int &key)
{
    key = j;
    bool in = dx * dx + dy * dy <= C.t_nbr && j != i;
    if (GRID) {
        const uint32_t cj = N.cell[j];
        const int sx = (int)(cj & 0xffffu) - (int)(me & 0xffffu) + 1;
        const int sy = (int)(cj >> 16) - (int)(me >> 16) + 1;
        in = in && (unsigned)sx <= 2u && (unsigned)sy <= 2u;
        key += (3 * sy + sx) * WIDE_MAX_AGENTS;
    }
    return in;
}

// Contact forces of an agent from its `n` candidates: its capped list in list order.  A pass
// over them counts the members and keeps the NK smallest keys above `last` of those that may
// touch: where the cap does not bite and no more may touch, those are the list's whole force.
// Otherwise pass after pass takes the next NK of the close ones or, where the cap bites, of all
// members.  (Taken one at a time, a pass for each, crowded agents bound the substep: 461 envs x
// 130 agents, 60 per unit area, 16 substeps forward 515 us, now 290, the full traversal 270; 857 x
// 70, 30 per unit area, 335, 188 and 175.)
template <typename T, bool GRID>
__device__ __forceinline__ void near_forces(const Cst<T> &C, const WideLds<T> &W,
                                            const NearLds<T> &N, const WLane<T> &L,
                                            const St<T> &st, int n, T &fx, T &fy, NearRec &rec,
                                            bool keep)
{
    constexpr int NK = 4;
    const uint32_t me = GRID ? N.cell[L.i] : 0u;
    int listed = 0, near = 0, ks[NK];
    auto pass = [&](bool all, int last) {
        listed = near = 0;
#pragma unroll
        for (int c = 0; c < NK; ++c) ks[c] = CUT_ALL;
        for (int e = 0; e < n; e += 4) {
            const uint64_t w = N.cand[(e >> 2) * N.AP + L.i];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int j = (int)((uint32_t)(w >> (16 * u)) & 0xffffu);
                const T dx = st.px - W.px[j], dy = st.py - W.py[j];
                int key;
                const bool in = near_key<T, GRID>(C, W, N, L.i, me, j, dx, dy, key);
                const bool close = in && !pair_apart(dx, dy, L.pr.radius + W.rad[j] + C.margin);
                listed += in ? 1 : 0;
                near += close ? 1 : 0;
                int x = (all ? in : close) && key > last ? key : CUT_ALL;
#pragma unroll
                for (int c = 0; c < NK; ++c) {
                    const int lo = x < ks[c] ? x : ks[c];
                    x = x < ks[c] ? ks[c] : x;
                    ks[c] = lo;
                }
            }
        }
    };
    pass(false, -1);
    const bool cut = listed > C.K;
    rec.slow = cut;
    if (!cut && near <= NK) {
        for (int c = 0; c < near; ++c) {
            near_pair(C, W, L, st, GRID ? ks[0] % WIDE_MAX_AGENTS : ks[0], fx, fy, rec, keep);
#pragma unroll
            for (int k = 0; k + 1 < NK; ++k) ks[k] = ks[k + 1];
        }
        return;
    }
    int left = cut ? C.K : near;
    if (cut) pass(true, -1);
    for (;;) {
        const int last = ks[NK - 1];
#pragma unroll 1
        for (int c = 0; c < NK && c < left; ++c) {
            near_pair(C, W, L, st, GRID ? ks[0] % WIDE_MAX_AGENTS : ks[0], fx, fy, rec, keep);
#pragma unroll
            for (int k = 0; k + 1 < NK; ++k) ks[k] = ks[k + 1];
        }
        left -= NK;
        if (left <= 0) break;
        pass(cut, last);
    }
}

// The same from the full traversal.  KEEP is compiled in: in this pair loop the record costs a
// rollout without a tape where it is only branched around (461 envs x 130 agents, 60 per unit
// area, neighbours within 0.3, 64 substeps: 1470 us recorded, 1388 branched around, 1345).
template <typename T, bool GRID, bool KEEP>
__device__ __forceinline__ void full_forces(const Cst<T> &C, const WideLds<T> &W,
                                            const GridFrame<T> &G, const WLane<T> &L,
                                            const St<T> &st, T &fx, T &fy, NearRec &rec)
{
    int listed = 0;
    visit_list<T, GRID>(W, C.A, G, L.i, st.px, st.py, C.t_nbr, C.K, false, [&](int j, int32_t) {
        near_pair(C, W, L, st, j, fx, fy, rec, KEEP);
        ++listed;
    });
    if (KEEP && listed >= C.K) rec.slow = true;  // maybe truncated
}

template <typename T, bool DRONE, bool GRID, int APT, unsigned F>
__global__ __launch_bounds__(1024) void k_swarm_fwd(const Cst<T> Cin, const Args<T> g)
{
    const Cst<T> C = fold_cst<F>(Cin);
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int32_t wsum[16];
    const int AP = (int)blockDim.x * APT;
    const WideLds<T> W = wide_lds<T>(smem, AP);
    const NearLds<T> N = near_lds<T, GRID>(smem, AP);
    const GridFrame<T> G = grid_frame(C, (const T *)nullptr);
    WLane<T> L[APT];
    wide_lanes<T, false, APT, F>(C, g, W, WBoxLds<T>{}, L);
    St<T> st[APT];
#pragma unroll
    for (int k = 0; k < APT; ++k) load_state<T, DRONE>(g.s0.f, L[k].idx, 0, st[k]);
    const size_t EA = (size_t)C.E * C.A;
    // the search's frame: the world's bounds, or the box of the rollout's input
    Box4<T> box = {C.bmin_x, C.bmin_y, C.bmax_x, C.bmax_y};
    if (C.collisions && !(box.mnx < box.mxx)) {
        box = box_none<T>();
#pragma unroll
        for (int k = 0; k < APT; ++k) box_join(box, Box4<T>{st[k].px, st[k].py, st[k].px, st[k].py});
        box_wave(box);
        T *const red = W.px;  // (one box per wave, before the first positions)
        if ((threadIdx.x & 63) == 0) {
            T *o = red + 4 * (threadIdx.x >> 6);
            o[0] = box.mnx;
            o[1] = box.mny;
            o[2] = box.mxx;
            o[3] = box.mxy;
        }
        __syncthreads();
        for (int w = 0; w < (int)blockDim.x / 64; ++w)
            box_join(box, Box4<T>{red[4 * w], red[4 * w + 1], red[4 * w + 2], red[4 * w + 3]});
    }
    const bool taped = g.fsum != nullptr;
    // The skin bears two steps' motion, or what a shorter rollout's own substeps need (none for
    // a single one: 200 envs x 300 agents, 15 per unit area, neighbours within 0.3, one substep
    // 68 us with the whole skin, 34 without, 48 by the full traversal).
    const int moves = g.nsteps * C.S - 1;
    const T part = moves < 2 * C.S ? T(moves) / T(2 * C.S) : T(1);
    NearGrid<T> H = near_grid(C, box, part, AP);
    bool whole = moves > 0 && (GRID || C.A > NEAR_FULL);  // a quarter is left to take
    bool dense = N.cap == 0;   // the full traversal   (both the same in every thread)
    T rx[APT], ry[APT];        // where the candidates were found
    int nc[APT];               // how many there are
#pragma unroll
    for (int k = 0; k < APT; ++k) {
        rx[k] = ry[k] = __builtin_nan("");  // none yet: moved
        nc[k] = 0;
    }
    for (int t = 0; t < g.nsteps; ++t) {
        T a[APT][4];
#pragma unroll
        for (int k = 0; k < APT; ++k) load_act(g.act, (size_t)t * EA + L[k].idx, C.ad, a[k]);
        for (int s = 0; s < C.S; ++s) {
            T Fx[APT], Fy[APT];
#pragma unroll
            for (int k = 0; k < APT; ++k) Fx[k] = Fy[k] = T(0);
            if (C.needs_forces) {
                if (C.collisions) {
                    if (!dense) {
                        bool far = false;
#pragma unroll
                        for (int k = 0; k < APT; ++k) {
                            const T dx = st[k].px - rx[k], dy = st[k].py - ry[k];
                            far = far || (L[k].active && !(dx * dx + dy * dy <= H.half2));
                        }
                        vote_put(N.moved, far);
                    }
                    __syncthreads();  // the previous substep's readers are done
                    bool find = !dense && vote_get(N.moved);
#pragma unroll
                    for (int k = 0; k < APT; ++k) {
                        wide_put(W, L[k], st[k], (const WBoxLds<T> *)nullptr);
                        if (GRID && !dense)
                            N.cell[L[k].i] =
                                (uint32_t)grid_axis(st[k].px, G.ox, G.cs, G.bins) |
                                (uint32_t)grid_axis(st[k].py, G.oy, G.cs, G.bins) << 16;
                    }
                    if (find)
                        for (int c = threadIdx.x; c < H.nx * H.ny; c += blockDim.x) N.start[c] = 0;
                    __syncthreads();
                    while (find) {
                        int at[APT], slot[APT];
#pragma unroll
                        for (int k = 0; k < APT; ++k) {
                            at[k] = near_axis(st[k].py, H.oy, H.iy, H.ny) * H.nx +
                                    near_axis(st[k].px, H.ox, H.ix, H.nx);
                            slot[k] = L[k].active ? atomicAdd(&N.start[at[k]], 1) : 0;
                        }
                        __syncthreads();
                        block_exclusive_scan(N.start, H.nx * H.ny, N.scan);
#pragma unroll
                        for (int k = 0; k < APT; ++k)
                            if (L[k].active) N.sorted[N.start[at[k]] + slot[k]] = (uint16_t)L[k].i;
                        __syncthreads();
                        bool over = false;
#pragma unroll
                        for (int k = 0; k < APT; ++k) {
                            rx[k] = st[k].px;
                            ry[k] = st[k].py;
                            if (!L[k].active) continue;
                            nc[k] = near_find(W, N, H, L[k].i, st[k].px, st[k].py);
                            over = over || nc[k] > N.cap;
                        }
                        vote_put(N.over, over);
                        __syncthreads();
                        find = vote_get(N.over);
                        if (!find) break;
                        __syncthreads();  // before the sort, or all its LDS, is used again
                        if (whole) {
                            whole = false;
                            H = near_grid(C, box, T(0.25) * part, AP);
                            for (int c = threadIdx.x; c < H.nx * H.ny; c += blockDim.x) N.start[c] = 0;
                            __syncthreads();
                        } else {
                            dense = true;
                            find = false;
                        }
                    }
                    if (GRID && dense) grid_build(W, C.A, G, wsum);
                }
#pragma unroll
                for (int k = 0; k < APT; ++k) {
                    T fx = T(0), fy = T(0);
                    NearRec rec;
                    if (C.collisions && L[k].active) {
                        if (!dense)
                            near_forces<T, GRID>(C, W, N, L[k], st[k], nc[k], fx, fy, rec, taped);
                        else if (taped)
                            full_forces<T, GRID, true>(C, W, G, L[k], st[k], fx, fy, rec);
                        else
                            full_forces<T, GRID, false>(C, W, G, L[k], st[k], fx, fy, rec);
                    }
                    T sx, sy;
                    wide_static_forces(C, g, L[k], st[k], sx, sy);
                    Fx[k] = fx + sx;
                    Fy[k] = fy + sy;
                    if (taped && L[k].active) {
                        const size_t q = ((size_t)t * C.S + s) * EA + L[k].idx;
                        g.fsum[2 * q] = Fx[k];
                        g.fsum[2 * q + 1] = Fy[k];
                        if (C.collisions) {
                            g.touch[q] = rec.first();
                            if (rec.second()) g.touch2[q] = rec.w1;
                        }
                    }
                }
            }
#pragma unroll
            for (int k = 0; k < APT; ++k) {
                St<T> nx;
                integrate<T, DRONE>(C, L[k].pr, st[k], a[k], Fx[k], Fy[k], nx);
                st[k] = nx;
            }
        }
#pragma unroll
        for (int k = 0; k < APT; ++k) {
            if (!L[k].active) continue;
            if (t + 1 < g.nsteps)
                store_state<T, DRONE>(g.traj.f, (size_t)t * EA + L[k].idx, st[k]);
            else
                store_state<T, DRONE>(g.fin.f, L[k].idx, st[k]);
        }
    }
}

// Reverse of one touching pair, both sides (own and reverse).
template <typename T>
__device__ __forceinline__ void near_pair_adj(const Cst<T> &C, const WideLds<T> &W,
                                              const WLane<T> &L, const St<T> &in, T wFx, T wFy,
                                              int j, St<T> &gi)
{
    pair_adj_combined(C, in.px - W.px[j], in.py - W.py[j], in.vx - W.vx[j], in.vy - W.vy[j],
                      L.pr.radius + W.rad[j] + C.margin, wFx - W.wfx[j], wFy - W.wfy[j], gi.px,
                      gi.py, gi.vx, gi.vy);
}

template <typename T, bool DRONE, bool GRID, int APT, unsigned F>
__global__ __launch_bounds__(1024) void k_swarm_bwd(const Cst<T> Cin, const Args<T> g)
{
    const Cst<T> C = fold_cst<F>(Cin);
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int32_t wsum[16];
    const int AP = (int)blockDim.x * APT;
    const WideLds<T> W = wide_lds<T>(smem, AP);
    const WBoxLds<T> B = {};
    const GridFrame<T> G = grid_frame(C, (const T *)nullptr);
    WLane<T> L[APT];
    wide_lanes<T, false, APT, F>(C, g, W, B, L);
    const size_t EA = (size_t)C.E * C.A;
    const bool taped = g.fsum != nullptr;
    St<T> gs[APT];
#pragma unroll
    for (int k = 0; k < APT; ++k) st_zero(gs[k]);
    for (int t = g.nsteps - 1; t >= 0; --t) {
        St<T> st0[APT];
        T a[APT][4], ga[APT][4];
#pragma unroll
        for (int k = 0; k < APT; ++k) {
            if (L[k].active) {
                if (t == g.nsteps - 1)
                    add_adj<T, DRONE>(g.afin.f, L[k].idx, gs[k]);
                else
                    add_adj<T, DRONE>(g.atraj.f, (size_t)t * EA + L[k].idx, gs[k]);
            }
            if (t == 0)
                load_state<T, DRONE>(g.s0.f, L[k].idx, 0, st0[k]);
            else
                load_state<T, DRONE>(g.traj.f, L[k].idx, (size_t)(t - 1) * EA, st0[k]);
            load_act(g.act, (size_t)t * EA + L[k].idx, C.ad, a[k]);
            for (int q = 0; q < 4; ++q) ga[k][q] = T(0);
        }
        const size_t row = (size_t)t * C.S * EA;
        for (int s = C.S - 1; s >= 0; --s) {
            // the substep's input, integrated from the step's checkpoint
            St<T> in[APT];
            T Fx[APT], Fy[APT];
            uint64_t touch[APT];
            int32_t cut[APT];
#pragma unroll
            for (int k = 0; k < APT; ++k) {
                in[k] = st0[k];
                Fx[k] = Fy[k] = T(0);
                touch[k] = ~0ull;
                cut[k] = CUT_ALL;
            }
            if (taped) {
#pragma unroll
                for (int k = 0; k < APT; ++k) {
                    const size_t at = row + L[k].idx;
                    if (C.collisions && L[k].active) touch[k] = g.touch[at + (size_t)s * EA];
                    for (int q = 0; q <= s; ++q) {
                        const T *f = g.fsum + 2 * (at + (size_t)q * EA);
                        Fx[k] = f[0];
                        Fy[k] = f[1];
                        if (q == s) break;
                        St<T> nx;
                        integrate<T, DRONE>(C, L[k].pr, in[k], a[k], Fx[k], Fy[k], nx);
                        in[k] = nx;
                    }
                }
            } else {
                for (int q = 0; q < s; ++q)
                    wide_substep<T, DRONE, GRID, false, APT>(C, g, W, B, G, L, a, in, wsum);
                if (C.needs_forces) {
                    if (C.collisions) wide_publish_all<T, GRID, APT>(C, W, G, L, in, wsum);
#pragma unroll
                    for (int k = 0; k < APT; ++k)
                        wide_forces<T, GRID>(C, g, W, G, L[k], in[k], Fx[k], Fy[k], cut[k]);
                }
            }
            St<T> gi[APT];
            T gFx[APT], gFy[APT];
#pragma unroll
            for (int k = 0; k < APT; ++k)
                integrate_adj<T, DRONE>(C, L[k].pr, in[k], a[k], Fx[k], Fy[k], gs[k], gi[k], ga[k],
                                        gFx[k], gFy[k]);
            if (C.needs_forces) {
                bool full = !taped;  // the same in every thread
                if (C.collisions) {
                    if (taped) {
                        bool slow = false;
#pragma unroll
                        for (int k = 0; k < APT; ++k) slow = slow || (uint32_t)(touch[k] >> 48) == NEAR_SLOW;
                        __syncthreads();  // the previous substep's readers are done
#pragma unroll
                        for (int k = 0; k < APT; ++k)
                            wide_put(W, L[k], in[k], (const WBoxLds<T> *)nullptr);
                        vote_put(wsum, slow);
                    }
#pragma unroll
                    for (int k = 0; k < APT; ++k) {
                        // the force adjoint divided by the damping denominator
                        W.wfx[L[k].i] = gFx[k] * L[k].inv_dd;
                        W.wfy[L[k].i] = gFy[k] * L[k].inv_dd;
                        if (!taped) W.cut[L[k].i] = cut[k];
                    }
                    __syncthreads();
                    if (taped && vote_get(wsum)) {
                        full = true;
                        // the lists' ends, from the traversal the forward's forces came from
                        if (GRID) {
                            __syncthreads();  // the votes are read before the sort's scan
                            grid_build(W, C.A, G, wsum);
                        }
#pragma unroll
                        for (int k = 0; k < APT; ++k) {
                            T fx, fy;
                            wide_forces<T, GRID>(C, g, W, G, L[k], in[k], fx, fy, cut[k]);
                            W.cut[L[k].i] = cut[k];
                        }
                        __syncthreads();
                    }
                }
#pragma unroll
                for (int k = 0; k < APT; ++k) {
                    if (!L[k].active) continue;
                    if (full) {
                        wide_agent_adj<T, GRID, false>(C, g, W, B, G, L[k], in[k], gFx[k], gFy[k],
                                                       cut[k], gi[k]);
                        continue;
                    }
                    if (C.collisions) {
                        const T wFx = gFx[k] * L[k].inv_dd, wFy = gFy[k] * L[k].inv_dd;
                        uint64_t w = touch[k];
                        uint32_t j = (uint32_t)w & 0xffffu;
                        for (int c = 1; j != NEAR_NONE; ++c) {
                            near_pair_adj(C, W, L[k], in[k], wFx, wFy, (int)j, gi[k]);
                            w >>= 16;
                            if (c == 4) w = g.touch2[row + (size_t)s * EA + L[k].idx];
                            j = c < NEAR_TOUCH ? (uint32_t)w & 0xffffu : NEAR_NONE;
                        }
                    }
                    wide_static_adj(C, g, L[k], in[k], gFx[k], gFy[k], gi[k]);
                }
            }
#pragma unroll
            for (int k = 0; k < APT; ++k) gs[k] = gi[k];
        }
#pragma unroll
        for (int k = 0; k < APT; ++k) {
            if (!L[k].active) continue;
            T *pa = g.aact + ((size_t)t * EA + L[k].idx) * C.ad;
            for (int q = 0; q < C.ad; ++q) pa[q] = q < 4 ? ga[k][q] : T(0);
        }
    }
#pragma unroll
    for (int k = 0; k < APT; ++k)
        if (L[k].active) store_adj<T, DRONE>(g.a0.f, L[k].idx, gs[k]);
}

// ---------------------------------------------------------------------- launchers

// boxes: a box world (box agents or wheel contacts; never with drones).  feat: the FT_* paths
// the world uses; float32 fleets whose features a profile covers run its instances (holonomic
// fleets between walls; 2-D fleets with obstacles and walls), every other the general one.
#define SWARP_SWARM_LAUNCH(KERNEL, DRONE, P)                                                       \
    {                                                                                              \
        if (grid) hipLaunchKernelGGL((KERNEL<T, DRONE, true, APT, P>), g, b, shm, st, C, a);       \
        else hipLaunchKernelGGL((KERNEL<T, DRONE, false, APT, P>), g, b, shm, st, C, a);           \
        return;                                                                                    \
    }
#define SWARP_SWARM_DISPATCH(KERNEL, BOX_KERNEL, SHM)                                              \
    if (boxes) {                                                                                   \
        const size_t shm = wide_shm<T>(C, true);                                                   \
        if (grid) hipLaunchKernelGGL((BOX_KERNEL<T, true, APT, FT_ALL>), g, b, shm, st, C, a);     \
        else hipLaunchKernelGGL((BOX_KERNEL<T, false, APT, FT_ALL>), g, b, shm, st, C, a);         \
        return;                                                                                    \
    }                                                                                              \
    const size_t shm = SHM;                                                                        \
    if (drone) SWARP_SWARM_LAUNCH(KERNEL, true, FT_ALL)                                            \
    if constexpr (sizeof(T) == 4) {                                                                \
        if ((feat & ~FT_PROF_BODY) == 0u) SWARP_SWARM_LAUNCH(KERNEL, false, FT_PROF_BODY)          \
        if ((feat & ~FT_PROF_2D) == 0u) SWARP_SWARM_LAUNCH(KERNEL, false, FT_PROF_2D)              \
    }                                                                                              \
    SWARP_SWARM_LAUNCH(KERNEL, false, FT_ALL)

// The launchers of one agents-per-thread count (each count its own compilation unit).
template <typename T, int APT>
void launch_wide_fwd_apt(bool drone, bool boxes, const Cst<T> &C, const Args<T> &a, unsigned feat,
                         hipStream_t st)
{
    const dim3 g(C.E), b(wide_geom(C.A).threads);
    const bool grid = C.grid_bins > 0;
    const int NC = grid ? C.grid_bins * C.grid_bins : 0;
    SWARP_SWARM_DISPATCH(k_swarm_fwd, k_wide_fwd, swarm_fwd_lds<T>(wide_geom(C.A).slots, NC))
}

template <typename T, int APT>
void launch_wide_bwd_apt(bool drone, bool boxes, const Cst<T> &C, const Args<T> &a, unsigned feat,
                         hipStream_t st)
{
    const dim3 g(C.E), b(wide_geom(C.A).threads);
    const bool grid = C.grid_bins > 0;
    SWARP_SWARM_DISPATCH(k_swarm_bwd, k_wide_bwd, wide_shm<T>(C, false))
}
#undef SWARP_SWARM_DISPATCH
#undef SWARP_SWARM_LAUNCH

template <typename T>
inline void launch_wide_fwd(bool drone, bool boxes, const Cst<T> &C, const Args<T> &a,
                            unsigned feat, hipStream_t st)
{
    switch (wide_geom(C.A).apt) {
    case 1: launch_wide_fwd_apt<T, 1>(drone, boxes, C, a, feat, st); break;
    case 2: launch_wide_fwd_apt<T, 2>(drone, boxes, C, a, feat, st); break;
    default: launch_wide_fwd_apt<T, 4>(drone, boxes, C, a, feat, st); break;
    }
}

template <typename T>
inline void launch_wide_bwd(bool drone, bool boxes, const Cst<T> &C, const Args<T> &a,
                            unsigned feat, hipStream_t st)
{
    switch (wide_geom(C.A).apt) {
    case 1: launch_wide_bwd_apt<T, 1>(drone, boxes, C, a, feat, st); break;
    case 2: launch_wide_bwd_apt<T, 2>(drone, boxes, C, a, feat, st); break;
    default: launch_wide_bwd_apt<T, 4>(drone, boxes, C, a, feat, st); break;
    }
}

}  // namespace swarp
