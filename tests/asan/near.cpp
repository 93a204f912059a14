// The candidate words of the wide disc kernels (swarm.hpp) on the host: near_find packs four
// 16-bit ids to a word, near_forces takes them out again -- one agent, every number of
// candidates up to and past the list's room, whole and truncated lists.  Built plain, and under
// the type sanitizer, which reports a word touched as values of another type (accesses that
// the compiler may reorder).
#include <stdio.h>

#include "swarm.hpp"

using namespace swarp;

namespace {

template <typename T> int check(int A, int near, int K)
{
    const int AP = (A + 63) / 64 * 64;
    std::vector<unsigned char> lds(swarm_fwd_lds<T>(AP, 0));
    const WideLds<T> W = wide_lds<T>(lds.data(), AP);
    const NearLds<T> N = near_lds<T, false>(lds.data(), AP);
    // agents 1 .. near lie within reach of agent 0, in descending order in the sort
    for (int j = 0; j < A; ++j) {
        W.px[j] = j <= near ? T(0.01) * T(j) : T(5);
        W.py[j] = W.vx[j] = W.vy[j] = T(0);
        W.rad[j] = T(0.5);
        N.sorted[j] = (uint16_t)(A - 1 - j);
    }
    N.start[0] = 0;
    N.start[1] = A;
    Cst<T> C;
    memset(&C, 0, sizeof C);
    C.t_nbr = T(1);
    C.eps2 = T(1e-10);
    C.k = T(100);
    C.K = K;
    NearGrid<T> H = {T(0), T(0), T(0.1), T(0.1), 1, 1, T(1), T(0)};
    WLane<T> L;
    memset((void *)&L, 0, sizeof L);
    L.active = true;
    L.pr.radius = T(0.5);
    L.ddv = divisor(T(1), true);
    St<T> st;
    st_zero(st);
    const int found = near_find(W, N, H, 0, st.px, st.py);
    int bad = near > N.cap ? found <= N.cap : found != near;  // (it stops once they overflow)
    for (int e = 0; e < near && e < N.cap; ++e)
        bad += (int)(N.cand[(e >> 2) * AP] >> (16 * (e & 3)) & 0xffffu) != near - e;
    if (near > N.cap) return bad;
    T fx = T(0), fy = T(0);
    NearRec rec;
    near_forces<T, false>(C, W, N, L, st, near, fx, fy, rec, true);
    const int listed = near < K ? near : K;  // every listed agent touches
    bad += rec.n != listed || rec.slow != (near > K || listed > NEAR_TOUCH);
    for (int e = 0; e < listed && e < NEAR_TOUCH; ++e)
        bad += (int)((e < 4 ? rec.w0 : rec.w1) >> (16 * (e & 3)) & 0xffffu) != e + 1;
    return bad;
}

}  // namespace

int main()
{
    int bad = 0;
    for (int near = 0; near <= NEAR_MAX + 3; ++near)
        for (int K = 1; K <= 20; K += 3) bad += check<float>(70, near, K) + check<double>(70, near, K);
    printf("%d wrong\n", bad);
    return bad != 0;
}
