// The COO radius graph's kernels and entry points (coo.hip) on the host under the sanitizers:
// buffers of exactly the extents the ABI documents, odd sizes, counts outside [0, K], an index
// buffer on a 4-byte boundary, workgroups of one part and of several.  Edges equal a plain loop's.
#include <stdio.h>

#include <random>
#include <string>

#include "coo.hip"

namespace swarp {
std::string message;
int set_error(const char *m)
{
    message = m;
    return m[0] ? -1 : 0;
}
}  // namespace swarp

namespace {

std::mt19937 rng(7);

// A heap block of exactly n elements.
template <typename T> T *block(size_t n) { return (T *)malloc(n * sizeof(T) + (n == 0)); }

int check(int E, int A, int K, double fill, int shift, int64_t per)
{
    const int64_t n = (int64_t)E * A;
    int32_t *cnt = block<int32_t>(n), *buf = block<int32_t>(n * K + shift), *idx = buf + shift;
    std::vector<int64_t> want[2];
    std::uniform_real_distribution<double> u(0, 1);
    for (int64_t i = 0; i < n; ++i) {
        cnt[i] = u(rng) < fill ? (int32_t)(u(rng) * (K + 4)) - 1 : 0;  // -1 .. K + 2
        for (int k = 0; k < K; ++k) {
            idx[i * K + k] = (int32_t)(u(rng) * A);
            if (k >= cnt[i]) continue;
            want[0].push_back(i / A * A + idx[i * K + k]);
            want[1].push_back(i);
        }
    }
    const int64_t N = (int64_t)want[0].size();
    const int64_t tiles = per ? (n + per - 1) / per : swarp_edge_tiles(E, A);
    int64_t *sums = block<int64_t>(tiles), *host = block<int64_t>(tiles), *out = block<int64_t>(2 * N);
    int64_t got = -1;
    int bad = 0;
    if (per) {  // several parts a workgroup, which the entry points take above 2 M agents
        const int64_t agents = per / EDGE_TILE * EDGE_PART;
        hipLaunchKernelGGL(k_edge_sums, dim3((unsigned)tiles), dim3(EDGE_BLOCK), 0, nullptr, n, per, K,
                           cnt, sums, host);
        got = 0;
        for (int64_t t = 0; t < tiles; ++t) got += host[t];
        hipLaunchKernelGGL((k_edge_fill<false>), dim3((unsigned)((n + agents - 1) / agents)),
                           dim3(EDGE_BLOCK), 0, nullptr, n, per, A, K, idx, cnt, sums, N, out);
    } else {
        bad += swarp_edge_count(E, A, K, cnt, sums, host, &got, nullptr) != 0;
        bad += swarp_edge_fill(E, A, K, idx, cnt, sums, N, out, nullptr) != 0;
    }
    bad += got != N;
    for (int64_t e = 0; e < N; ++e) bad += out[e] != want[0][e] || out[N + e] != want[1][e];
    if (bad) printf("%d x %d, K = %d, per %lld: %d wrong\n", E, A, K, (long long)per, bad);
    free(cnt);
    free(buf);
    free(sums);
    free(host);
    free(out);
    return bad != 0;
}

// A wait that fails is reported once, by the call itself: the next launch's own check finds
// nothing left over.
int check_failed_wait()
{
    int32_t cnt[3] = {1, 0, 2};
    int64_t sums[1], host[1], n = 0;
    emu::sync_error = hipErrorLaunchFailure;
    const int rc = swarp_edge_count(1, 3, 2, cnt, sums, host, &n, nullptr);
    const bool told = rc != 0 && !swarp::message.empty();
    const bool clean = hipGetLastError() == hipSuccess;
    if (!told || !clean) printf("failed wait: reported %d, left over %d\n", told, !clean);
    return !told || !clean;
}

}  // namespace

int main()
{
    int bad = check_failed_wait();
    bad += check(1, 1, 1, 1.0, 0, 0);
    bad += check(1, 513, 5, 0.7, 0, 0);    // a workgroup and one agent, rows not 16-byte pieces
    bad += check(3, 171, 4, 0.7, 1, 0);    // 16-byte rows on a 4-byte boundary
    bad += check(683, 3, 8, 0.5, 0, 0);    // 2049 agents: a tile and one
    bad += check(4, 512, 16, 0.3, 0, 0);   // exactly one tile
    bad += check(1, 700, 3, 0.0, 0, 0);    // no edges
    bad += check(9, 1001, 4, 0.4, 0, 2 * EDGE_TILE);
    bad += check(1, 4097, 6, 0.6, 0, 2 * EDGE_TILE);  // a tile of two parts a workgroup and one agent
    bad += check(5, 1300, 2, 1.0, 0, 3 * EDGE_TILE);
    printf("%d case(s) failed\n", bad);
    return bad ? 1 : 0;
}
