// The host rules of the GEMM launches over the extremes of what they accept
// (run on the CPU: no launch, no device).  Prints the calls that ask for more
// than a launch can have and returns their number.
#include <cstdint>
#include <cstdio>

#include "../../lite_ssm_amd/csrc/internal.hpp"

using namespace lssm;

int main() {
    int bad = 0;
    for (int wfmt : {LSSM_W_DENSE, LSSM_W_Q4_B32, LSSM_W_Q4_G64, LSSM_W_Q8_G32})
        for (uint32_t K : {64u, 128u, 192u, 2560u, 8192u})
            for (uint32_t N : {1u, 63u, 64u, 65u, 128u, 768u, 2560u, 4096u, 18560u})
                for (uint64_t M = 1; M * K * 2 < (1ull << 31); M = M + M / 8 + 1) {
                    GemmArgs a{};
                    a.x = a.w = a.s = reinterpret_cast<const void*>(4096);
                    a.y = reinterpret_cast<void*>(4096);
                    a.act = LSSM_BF16;
                    a.wfmt = wfmt;
                    a.M = (uint32_t)M;
                    a.N = a.y_stride = N;
                    a.K = a.x_stride = K;
                    a.ws = reinterpret_cast<float*>(16);
                    a.ws_floats = GEMM_WS_FLOATS;
                    const GemmMidPlan p = gemm_mid_plan(a);
                    if (p.bm == 0) continue;
                    // the workspace is as large as any plan needs it
                    a.ws_floats = (size_t)1 << 40;
                    const GemmMidPlan big = gemm_mid_plan(a);
                    if (big.bm != p.bm || big.bn != p.bn || big.split != p.split) {
                        printf("format %d, %llu x %u x %u: %u slices of %d x %d, %u of %d x %d with more workspace\n", wfmt,
                               (unsigned long long)M, N, K, p.split, p.bm, p.bn, big.split, big.bm, big.bn);
                        ++bad;
                    }
                    const uint64_t rows = (M + p.bm - 1) / p.bm;
                    const bool split_ok = p.split == 1 || (uint64_t)p.split * M * N <= GEMM_WS_FLOATS;
                    if (rows > 65535 || !split_ok || K / 64 % p.split != 0) {
                        printf("format %d, %llu x %u x %u: %d x %d tiles, %llu of them in M, %u slices\n", wfmt,
                               (unsigned long long)M, N, K, p.bm, p.bn, (unsigned long long)rows, p.split);
                        ++bad;
                    }
                }
    return bad != 0;
}
