// gemm_f32.hip — fp32 activations: Y[M, N] = epi(X[M, K] . deq(W)[N, K]^T) on
// v_mfma_f32_32x32x2_f32, for dense fp32 and block-quantized weights.  With
// fp32 activations r() is the identity and q s is exact in fp32, so the GEMM
// and the GEMV rule (linear.metal:253-343, 440-474, 492-574) are one and the
// same, and the products and sums stay fp32 throughout.
//
// Bound by the fp32 matrix rate (256 FLOP per CU and cycle, an eighth of the
// 16-bit one's LDS need), so the tiles only have to keep the four SIMDs busy:
// each wave owns one 32 x 32 accumulator tile, KW of them share an output tile
// and split every K step (their sums meet in LDS), so that a grid of few tiles
// can be cut finer:
//   64 x 64 (four waves, KW 1), 32 x 64 (four, KW 2), 32 x 32 (eight, KW 8)
// A K step is 32 KW wide.  Two register sets, loads two steps ahead as written:
// as compiled the tiles of 32 rows request a step's loads near the end of the
// step before it is stored and wait for them among the next MFMAs (300 x 3352 x
// 768, 26 us: MFMA 49 % busy; the waves wait to issue two thirds of their cycles).  LDS
// is double-buffered, one barrier per step.  LDS rows are padded by 16
// bytes (pitch 4 mod 64 banks): the 16-byte fragment reads of 16 consecutive
// rows hit distinct banks.  A lane reads four consecutive k of its row for
// four MFMAs: the k order inside the product is the same for both operands.
#include "common.hpp"
#include "internal.hpp"

namespace lssm {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// Eight consecutive quantized weights of one row and their scale.
template <int FMT> struct FRaw { uint32_t q; uint32_t s; };
template <> struct FRaw<LSSM_W_Q8_G32> { u32x2 q; uint32_t s; };

template <int FMT, int EPI, int BM, int BN, int KW>
__global__ __launch_bounds__(64 * (BM / 32) * (BN / 32) * KW) void gemm_f32_kernel(GemmArgs a) {
    constexpr int F_NT = 64 * (BM / 32) * (BN / 32) * KW;   // one 32 x 32 tile per wave
    constexpr bool DENSE = FMT == LSSM_W_DENSE;
    constexpr int BK = 32 * KW, PITCH = BK + 4;
    constexpr int XV = BM * BK / 4 / F_NT;            // 16-byte pieces of X per thread and step
    constexpr int DV = BN * BK / 4 / F_NT;            // of dense W
    constexpr int QV = BN * BK / 8 / F_NT;            // 8-weight pieces of quantized W
    constexpr uint32_t GS = FMT == LSSM_W_Q4_G64 ? 64 : 32;
    constexpr int LDS_F = 2 * (BM + BN) * PITCH;
    static_assert(KW == 1 || LDS_F >= F_NT * 16, "the waves' sums reuse the tiles");
    __shared__ __attribute__((aligned(16))) float lds[LDS_F];
    float* Xs = lds;
    float* Ws = lds + 2 * BM * PITCH;

    // XCD x (linear block id % 8) takes a contiguous run of the tiles in
    // N-major order: all M tiles of a column tile read W through one L2
    const uint32_t mts = gridDim.y, total = gridDim.x * mts;
    const uint32_t lin = blockIdx.x + gridDim.x * blockIdx.y;
    const uint32_t xcd = lin % 8, tile = xcd * (total / 8) + min(xcd, total % 8) + lin / 8;
    const uint32_t m0 = (tile % mts) * BM, n0 = (tile / mts) * BN;

    const int t = threadIdx.x, lane = t % WAVE;
    const int w = __builtin_amdgcn_readfirstlane(t / WAVE);
    const int kw = w % KW, wt = w / KW;
    const int wm = wt % (BM / 32), wn = wt / (BM / 32);
    const uint32_t K = a.K, KT = (K + BK - 1) / BK;
    const float* X = (const float*)a.x;

    struct Regs {
        f32x4 x[XV];
        f32x4 d[DENSE ? DV : 1];
        FRaw<FMT> q[DENSE ? 1 : QV];
    };
    // Rows past M / N re-read the last row (never stored); k past K (K is a
    // multiple of 32, a step may be wider) reads k 0 and is zeroed at the
    // store to LDS.
    auto load = [&](uint32_t kt, Regs& r) {
        const uint32_t k0 = min(kt, KT - 1) * BK;
#pragma unroll
        for (int i = 0; i < XV; ++i) {
            const uint32_t id = t + F_NT * i, row = id / (BK / 4), k = k0 + 4 * (id % (BK / 4));
            r.x[i] = *reinterpret_cast<const f32x4*>(X + (size_t)min(m0 + row, a.M - 1) * a.x_stride + (k < K ? k : 0));
        }
        if constexpr (DENSE) {
#pragma unroll
            for (int i = 0; i < DV; ++i) {
                const uint32_t id = t + F_NT * i, row = id / (BK / 4), k = k0 + 4 * (id % (BK / 4));
                r.d[i] = *reinterpret_cast<const f32x4*>((const float*)a.w + (size_t)min(n0 + row, a.N - 1) * K + (k < K ? k : 0));
            }
        } else {
#pragma unroll
            for (int i = 0; i < QV; ++i) {
                const uint32_t id = t + F_NT * i, row = id / (BK / 8), kk = k0 + 8 * (id % (BK / 8));
                const uint32_t k = kk < K ? kk : 0;
                const size_t n = min(n0 + row, a.N - 1);
                if constexpr (FMT == LSSM_W_Q8_G32) r.q[i].q = *reinterpret_cast<const u32x2*>((const uint8_t*)a.w + n * K + k);
                else r.q[i].q = *reinterpret_cast<const uint32_t*>((const uint8_t*)a.w + n * (K / 2) + k / 2);
                r.q[i].s = ((const uint16_t*)a.s)[n * (K / GS) + k / GS];
            }
        }
    };
    auto store = [&](uint32_t kt, const Regs& r) {
        const uint32_t k0 = kt * BK, buf = kt & 1;
        const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < XV; ++i) {
            const uint32_t id = t + F_NT * i, row = id / (BK / 4), c = 4 * (id % (BK / 4));
            *reinterpret_cast<f32x4*>(Xs + (buf * BM + row) * PITCH + c) = KW == 1 || k0 + c < K ? r.x[i] : zero;
        }
        if constexpr (DENSE) {
#pragma unroll
            for (int i = 0; i < DV; ++i) {
                const uint32_t id = t + F_NT * i, row = id / (BK / 4), c = 4 * (id % (BK / 4));
                *reinterpret_cast<f32x4*>(Ws + (buf * BN + row) * PITCH + c) = KW == 1 || k0 + c < K ? r.d[i] : zero;
            }
        } else {
#pragma unroll
            for (int i = 0; i < QV; ++i) {
                const uint32_t id = t + F_NT * i, row = id / (BK / 8), c = 8 * (id % (BK / 8));
                const float s = KW == 1 || k0 + c < K ? fp16_bits_to_f((uint16_t)r.q[i].s) : 0.0f;
                f32x4 lo, hi;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if constexpr (FMT == LSSM_W_Q8_G32) {
                        lo[e] = (float)(((int)(r.q[i].q[0] << (24 - 8 * e))) >> 24) * s;
                        hi[e] = (float)(((int)(r.q[i].q[1] << (24 - 8 * e))) >> 24) * s;
                    } else {
                        lo[e] = (float)(((int)(r.q[i].q << (28 - 4 * e))) >> 28) * s;
                        hi[e] = (float)(((int)(r.q[i].q << (12 - 4 * e))) >> 28) * s;
                    }
                }
                float* dst = Ws + (buf * BN + row) * PITCH + c;
                *reinterpret_cast<f32x4*>(dst) = lo;
                *reinterpret_cast<f32x4*>(dst + 4) = hi;
            }
        }
    };
    // waits for this wave's LDS accesses only: loads in flight cross it
    auto barrier = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    floatx16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
    // lane l: row l % 32 of the wave's 32, k = 8 j + 4 (l / 32) .. + 3
    auto compute = [&](uint32_t kt) {
        const uint32_t buf = kt & 1;
        const float* xp = Xs + (buf * BM + 32 * wm + lane % 32) * PITCH + 32 * kw + 4 * (lane / 32);
        const float* wp = Ws + (buf * BN + 32 * wn + lane % 32) * PITCH + 32 * kw + 4 * (lane / 32);
        f32x4 xf[4], wf[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            xf[j] = *reinterpret_cast<const f32x4*>(xp + 8 * j);
            wf[j] = *reinterpret_cast<const f32x4*>(wp + 8 * j);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(xf[j][e], wf[j][e], acc, 0, 0, 0);
    };

    Regs r0, r1;
    load(0, r0);
    load(1, r1);
    store(0, r0);
    barrier();
    // step kt: request step kt + 2, multiply step kt, write step kt + 1 (past
    // the end the last step is re-read and the idle buffer written)
    auto step = [&](uint32_t kt, Regs& ld, const Regs& wr) {
        load(kt + 2, ld);
        compute(kt);
        store(kt + 1, wr);
        barrier();
    };
    uint32_t kt = 0;
    for (; kt + 1 < KT; kt += 2) {
        step(kt, r0, r1);
        step(kt + 1, r1, r0);
    }
    if (kt < KT) step(kt, r0, r1);

    // element r of lane l: row (r / 4) 8 + (l / 32) 4 + r % 4, column l % 32
    float* Y = (float*)a.y;
    const float* R = (const float*)a.res;
    auto out = [&](int r, float v) {
        const uint32_t m = m0 + 32 * wm + (r / 4) * 8 + (lane / 32) * 4 + r % 4;
        const uint32_t n = n0 + 32 * wn + lane % 32;
        if (m >= a.M || n >= a.N) return;
        const size_t yi = (size_t)m * a.y_stride + n;
        if (a.row_scale) v *= a.row_scale[m];
        if (n < a.silu_cols) v = silu_fast(v);
        if (EPI == LSSM_EPI_SILU) v = silu_f(v);
        if (EPI == LSSM_EPI_ADD) v = R[yi] + v;
        Y[yi] = v;
    };
    if constexpr (KW == 1) {
#pragma unroll
        for (int r = 0; r < 16; ++r) out(r, acc[r]);
    } else {
        // the KW sums of a tile in LDS; wave kw adds and stores 16 / KW of
        // the elements, in the order of the waves
        constexpr int RW = 16 / KW;
        float* mine = lds + (size_t)w * 16 * WAVE;
#pragma unroll
        for (int r = 0; r < 16; ++r) mine[r * WAVE + lane] = acc[r];
        barrier();
        const float* tsum = lds + (size_t)(wt * KW) * 16 * WAVE + lane;
#pragma unroll
        for (int i = 0; i < RW; ++i) {
            const int r = kw * RW + i;
            float v = 0.0f;
#pragma unroll
            for (int q = 0; q < KW; ++q) v += tsum[(q * 16 + r) * WAVE];
            out(r, v);
        }
    }
}

template <int FMT, int EPI>
hipError_t go_f32_tile(hipStream_t s, const GemmArgs& a) {
    auto tiles = [&](uint32_t bm, uint32_t bn) { return ((a.M + bm - 1) / bm) * (size_t)((a.N + bn - 1) / bn); };
    auto run = [&](auto kern, uint32_t bm, uint32_t bn, int nt) {
        kern<<<dim3((a.N + bn - 1) / bn, (a.M + bm - 1) / bm), nt, 0, s>>>(a);
        return hipGetLastError();
    };
    // One block per CU at most: the smallest tile, eight waves splitting K
    // (16 x 768 x 1536: 12.1 us against 22.4 and 32.8 in the larger tiles).
    // Else a CU's share of the tiles times what each costs there: at K 768, r
    // tiles per CU take 4.5 + 12.6 r us (64 x 64) or 5 + 7.4 r (32 x 64), so
    // 300 x 3352 (r 2 and 3) runs 30.2 and 26.2, 2000 x 3352 (r 7 and 14) 93.3
    // and 108.0; 32 x 32 tiles are behind there (27.7 and 137.5).  One thread
    // per output, the form before: 3486 us at 300 x 3352.
    const size_t cus = num_cus();
    auto cost = [&](uint32_t bm, uint32_t bn, uint32_t c) { return (tiles(bm, bn) + cus - 1) / cus * c; };
    if (tiles(32, 32) <= cus) return run(gemm_f32_kernel<FMT, EPI, 32, 32, 8>, 32, 32, 512);
    if (cost(64, 64, 126) <= cost(32, 64, 74)) return run(gemm_f32_kernel<FMT, EPI, 64, 64, 1>, 64, 64, 256);
    return run(gemm_f32_kernel<FMT, EPI, 32, 64, 2>, 32, 64, 256);
}

template <int FMT>
hipError_t go_f32(hipStream_t s, const GemmArgs& a) {
    switch (a.epi) {
        case LSSM_EPI_SILU: return go_f32_tile<FMT, LSSM_EPI_SILU>(s, a);
        case LSSM_EPI_ADD: return go_f32_tile<FMT, LSSM_EPI_ADD>(s, a);
        default: return go_f32_tile<FMT, LSSM_EPI_NONE>(s, a);
    }
}

}  // namespace

bool gemm_f32_takes(const GemmArgs& a) {
    // 16-byte loads of X (and dense W) rows, whole 32-k pieces, grid.y of M tiles
    return a.act == LSSM_F32 && a.K >= 32 && a.K % 32 == 0 && (a.wfmt != LSSM_W_Q4_G64 || a.K % 64 == 0) &&
           a.x_stride % 4 == 0 && (uintptr_t)a.x % 16 == 0 && (uintptr_t)a.w % 16 == 0 && !a.y2 &&
           (a.M + 31) / 32 <= 65535;
}

hipError_t launch_gemm_f32(hipStream_t s, const GemmArgs& a) {
    if (a.M == 0 || a.N == 0) return hipSuccess;
    if (!gemm_f32_takes(a)) return hipErrorInvalidValue;
    switch (a.wfmt) {
        case LSSM_W_Q4_B32: return go_f32<LSSM_W_Q4_B32>(s, a);
        case LSSM_W_Q4_G64: return go_f32<LSSM_W_Q4_G64>(s, a);
        case LSSM_W_Q8_G32: return go_f32<LSSM_W_Q8_G32>(s, a);
        default: return go_f32<LSSM_W_DENSE>(s, a);
    }
}

}  // namespace lssm
