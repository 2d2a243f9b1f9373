// gemm_mid.hip — MFMA GEMM for grids too small for gemm2_kernel's 256-row
// tiles: prompts of some tens to some hundreds of rows.
#include <algorithm>

#include "gemm_core.hpp"

namespace lssm {

namespace {

// ---------------------------------------------------------------------------
// A block owns a BM x BN tile of Y.  Waves 0..3 compute, 2 x 2, each (BM /
// 2) x (BN / 2) in v_mfma_f32_32x32x16; they also DMA X into a ring of XS
// stages (64 k each), XS - 1 steps ahead.  The other waves handle W: dense by
// DMA into a ring of as many stages (four waves), quantized through four
// register sets (loads four steps ahead), dequantized to r(q s)
// (linear.metal:538) into a ring of four (eight waves).  One barrier per step; before it a wave
// waits for what the step after the next one reads (stages kt + 1 and kt + 2 are
// complete when step kt ends) and for its own reads of the slots that are
// refilled behind it.  The next step's first fragments are read before the
// barrier, but the compiler waits for all reads in flight at a step's first
// MFMAs, those of its last sub-step just behind the barrier among them: an LDS
// latency a step, which bounds the large K (777 x 4096 x 8192 dense, 70 us:
// MFMA 44 % busy, LDS 22 %, no bank conflicts).
// A step of these small tiles takes a fraction of a memory latency, which
// gemm2_kernel's two steps of prefetch do not cover: hence the deep rings.
// ---------------------------------------------------------------------------
template <int FMT, int BM, int BN> struct MidShape {
    static constexpr bool DENSE = FMT == LSSM_W_DENSE;
    static constexpr int ROW = G2K * 2;                                   // LDS row bytes
    static constexpr int FIT = 163840 / ((BM + BN) * ROW);
    static constexpr int XS = DENSE ? (FIT < 6 ? FIT : 6) : 6;
    static constexpr int SB = DENSE ? XS : 4;
    static constexpr int PROD = DENSE ? 4 : 8;                            // producer waves
    static constexpr int LDS = (XS * BM + SB * BN) * ROW;
    static_assert(LDS <= 163840 && XS >= 4, "LDS");
};

template <int N> __device__ __forceinline__ void wait_vm() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
template <int VM, int LGKM> __device__ __forceinline__ void wait_vm_lds() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(%1)" ::"n"(VM), "n"(LGKM) : "memory");
}

template <int FMT, typename T, int BM, int BN>
__global__ __launch_bounds__(64 * (4 + MidShape<FMT, BM, BN>::PROD)) void gemm_mid_kernel(GemmArgs a) {
    using S = MidShape<FMT, BM, BN>;
    constexpr bool DENSE = S::DENSE;
    constexpr int XS = S::XS, SB = S::SB;
    constexpr int WM = BM / 2, WN = BN / 2, MI = WM / 32, NI = WN / 32;
    __shared__ __attribute__((aligned(16))) T As[XS][BM * G2K];
    __shared__ __attribute__((aligned(16))) T Bs[SB][BN * G2K];
    using Op = MfmaOp<T>;
    using frag = typename Op::frag;

    const int t = threadIdx.x;
    const int lane = t % WAVE;
    const int w = __builtin_amdgcn_readfirstlane(t / WAVE);
    uint32_t tm, tn;
    xcd_tile_grouped(8, tm, tn);
    const uint32_t m0 = tm * BM, n0 = tn * BN;
    // split K (gridDim.z > 1): slice z takes steps z KT .. + KT and writes its
    // fp32 sums to a.ws
    const uint32_t K = a.K, KT = K / G2K / gridDim.z, kz = blockIdx.z * KT * G2K;
    auto barrier = [] {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };

    if (w >= 4) {
        // ---------------- W ----------------
        const int q = w - 4;
        const uint32_t p = t - 256;
        if constexpr (DENSE) {
            // producer wave q fills tile rows BN / 4 q .., 8 rows per
            // instruction (lane i: row run + i / 8, physical slot i % 8 =
            // logical slot (i % 8) ^ swz(row)); rows past N re-read row N - 1
            constexpr int PW = BN / 4, PJ = PW / 8;
            const char* wq[PJ];
#pragma unroll
            for (int j = 0; j < PJ; ++j) {
                const uint32_t row = PW * q + 8 * j + lane / 8;
                const uint32_t sl = (lane % 8) ^ swz(row);
                wq[j] = (const char*)a.w + ((size_t)min(n0 + row, a.N - 1) * K + kz + 8 * sl) * sizeof(T);
            }
            const uint32_t bs0 = lds_addr(&Bs[0][0]) + PW * q * S::ROW;
            auto dma_w = [&](uint32_t kt) {
                const uint32_t src = min(kt, KT - 1) * S::ROW, dst = bs0 + (kt % SB) * (BN * S::ROW);
#pragma unroll
                for (int j = 0; j < PJ; ++j) lds_dma16_asm(wq[j] + src, dst + 8 * j * S::ROW);
            };
            for (uint32_t s = 0; s < XS - 1; ++s) dma_w(s);
            wait_vm<PJ * (XS - 3)>();
            barrier();
            for (uint32_t kt = 0; kt < KT; ++kt) {
                dma_w(kt + XS - 1);
                wait_vm<PJ * (XS - 3)>();
                barrier();
            }
            wait_vm<0>();
            return;
        } else {
            // thread p: UPT pieces of 8 k of row p / TPR of the tile
            constexpr int UPT = BN * G2K / 8 / (64 * S::PROD), TPR = 8 / UPT;
            const uint32_t br = p / TPR, c0 = (p % TPR) * UPT;
            constexpr uint32_t GS = FMT == LSSM_W_Q4_G64 ? 64 : 32;
            const size_t nrow = min(n0 + br, a.N - 1);
            const char* wq = (const char*)a.w + nrow * (FMT == LSSM_W_Q8_G32 ? K : K / 2) + (FMT == LSSM_W_Q8_G32 ? kz : kz / 2);
            const uint16_t* sp = (const uint16_t*)a.s + nrow * (K / GS) + kz / GS;
            struct R {
                uint32_t q[FMT == LSSM_W_Q8_G32 ? 2 : 1], s;
            };
            auto load_w = [&](uint32_t kt, R (&r)[UPT]) {
#pragma unroll
                for (int h = 0; h < UPT; ++h) {
                    const uint32_t k = min(kt, KT - 1) * G2K + 8 * (c0 + h);
                    if constexpr (FMT == LSSM_W_Q8_G32) {
                        const u32x2 v = *reinterpret_cast<const u32x2*>(wq + k);
                        r[h].q[0] = v[0];
                        r[h].q[1] = v[1];
                    } else {
                        r[h].q[0] = *reinterpret_cast<const uint32_t*>(wq + k / 2);
                    }
                    r[h].s = sp[k / GS];
                }
            };
            const uint32_t sw = swz(br);
            auto store_w = [&](uint32_t slot, const R (&r)[UPT]) {
                T* Brow = Bs[slot] + br * G2K;
#pragma unroll
                for (int h = 0; h < UPT; ++h) {
                    const float s = fp16_bits_to_f((uint16_t)r[h].s), c = dequant_bias<FMT>(s);
                    *reinterpret_cast<u32x4*>(Brow + 8 * ((c0 + h) ^ sw)) =
                        dequant8<FMT, T>(r[h].q[0], FMT == LSSM_W_Q8_G32 ? r[h].q[1] : 0u, s, c);
                }
            };
            R r[4][UPT];
#pragma unroll
            for (int i = 0; i < 4; ++i) load_w(i, r[i]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                store_w(i, r[i]);
                load_w(i + 4, r[i]);
                __builtin_amdgcn_sched_barrier(0);
            }
            // stages 0 and 1 written (a wave's LDS writes complete in order)
            asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(UPT) : "memory");
            barrier();
            // step kt writes stage kt + 3 (its loads were issued four steps
            // ago), loads stage kt + 7 and ends when stage kt + 2 is written
            // (past the end the last stage again, into an idle slot)
            for (uint32_t kt = 0; kt < KT; kt += 4) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (kt + i >= KT) break;                   // wave-uniform
                    store_w((i + 3) % 4, r[(i + 3) % 4]);
                    __builtin_amdgcn_sched_barrier(0);
                    load_w(kt + i + 7, r[(i + 3) % 4]);
                    asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(UPT) : "memory");
                    barrier();
                }
            }
            return;
        }
    }

    // ---------------- compute waves ----------------
    const int wm = w / 2, wn = w % 2;
    constexpr int XR = BM / 4, XJ = XR / 8;                    // X rows each wave loads, DMA instructions per step
    uint32_t xo[XJ];
#pragma unroll
    for (int j = 0; j < XJ; ++j) {
        const uint32_t row = XR * w + 8 * j + lane / 8, xl = (lane % 8) ^ swz(row);
        xo[j] = (min(m0 + row, a.M - 1) * a.x_stride + 8 * xl) * (uint32_t)sizeof(T);
    }
    const uint32_t as0 = lds_addr(&As[0][0]) + XR * w * S::ROW;
    auto dma_x = [&](uint32_t kt, uint32_t slot, int j) {
        const char* base = (const char*)a.x + ((size_t)kz + (size_t)min(kt, KT - 1) * G2K) * sizeof(T);
        lds_dma16_asm(base + xo[j], as0 + slot * (BM * S::ROW) + 8 * j * S::ROW);
    };
    // row scales of the wave's rows, one a lane, taken by readlane in the epilogue
    float rs = 1.0f;
    if (a.row_scale && gridDim.z == 1) rs = a.row_scale[min(m0 + wm * WM + lane % WM, a.M - 1)];

    // one MFMA a sub-step would be a chain of its latencies: two sums then
    constexpr int NA = MI * NI == 1 ? 2 : 1;
    floatx16 accs[NA][MI][NI];
#pragma unroll
    for (int h = 0; h < NA; ++h)
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NI; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) accs[h][i][j][r] = 0.0f;
    // fragment rows are 32 i + lane % 32 of the wave's rows: swz(row) == swz(lane % 32)
    uint32_t fo[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) fo[ks] = (lane % 32) * G2K + 8 * ((2 * ks + lane / 32) ^ swz(lane % 32));
    // fragments of four sub-steps, read three ahead of their MFMAs (see above)
    frag af[4][MI], bf[4][NI];
    auto rd = [&](uint32_t xs, uint32_t bs, int ks, int b) {
        const T* Ab = As[xs] + (wm * WM) * G2K;
        const T* Bb = Bs[bs] + (wn * WN) * G2K;
#pragma unroll
        for (int i = 0; i < MI; ++i) af[b][i] = *reinterpret_cast<const frag*>(Ab + 32 * i * G2K + fo[ks]);
#pragma unroll
        for (int j = 0; j < NI; ++j) bf[b][j] = *reinterpret_cast<const frag*>(Bb + 32 * j * G2K + fo[ks]);
    };
    for (uint32_t s = 0; s < XS - 1; ++s)
        for (int j = 0; j < XJ; ++j) dma_x(s, s, j);
    wait_vm<XJ * (XS - 3)>();
    barrier();                                                 // stages 0 and 1 in LDS
    rd(0, 0, 0, 0);
    rd(0, 0, 1, 1);
    rd(0, 0, 2, 2);
    uint32_t xs = 0, bs = 0, xd = XS - 1;                      // stage slots: read, read, filled
    for (uint32_t kt = 0; kt < KT; ++kt) {
        const uint32_t xn = xs + 1 == XS ? 0 : xs + 1, bn = bs + 1 == SB ? 0 : bs + 1;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            if (ks == 0) rd(xs, bs, 3, 3);
            else rd(xn, bn, ks - 1, ks - 1);
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NI; ++j) accs[ks % NA][i][j] = Op::mma(af[ks][i], bf[ks][j], accs[ks % NA][i][j]);
            __builtin_amdgcn_sched_group_barrier(0x100, MI + NI, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, MI * NI, 0);
            // stage kt + XS - 1 of X, spread over the sub-steps
            if (ks < XJ) dma_x(kt + XS - 1, xd, ks);
        }
        xs = xn;
        bs = bn;
        xd = xd + 1 == XS ? 0 : xd + 1;
        // stage kt + 2 of X landed, and this wave's reads of stage kt done:
        // behind the barrier its slot is filled again.  (LDS reads complete in
        // order, and only those of the last three sub-steps, all of stage kt +
        // 1, may be outstanding; the first sub-step's DMA keeps them behind.)
        wait_vm_lds<XJ * (XS - 3), 3 * (MI + NI)>();
        barrier();
    }
    wait_vm<0>();
    floatx16(&acc)[MI][NI] = accs[0];
    if constexpr (NA == 2) acc[0][0] += accs[1][0][0];

    // element r of lane l: row (r / 4) 8 + (l / 32) 4 + r % 4, column l % 32
    if (gridDim.z > 1) {
        float* ws = a.ws + (size_t)blockIdx.z * a.M * a.N;
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NI; ++j) {
                const uint32_t n = n0 + wn * WN + j * 32 + lane % 32;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const uint32_t m = m0 + wm * WM + i * 32 + (r / 4) * 8 + (lane / 32) * 4 + r % 4;
                    if (m < a.M && n < a.N) ws[(size_t)m * a.N + n] = acc[i][j][r];
                }
            }
        return;
    }
    T* Y = (T*)a.y;
    const T* Rz = (const T*)a.res;
    const int epi = a.epi;
    auto value = [&](float v, int i, int r, uint32_t n) {
        if (a.row_scale) {
            const int r0 = i * 32 + (r / 4) * 8 + r % 4;
            const float s0 = readlane_f(rs, r0), s1 = readlane_f(rs, r0 + 4);
            v *= lane < 32 ? s0 : s1;
        }
        if (n < a.silu_cols) v = silu_fast(v);
        if (epi == LSSM_EPI_SILU) v = silu_f(v);
        return from_f<T>(v);
    };
    const bool vec = a.y_stride % 8 == 0 && (uintptr_t)a.y % 16 == 0 &&
                     (epi != LSSM_EPI_ADD || (uintptr_t)a.res % 16 == 0);
    if (!vec) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NI; ++j) {
                const uint32_t n = n0 + wn * WN + j * 32 + lane % 32;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const uint32_t m = m0 + wm * WM + i * 32 + (r / 4) * 8 + (lane / 32) * 4 + r % 4;
                    const T v = value(acc[i][j][r], i, r, n);
                    if (m < a.M && n < a.N) {
                        const size_t yi = (size_t)m * a.y_stride + n;
                        Y[yi] = epi == LSSM_EPI_ADD ? from_f<T>(to_f(Rz[yi]) + to_f(v)) : v;
                    }
                }
            }
        return;
    }
    // the rounded tile through LDS (over the X stages), out in 16-byte runs;
    // 16-byte slot s of row r sits at s ^ 4 ((r / 4) % 2): rows r and r + 4
    // (one store instruction) fall in different banks
    constexpr uint32_t RB = BN * 2, SPR = BN / 8;
    char* out = reinterpret_cast<char*>(&As[0][0]);
    static_assert(BM * RB <= XS * BM * S::ROW, "the tile fits the X stages");
    auto slot_of = [](uint32_t r, uint32_t sl) { return sl ^ (4u * ((r >> 2) & 1u)); };
    barrier();                                                 // every wave's DMAs and reads done
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) {
            const uint32_t c = wn * WN + j * 32 + lane % 32;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const uint32_t rr = wm * WM + i * 32 + (r / 4) * 8 + (lane / 32) * 4 + r % 4;
                *reinterpret_cast<T*>(out + rr * RB + 16 * slot_of(rr, c / 8) + 2 * (c % 8)) = value(acc[i][j][r], i, r, n0 + c);
            }
        }
    __builtin_amdgcn_s_waitcnt(0xC07F);
    barrier();
#pragma unroll 4
    for (uint32_t q = t; q < BM * SPR; q += 256) {
        const uint32_t R = q / SPR, sl = q % SPR;
        const u32x4 st = *reinterpret_cast<const u32x4*>(out + R * RB + 16 * slot_of(R, sl));
        const uint32_t m = m0 + R, n = n0 + 8 * sl;
        if (m >= a.M) continue;
        const size_t yi = (size_t)m * a.y_stride + n;
        if (n + 8 <= a.N) {
            u32x4 o = st;
            if (epi == LSSM_EPI_ADD) {
                const u32x4 rv = *reinterpret_cast<const u32x4*>(Rz + yi);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float lo = f_of_bits<T>((uint16_t)rv[e]) + f_of_bits<T>((uint16_t)st[e]);
                    const float hi = f_of_bits<T>((uint16_t)(rv[e] >> 16)) + f_of_bits<T>((uint16_t)(st[e] >> 16));
                    o[e] = (uint32_t)__builtin_bit_cast(uint16_t, from_f<T>(lo)) |
                           ((uint32_t)__builtin_bit_cast(uint16_t, from_f<T>(hi)) << 16);
                }
            }
            *reinterpret_cast<u32x4*>(Y + yi) = o;
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                if (n + e >= a.N) break;
                float v = f_of_bits<T>((uint16_t)(st[e / 2] >> (16 * (e % 2))));
                if (epi == LSSM_EPI_ADD) v = to_f(Rz[yi + e]) + v;
                Y[yi + e] = from_f<T>(v);
            }
        }
    }
}

template <int FMT, typename T>
hipError_t mid_go(hipStream_t s, const GemmArgs& a, int bm, int bn, uint32_t S) {
    const dim3 grid((a.N + bn - 1) / bn, (a.M + bm - 1) / bm, S);
    const int nt = 64 * (4 + MidShape<FMT, 64, 64>::PROD);
    if (bm == 128 && bn == 128) gemm_mid_kernel<FMT, T, 128, 128><<<grid, nt, 0, s>>>(a);
    else if (bm == 128) gemm_mid_kernel<FMT, T, 128, 64><<<grid, nt, 0, s>>>(a);
    else gemm_mid_kernel<FMT, T, 64, 64><<<grid, nt, 0, s>>>(a);
    return hipGetLastError();
}

template <typename T>
hipError_t mid_fmt(hipStream_t s, const GemmArgs& a, int bm, int bn, uint32_t S) {
    switch (a.wfmt) {
        case LSSM_W_Q4_B32: return mid_go<LSSM_W_Q4_B32, T>(s, a, bm, bn, S);
        case LSSM_W_Q4_G64: return mid_go<LSSM_W_Q4_G64, T>(s, a, bm, bn, S);
        case LSSM_W_Q8_G32: return mid_go<LSSM_W_Q8_G32, T>(s, a, bm, bn, S);
        default: return mid_go<LSSM_W_DENSE, T>(s, a, bm, bn, S);
    }
}

// The K slices' fp32 sums added in slice order, then the epilogue: r(v),
// r(silu(v)) or r(res + r(v)).
template <typename T>
__global__ __launch_bounds__(256) void gemm_split_sum_kernel(GemmArgs a, uint32_t S) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x, MN = (size_t)a.M * a.N;
    if (i >= MN) return;
    float v = 0.0f;
    for (uint32_t z = 0; z < S; ++z) v += a.ws[z * MN + i];
    const uint32_t m = (uint32_t)(i / a.N), n = (uint32_t)(i % a.N);
    const size_t yi = (size_t)m * a.y_stride + n;
    if (a.row_scale) v *= a.row_scale[m];
    if (n < a.silu_cols) v = silu_fast(v);
    if (a.epi == LSSM_EPI_SILU) v = silu_f(v);
    if (a.epi == LSSM_EPI_ADD) v = to_f(((const T*)a.res)[yi]) + rnd<T>(v);
    ((T*)a.y)[yi] = from_f<T>(v);
}

// The same, four consecutive outputs a thread (N a multiple of 4): 16-byte
// loads of the slices' sums.
template <typename T>
__global__ __launch_bounds__(256) void gemm_split_sum4_kernel(GemmArgs a, uint32_t S) {
    const size_t q = (size_t)blockIdx.x * 256 + threadIdx.x, MN = (size_t)a.M * a.N;
    if (4 * q >= MN) return;
    floatx4 v = {0.0f, 0.0f, 0.0f, 0.0f};
    for (uint32_t z = 0; z < S; ++z) {
        const floatx4 p = reinterpret_cast<const floatx4*>(a.ws + z * MN)[q];
        v[0] += p[0];
        v[1] += p[1];
        v[2] += p[2];
        v[3] += p[3];
    }
    const uint32_t m = (uint32_t)(4 * q / a.N), n = (uint32_t)(4 * q % a.N);
    const size_t yi = (size_t)m * a.y_stride + n;
    T o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float x = v[e];
        if (a.row_scale) x *= a.row_scale[m];
        if (n + e < a.silu_cols) x = silu_fast(x);
        if (a.epi == LSSM_EPI_SILU) x = silu_f(x);
        if (a.epi == LSSM_EPI_ADD) x = to_f(((const T*)a.res)[yi + e]) + rnd<T>(x);
        o[e] = from_f<T>(x);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) ((T*)a.y)[yi + e] = o[e];
}

template <typename T> hipError_t mid_run(hipStream_t s, const GemmArgs& a, const GemmMidPlan& p) {
    const hipError_t e = mid_fmt<T>(s, a, p.bm, p.bn, p.split);
    if (e != hipSuccess || p.split == 1) return e;
    const size_t MN = (size_t)a.M * a.N;
    if (a.N % 4 == 0 && (uintptr_t)a.ws % 16 == 0)
        gemm_split_sum4_kernel<T><<<(unsigned)((MN / 4 + 255) / 256), 256, 0, s>>>(a, p.split);
    else
        gemm_split_sum_kernel<T><<<(unsigned)((MN + 255) / 256), 256, 0, s>>>(a, p.split);
    return hipGetLastError();
}

}  // namespace

// The estimate, in hundredths of a microsecond: 2 us for the launch, then for
// each of a CU's blocks a start and an end and its K steps, fitted to the
// measured times (us, start + end and per step of 64; quantized / dense):
// 128 x 128 5 and 0.57, 128 x 64 3 and 0.45 / 0.35, 64 x 64 2.5 and 0.27 / 0.21.
// In a single round that leaves CUs idle a step takes 0.3 + 0.7 of the filled
// share of that (the L2 is shared), down to 0.54 / 0.40, 0.37 / 0.27.  Two
// quantized 64 x 64 blocks share a CU (LDS) and take 1.5 x one.  Splitting K
// costs a launch that adds the slices: 3 us and their bytes, written and read,
// at 5 TB/s.
// Measured against the kernels that ran before (us): 100 x 10576 x 2560 int4
// 47.6 -> 17.8, 300 -> 39.4 -> 30.9; 100 x 2560 x 5120 int4 108 -> 15.2; 777 x
// 4096 x 8192 dense 108 -> 71; 200 x 768 x 1536 int8 28.0 -> 10.3.
GemmMidPlan gemm_mid_plan(const GemmArgs& a) {
    GemmMidPlan best;
    if (a.y2 || a.K % G2K != 0 || (uint64_t)a.M * a.x_stride * 2 >= (1ull << 31)) return best;
    const bool dense = a.wfmt == LSSM_W_DENSE;
    const uint64_t cus = num_cus(), KT = a.K / G2K;
    const uint32_t gs = dense ? 1u : wfmt_group(a.wfmt);
    struct Tile {
        int bm, bn;
        uint32_t ends, q, q_min, d, d_min;
    };
    for (const Tile& t : {Tile{128, 128, 500, 57, 54, 57, 40}, Tile{128, 64, 300, 45, 37, 35, 27}, Tile{64, 64, 250, 27, 27, 21, 21}}) {
        if (((uint64_t)a.M + t.bm - 1) / t.bm > 65535) continue;      // (grid.y)
        const uint64_t tiles = (uint64_t)((a.M + t.bm - 1) / t.bm) * ((a.N + t.bn - 1) / t.bn);
        const bool pair = !dense && t.bm == 64;
        for (uint32_t S : {1u, 2u, 3u, 4u, 5u, 6u, 8u}) {
            if (S > 1 && (!a.ws || KT % S != 0 || KT / S < 4 || (a.K / S) % gs != 0 ||
                          tiles * S > (pair ? 2 : 1) * cus || (uint64_t)S * a.M * a.N > a.ws_floats))
                continue;
            const uint64_t n = (tiles * S + cus - 1) / cus;
            uint64_t step = 100 * (dense ? t.d : t.q);             // (in ten-thousandths)
            if (n == 1) step = std::max<uint64_t>(100 * (dense ? t.d_min : t.q_min), step * (3 * cus + 7 * tiles * S) / (10 * cus));
            uint64_t cost = n * (t.ends + KT / S * step / 100);
            if (pair && n > 1) cost = cost * 3 / 4;
            cost += 200;
            if (S > 1) cost += 300 + (uint64_t)S * a.M * a.N * 8 / 50000;
            if (cost < best.cost) best = GemmMidPlan{t.bm, t.bn, S, cost};
        }
    }
    return best;
}

hipError_t launch_gemm_mid(hipStream_t s, const GemmArgs& a, const GemmMidPlan& p) {
    if (p.bm == 0) return hipErrorInvalidValue;
    if (a.act == LSSM_F16) return mid_run<f16>(s, a, p);
    if (a.act == LSSM_BF16) return mid_run<bf16>(s, a, p);
    return hipErrorInvalidValue;
}

}  // namespace lssm
