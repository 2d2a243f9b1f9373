// gemv_rows.hip — decode batches of 2..64 rows on MFMA with the GEMV rule, for
// every 16-bit activation type and weight format.
#include <algorithm>
#include <cstdlib>

#include "gemv_mma_core.hpp"

namespace lssm {

namespace {

// ---------------------------------------------------------------------------
// gemv_rows: decode batches of up to 64 rows for every 16-bit activation type
// and weight format, x packed in fragment order (launch_mma_pack).
// gemv_mmx_kernel's product with the K split free: 8 waves take contiguous
// runs of qpw quads and walk them through a ring of two quads of weights, scales
// and x in flight, so any K of whole quads runs.  A block owns CT tiles of 16
// W rows and all RT tiles of 16 batch rows, so W is read from memory once
// whatever the batch; x is re-read by every block from L2 (RT KB per 32 k,
// against CT tiles of W), which CT keeps near the W traffic.
// Bound by latency: 18560 x 4096 int8 x bf16 at 24 rows streams its 81 MB in 26.6
// us (3.1 TB/s) in one round of blocks of four ring turns each; VALU issue takes
// 28 % of the cycles, the MFMA pipe 8 %.
// (A ring of four: slower at every shape, its registers cost more than the
// loads in flight bring.  A persistent grid of such blocks over many tiles:
// the waves meet after every group, and the loop-carried ring spilled.)
// int4 x bf16: -136 sum(x) of the group enters as the MFMA's C operand, once
// per row tile for all CT tiles, instead of a subtraction per output.
// ---------------------------------------------------------------------------
constexpr int GR_W = 8;                          // waves per block: the K split
constexpr int GR_D = 2;                          // quads in flight per wave

template <int FMT, typename T> constexpr int scale_dwords() {   // per tile and quad
    return Mma<FMT, T>::G > 0 ? Mma<FMT, T>::GPQ / 2 : 1;
}

// acc += the products of one quad: w as loaded, s its scales, x in fragment order.
template <int FMT, typename T, int CT, int RT>
__device__ __forceinline__ void rows_quad(const u32x4 (&w)[CT], const uint32_t (&s)[CT][scale_dwords<FMT, T>()],
                                          const u32x4 (&x)[RT][Mma<FMT, T>::SPQ], floatx4 (&acc)[RT][CT]) {
    using P = Mma<FMT, T>;
    constexpr int GPQ = P::GPQ, SPG = P::SPG;
    u32x4 wq[CT];
#pragma unroll
    for (int t = 0; t < CT; ++t) wq[t] = mma_swap<FMT>(w[t]);
    if constexpr (P::G == 0) {
#pragma unroll
        for (int t = 0; t < CT; ++t)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) acc[rt][t] = mfma16<T>(x[rt][0], wq[t], acc[rt][t]);
    } else {
#pragma unroll
        for (int g = 0; g < GPQ; ++g) {
            floatx4 c0[RT];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                c0[rt] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
                if constexpr (P::BIAS) {
                    constexpr uint32_t M136 = 0xC308C308u;             // bf16 (-136, -136)
#pragma unroll
                    for (int e = 0; e < SPG; ++e)
                        c0[rt] = mfma16<T>(x[rt][g * SPG + e], u32x4{M136, M136, M136, M136}, c0[rt]);
                }
            }
#pragma unroll
            for (int t = 0; t < CT; ++t) {
                u32x4 u[SPG];
#pragma unroll
                for (int e = 0; e < SPG; ++e) u[e] = unpack_slice<FMT, T>(wq[t], g * SPG + e);
                const uint32_t sw = s[t][g / 2];
                const float sc = fp16_bits_to_f((uint16_t)((g & 1) ? sw >> 16 : sw & 0xFFFFu));
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) {
                    floatx4 d = c0[rt];
#pragma unroll
                    for (int e = 0; e < SPG; ++e) d = mfma16<T>(x[rt][g * SPG + e], u[e], d);
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[rt][t][i] = __builtin_fmaf(sc, d[i], acc[rt][t][i]);
                }
            }
        }
    }
}

template <int FMT, typename T, int CT, int RT, class Epi>
__global__ __launch_bounds__(64 * GR_W) void gemv_rows_kernel(GemvCore c, Epi epi, uint32_t M, uint32_t qpw) {
    using P = Mma<FMT, T>;
    using F = Fmt<FMT, T>;
    constexpr int SPQ = P::SPQ;
    constexpr int D = GR_D;
    constexpr int SW = scale_dwords<FMT, T>();
    extern __shared__ __attribute__((aligned(16))) uint32_t mm_lds[];

    const uint32_t K = c.K, N = c.N;
    const int lane = threadIdx.x % WAVE, li = lane % 16, lq = lane / 16;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const uint32_t quads = K / P::QK, rts = (M + 15) / 16;
    const uint32_t q0 = w * qpw, q1 = min(q0 + qpw, quads);    // q0 >= quads: a wave without work
    const uint32_t tiles = (N + 15) / 16, tile0 = blockIdx.x * CT;
    epi.pin();

    struct Slot {
        u32x4 w[CT], x[RT][SPQ];
        uint32_t s[CT][SW];
    };
    Slot ring[D];
    const u32x4* xf = reinterpret_cast<const u32x4*>(c.xp) + lane;
    const uint8_t* wp[CT];
    const uint32_t* sp[CT];
#pragma unroll
    for (int t = 0; t < CT; ++t) {
        const size_t n = min(16 * (tile0 + t) + li, N - 1);
        wp[t] = c.w + n * F::row_bytes(K) + 16 * lq;
        sp[t] = P::G > 0 ? reinterpret_cast<const uint32_t*>(c.s + n * (K / (P::G > 0 ? P::G : 1))) : nullptr;
    }
    // past the wave's last quad the next wave's are read, past the row's end its
    // last again (their products are skipped)
    auto load = [&](uint32_t q, Slot& r) {
        const uint32_t qa = min(q, quads - 1);
#pragma unroll
        for (int t = 0; t < CT; ++t) {
            r.w[t] = *reinterpret_cast<const u32x4*>(wp[t] + (size_t)64 * qa);
            if constexpr (P::G > 0) {
#pragma unroll
                for (int i = 0; i < SW; ++i) r.s[t][i] = sp[t][qa * SW + i];
            }
        }
        // (row tiles past the batch's last read that one; never stored)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int sl = 0; sl < SPQ; ++sl)
                r.x[rt][sl] = xf[((size_t)(min((uint32_t)rt, rts - 1) * quads + qa) * SPQ + sl) * WAVE];
    };
    floatx4 acc[RT][CT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int t = 0; t < CT; ++t) acc[rt][t] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    auto compute = [&](const Slot& r) { rows_quad<FMT, T, CT, RT>(r.w, r.s, r.x, acc); };
    constexpr uint32_t NT = 64 * GR_W, NO = RT * CT * 256;     // threads, output elements of the block
    constexpr int EPT = (NO + NT - 1) / NT;
    typename Epi::Pre pre[EPT];
    auto out_mn = [&](uint32_t o, uint32_t& m, uint32_t& n) {
        const uint32_t rt = o / (CT * 256), t = (o / 256) % CT, l = (o % 256) / 4, e = o % 4;
        m = 16 * rt + 4 * (l / 16) + e;
        n = 16 * (tile0 + t) + l % 16;
    };
    if (q0 < q1) {
#pragma unroll
        for (int d = 0; d < D; ++d) load(q0 + d, ring[d]);
    }
    // the epilogue's inputs, behind the first quads
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < EPT; ++k) {
        uint32_t m, n;
        out_mn(min(threadIdx.x + NT * k, NO - 1), m, n);
        pre[k] = epi.prefetch((int)min(m, M - 1), min(n, N - 1));
    }
    __builtin_amdgcn_sched_barrier(0);
    // (wave-uniform) full turns of the ring, then what is in flight
    uint32_t q = q0;
    for (; q + D < q1; q += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            compute(ring[d]);
            __builtin_amdgcn_sched_barrier(0);
            load(q + D + d, ring[d]);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int d = 0; d < D; ++d)
        if (q + d < q1) compute(ring[d]);

    // ---- the waves' partial sums of each output element, in wave order ----
    floatx4* red = reinterpret_cast<floatx4*>(mm_lds);          // [wave][row tile][tile][lane]
    const float* redf = reinterpret_cast<const float*>(mm_lds);
    const uint32_t nw = (quads + qpw - 1) / qpw;                // waves with work
    if (q0 < q1) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int t = 0; t < CT; ++t) red[((w * RT + rt) * CT + t) * WAVE + lane] = acc[rt][t];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < EPT; ++k) {
        const uint32_t o = threadIdx.x + NT * k;
        if (o < NO) {
            float v = 0.0f;
            for (uint32_t ww = 0; ww < nw; ++ww) v += redf[ww * NO + o];
            uint32_t m, n;
            out_mn(o, m, n);
            if (m < M && n < N && o / 256 % CT + tile0 < tiles) epi((int)m, n, v, pre[k]);
        }
    }
}

// The same product without x packed beforehand, for calls that may hold no
// scratch memory (captured into a graph): a block takes one tile of 16 W rows
// and one of 16 batch rows, forms the rows' 1 / rms and normalises x as it
// loads it, in gemv_rows_kernel's K split and order of sums, so the outputs are
// those of the packed form bit for bit.  Every block normalises all of its x.
template <int FMT, typename T, class Epi>
__global__ __launch_bounds__(64 * GR_W) void gemv_rows_norm_kernel(GemvCore c, Epi epi, uint32_t M, uint32_t qpw) {
    using P = Mma<FMT, T>;
    using F = Fmt<FMT, T>;
    constexpr int SPQ = P::SPQ, D = GR_D, SW = scale_dwords<FMT, T>();
    __shared__ floatx4 red[GR_W][WAVE];
    __shared__ float inv_rms[16];

    const uint32_t K = c.K, N = c.N, KO = K / 8;
    const int lane = threadIdx.x % WAVE, li = lane % 16, lq = lane / 16;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const uint32_t m0 = 16 * blockIdx.y, n0 = 16 * blockIdx.x;
    const uint32_t quads = K / P::QK, q0 = w * qpw, q1 = min(q0 + qpw, quads);
    epi.pin();

    const T* x = static_cast<const T*>(c.x);
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const u32x4* row = reinterpret_cast<const u32x4*>(x + (size_t)min(m0 + 2 * w + r, M - 1) * c.x_stride);
        float t = 0.0f;
        for (uint32_t i = 0; i < KO; i += WAVE) {
            const uint32_t cc = i + lane;
            t += wave_sum(octet_squares<T>(cc < KO ? row[cc] : u32x4{0u, 0u, 0u, 0u}));
        }
        if (lane == 0) inv_rms[2 * w + r] = row_inv_rms(t, K, c.eps);
    }
    __syncthreads();
    const float scale = inv_rms[li];

    struct Slot {
        u32x4 w[1], x[SPQ], n[SPQ];
        uint32_t s[1][SW];
    };
    Slot ring[D];
    // (rows past the batch re-read its last, never stored; W rows likewise)
    const T* xrow = x + (size_t)min(m0 + li, M - 1) * c.x_stride;
    const T* nw = static_cast<const T*>(c.norm_w);
    const size_t n = min(n0 + li, N - 1);
    const uint8_t* wp = c.w + n * F::row_bytes(K) + 16 * lq;
    const uint32_t* sp = P::G > 0 ? reinterpret_cast<const uint32_t*>(c.s + n * (K / (P::G > 0 ? P::G : 1))) : nullptr;
    auto load = [&](uint32_t q, Slot& r) {
        const uint32_t qa = min(q, quads - 1);
        r.w[0] = *reinterpret_cast<const u32x4*>(wp + (size_t)64 * qa);
        if constexpr (P::G > 0) {
#pragma unroll
            for (int i = 0; i < SW; ++i) r.s[0][i] = sp[qa * SW + i];
        }
#pragma unroll
        for (int sl = 0; sl < SPQ; ++sl) {
            int ch, po;
            mma_slice_pos<FMT>(sl, lq, ch, po);
            const uint32_t k = qa * P::QK + ch * P::WPC + 2 * po;
            r.x[sl] = *reinterpret_cast<const u32x4*>(xrow + k);
            r.n[sl] = *reinterpret_cast<const u32x4*>(nw + k);
        }
    };
    floatx4 acc[1][1] = {{floatx4{0.0f, 0.0f, 0.0f, 0.0f}}};
    auto compute = [&](const Slot& r) {
        u32x4 xf[1][SPQ];
#pragma unroll
        for (int sl = 0; sl < SPQ; ++sl) xf[0][sl] = octet_scaled<FMT, T>(r.x[sl], r.n[sl], scale);
        rows_quad<FMT, T, 1, 1>(r.w, r.s, xf, acc);
    };
    if (q0 < q1) {
#pragma unroll
        for (int d = 0; d < D; ++d) load(q0 + d, ring[d]);
    }
    const uint32_t o = threadIdx.x, ol = (o % 256) / 4;         // output element of threads 0 .. 255
    const uint32_t om = m0 + 4 * (ol / 16) + o % 4, on = n0 + ol % 16;
    const typename Epi::Pre pre = epi.prefetch((int)min(om, M - 1), min(on, N - 1));
    for (uint32_t q = q0; q < q1; q += D) {                     // (wave-uniform)
#pragma unroll
        for (int d = 0; d < D; ++d) {
            if (q + d < q1) compute(ring[d]);
            load(q + D + d, ring[d]);
        }
    }
    if (q0 < q1) red[w][lane] = acc[0][0];
    __syncthreads();
    if (o >= 256 || om >= M || on >= N) return;
    const float* redf = reinterpret_cast<const float*>(&red[0][0]);
    const uint32_t nw_run = (quads + qpw - 1) / qpw;            // waves with work
    float v = 0.0f;
    for (uint32_t ww = 0; ww < nw_run; ++ww) v += redf[ww * 256 + o];
    epi((int)om, on, v, pre);
}

// gemv_rows launch plan.  Row tiles 1, 2 or 4.  Tiles of W per block by rounds
// of one block per CU times the tiles of a round and a quarter tile's time per
// row tile for the re-read x; at most 5, or 3 at 33 rows and more, 2 for int4
// there (registers).  Measured, CT 1 / 2 / 3 / 5 (us, pack launch included):
// int8 x bf16 18560 x 4096 at 32 rows 33.8 / 34.1 / 32.7 / 28.9; 10576 x 2560
// at 32 rows 18.5 / 19.6 / 15.7 / 21.6.
struct RowsPlan {
    uint32_t ct = 0, rt = 0, qpw = 0, blocks = 0;
    size_t lds = 0;
};
template <int FMT, typename T> constexpr uint32_t rows_most(int rt) {
    if (rt == 4) return Mma<FMT, T>::SPQ == 4 ? 2u : 3u;
    return rt == 2 && Mma<FMT, T>::SPQ == 4 && __is_same(T, f16) ? 3u : 5u;
}
template <int FMT, typename T> bool rows_plan(uint32_t M, uint32_t N, uint32_t K, RowsPlan& p) {
    using P = Mma<FMT, T>;
    if (M < 1 || M > 64 || N == 0 || K == 0 || K % P::QK != 0 || K > 8192) return false;
    const uint32_t quads = K / P::QK, tiles = (N + 15) / 16, cus = num_cus();
    p.rt = M <= 16 ? 1 : (M <= 32 ? 2 : 4);
    uint64_t best = ~0ull;
    for (uint32_t ct = 1; ct <= rows_most<FMT, T>((int)p.rt); ++ct) {
        const uint64_t groups = (tiles + ct - 1) / ct, cost = (groups + cus - 1) / cus * (4 * ct + p.rt);
        if (cost < best) {
            best = cost;
            p.ct = ct;
        }
    }
    p.blocks = (tiles + p.ct - 1) / p.ct;
    p.qpw = (quads + GR_W - 1) / GR_W;
    p.lds = (size_t)GR_W * p.rt * p.ct * WAVE * 16;
    return p.lds <= MM_LDS_MAX;
}

template <int FMT, typename T, int CT, int RT, class Epi>
hipError_t rows_run(hipStream_t s, const GemvCore& c, const Epi& e, uint32_t M, const RowsPlan& p) {
    auto k = gemv_rows_kernel<FMT, T, CT, RT, Epi>;
    static const hipError_t attr = hipFuncSetAttribute(
        reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, (int)MM_LDS_MAX);
    if (attr != hipSuccess) return attr;
    k<<<p.blocks, WAVE * GR_W, p.lds, s>>>(c, e, M, p.qpw);
    return hipGetLastError();
}

template <int FMT, typename T, int RT, class Epi>
hipError_t rows_ct(hipStream_t s, const GemvCore& c, const Epi& e, uint32_t M, const RowsPlan& p) {
    constexpr uint32_t MOST = rows_most<FMT, T>(RT);
    switch (p.ct) {
        case 1: return rows_run<FMT, T, 1, RT, Epi>(s, c, e, M, p);
        case 2: return rows_run<FMT, T, 2, RT, Epi>(s, c, e, M, p);
        case 3:
            if constexpr (MOST >= 3) return rows_run<FMT, T, 3, RT, Epi>(s, c, e, M, p);
            break;
        case 4:
            if constexpr (MOST >= 4) return rows_run<FMT, T, 4, RT, Epi>(s, c, e, M, p);
            break;
        case 5:
            if constexpr (MOST >= 5) return rows_run<FMT, T, 5, RT, Epi>(s, c, e, M, p);
            break;
    }
    return hipErrorInvalidValue;
}

template <int FMT, typename T, class Epi>
hipError_t rows_go(hipStream_t s, const GemvCore& c, const Epi& e, uint32_t M, const RowsPlan& p) {
    if (p.rt == 1) return rows_ct<FMT, T, 1, Epi>(s, c, e, M, p);
    if (p.rt == 2) return rows_ct<FMT, T, 2, Epi>(s, c, e, M, p);
    return rows_ct<FMT, T, 4, Epi>(s, c, e, M, p);
}

template <typename T, class Epi>
bool rows_call(hipStream_t s, const GemvArgs& a, const Epi& e, hipError_t& err) {
    GemvCore c{a.x, a.x_stride, (const uint8_t*)a.w, (const uint16_t*)a.s, a.norm_w, a.eps, a.N, a.K, 1.0f / (float)a.K};
    c.xp = static_cast<const uint32_t*>(a.xpack);
    return all_fmt<T>(a.wfmt, [&](auto tag) -> bool {
        constexpr int FMT = decltype(tag)::value;
        RowsPlan p;
        const bool ok = !a.xpart && !a.yfrag && (uintptr_t)a.w % 16 == 0 && (uintptr_t)a.xpack % 16 == 0 &&
                        (FMT == LSSM_W_DENSE || (uintptr_t)a.s % 4 == 0) && rows_plan<FMT, T>(a.M, a.N, a.K, p);
        if (ok && c.xp) {
            err = rows_go<FMT, T, Epi>(s, c, e, a.M, p);
        } else if (ok && a.norm_w && (uintptr_t)a.x % 16 == 0 && (uintptr_t)a.norm_w % 16 == 0 && a.x_stride % 8 == 0) {
            gemv_rows_norm_kernel<FMT, T, Epi><<<dim3((a.N + 15) / 16, (a.M + 15) / 16), WAVE * GR_W, 0, s>>>(c, e, a.M, p.qpw);
            err = hipGetLastError();
        } else {
            err = hipErrorInvalidValue;
        }
        return true;
    });
}

}  // namespace

bool gemv_rows_takes(uint32_t M, uint32_t N, uint32_t K, int wfmt, int act) {
    auto takes = [&](auto tag) {
        using T = decltype(tag);
        return all_fmt<T>(wfmt, [&](auto ft) -> bool {
            RowsPlan p;
            return rows_plan<decltype(ft)::value, T>(M, N, K, p);
        });
    };
    return act == LSSM_F16 ? takes(f16{}) : act == LSSM_BF16 ? takes(bf16{}) : false;
}

bool dense_head_gemm(uint32_t N, uint32_t K, int wfmt, int act) {
    return wfmt == LSSM_W_DENSE && act != LSSM_F32 && K % 64 == 0 && K >= 2048 && K <= 8192 && N >= 128 * num_cus();
}

bool gemv_rows_pays(uint32_t M, uint32_t N, uint32_t K, int wfmt, int act) {
    if (!gemv_rows_takes(M, N, K, wfmt, act)) return false;
    if (M > 4 && dense_head_gemm(N, K, wfmt, act)) return false;
    // up to four rows: only where neither the VALU GEMV nor the staging MFMA
    // kernel has the shape (dense out_proj of the 8B at 4 rows: 168 -> 15 us)
    if (M <= 4) return !gemv1_takes(K, wfmt, act) && !gemv_mma_takes(M, N, K, wfmt, act);
    // The staging kernel needs no pack launch (about 3.5 us) but every block
    // normalises and stages all of x: it stays ahead while a CU stages at most
    // 25600 values (16 rows of K 1536: 7.2 against 7.8 us; 5 rows of 5120: 8.5
    // against 9.2; 16 rows of 2560: 11.9 against 10.5).
    const uint64_t staged = gemv_mma_staged(M, N, K, wfmt, act);
    return staged == 0 || staged > 25600;
}

bool launch_gemv_rows(hipStream_t s, const GemvArgs& a, hipError_t& err) {
    auto go = [&](auto tag) -> bool {
        using T = decltype(tag);
        return rows_call<T>(s, a, EpiPlain<T>{(T*)a.y, a.y_stride, (const T*)a.res, a.epi}, err);
    };
    return a.act == LSSM_F16 ? go(f16{}) : a.act == LSSM_BF16 ? go(bf16{}) : false;
}

bool launch_inproj_rows(hipStream_t s, const InprojDecodeArgs& a, hipError_t& err) {
    auto go = [&](auto tag) -> bool {
        using T = decltype(tag);
        return rows_call<T>(s, a.g, EpiInproj<T>{a.d_inner, a.xbc, a.H, a.dconv, (T*)a.conv_state, (const T*)a.conv_w,
                                                 (const T*)a.conv_b, (T*)a.z, (T*)a.xbc_act, (T*)a.dt}, err);
    };
    return a.g.act == LSSM_F16 ? go(f16{}) : a.g.act == LSSM_BF16 ? go(bf16{}) : false;
}

}  // namespace lssm
