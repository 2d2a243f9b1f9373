// gemv_mma_core.hpp — pieces shared by the MFMA decode GEMVs (gemv_mma.hip,
// gemv_rows.hip): how a quad of weight chunks splits into MFMA k-slices, the
// lane trades that keep a slice inside one scale group, and the unpacking.
#pragma once

#include "gemv_core.hpp"

namespace lssm {

namespace {

constexpr size_t MM_LDS_MAX = 150 * 1024;        // dynamic LDS (static: < 5 KiB)

template <int V> struct FmtTag {
    static constexpr int value = V;
};

template <int FMT, typename T> struct Mma {
    using F = Fmt<FMT, T>;
    static constexpr int WPC = F::WPC;
    static constexpr int NP = WPC / 2;                                  // pairs per chunk
    static constexpr int QK = 4 * WPC;                                  // k per quad
    static constexpr int G = F::G;                                      // 0: dense
    static constexpr int SPQ = FMT == LSSM_W_DENSE ? 1 : (FMT == LSSM_W_Q8_G32 ? 2 : 4);  // MFMAs per quad
    static constexpr int GPQ = G ? QK / G : 1;                          // scale groups per quad
    static constexpr int SPG = SPQ / GPQ;                               // MFMAs per group
    static constexpr bool BIAS = q4_bf16<FMT, T>();
};

// Chunk (within the quad) and pair offset of MFMA k-slice s of lane group q,
// after mma_swap: the x pairs that slice s meets in lane group q.
template <int FMT> __device__ __forceinline__ void mma_slice_pos(int s, int q, int& ch, int& po) {
    if constexpr (FMT == LSSM_W_Q4_G64) {
        ch = (q & 1) + 2 * (s >> 1);
        po = 4 * ((s & 1) + 2 * (q >> 1));
    } else if constexpr (FMT == LSSM_W_Q4_B32) {
        ch = s;
        po = 4 * q;
    } else if constexpr (FMT == LSSM_W_Q8_G32) {
        ch = (q & 1) + 2 * s;
        po = 4 * (q >> 1);
    } else {
        ch = q;
        po = 0;
    }
}

// Lane group q loaded chunk q of the quad (dwords C_q[0..3]).  After the
// 32-lane swap, lane group q holds C_{q&1}[2(q>>1)], C_{q&1}[2(q>>1)+1],
// C_{(q&1)+2}[2(q>>1)], C_{(q&1)+2}[2(q>>1)+1]: dwords 0-1 come from chunks
// 0-1 and dwords 2-3 from chunks 2-3 (one 64-wide group each).  After the
// 16-lane swap as well it holds C_0[q], C_1[q], C_2[q], C_3[q] (dword j from
// chunk j: one 32-wide group each).
template <int FMT> __device__ __forceinline__ u32x4 mma_swap(u32x4 v) {
    if constexpr (FMT == LSSM_W_DENSE) {
        return v;
    } else {
        const auto a = __builtin_amdgcn_permlane32_swap(v[0], v[2], false, false);
        const auto b = __builtin_amdgcn_permlane32_swap(v[1], v[3], false, false);
        u32x4 r = u32x4{a[0], b[0], a[1], b[1]};
        if constexpr (FMT == LSSM_W_Q4_B32) {
            const auto c = __builtin_amdgcn_permlane16_swap(r[0], r[1], false, false);
            const auto d = __builtin_amdgcn_permlane16_swap(r[2], r[3], false, false);
            r = u32x4{c[0], c[1], d[0], d[1]};
        }
        return r;
    }
}

// Pair q of an octet (8 consecutive k, 8-aligned) in pair_pos order: the
// positions (within the octet) of its two values.  Octets never straddle the
// pair structure of a chunk, so these are constants.
template <int FMT, typename T> __device__ __forceinline__ void octet_pos(int q, int& a, int& b) {
    if constexpr (q4_bf16<FMT, T>()) {
        a = ((q & 2) ? 1 : 0) + ((q & 1) ? 4 : 0);
        b = a + 2;
    } else if constexpr (is_q4<FMT>()) {
        a = q;
        b = q + 4;
    } else if constexpr (FMT == LSSM_W_Q8_G32) {
        a = 4 * (q / 2) + q % 2;
        b = a + 2;
    } else {
        a = 2 * q;
        b = a + 1;
    }
}

// The 8 weights of MFMA k-slice s of a swapped quad as packed pairs: dword s
// (int4), dwords 2s, 2s+1 (int8), the whole quad chunk (dense).
template <int FMT, typename T> __device__ __forceinline__ u32x4 unpack_slice(u32x4 v, int s) {
    if constexpr (FMT == LSSM_W_DENSE) {
        return v;
    } else if constexpr (FMT == LSSM_W_Q8_G32) {
        const Unpacked<FMT, T> u = unpack<FMT, T>(make_uint4(v[2 * s], v[2 * s + 1], 0u, 0u));
        return u32x4{u.p[0], u.p[1], u.p[2], u.p[3]};
    } else {
        const Unpacked<FMT, T> u = unpack<FMT, T>(make_uint4(v[s], 0u, 0u, 0u));
        return u32x4{u.p[0], u.p[1], u.p[2], u.p[3]};
    }
}

template <typename T> __device__ __forceinline__ floatx4 mfma16(u32x4 a, u32x4 b, floatx4 c) {
    if constexpr (__is_same(T, bf16))
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0, 0, 0);
}

// RMSNorm of x for these kernels (norm.metal:52-79), the same wherever a row is
// normalised: the squares of an octet (summed over the lanes by wave_sum, over
// the runs of 64 octets in order), 1 / rms of a row of K with that sum, and
// r(x w scale) of an octet in the unpack's pair order.
template <typename T> __device__ __forceinline__ float octet_squares(u32x4 xv) {
    float q = dot2(xv[0], xv[0], 0.0f, T{});
    q = dot2(xv[1], xv[1], q, T{});
    q = dot2(xv[2], xv[2], q, T{});
    return dot2(xv[3], xv[3], q, T{});
}
__device__ __forceinline__ float row_inv_rms(float squares, uint32_t K, float eps) {
    return 1.0f / sqrtf(squares / (float)K + eps);
}
template <int FMT, typename T> __device__ __forceinline__ u32x4 octet_scaled(u32x4 xv, u32x4 nv, float scale) {
    float v[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        v[2 * e] = lo_f<T>(xv[e]) * lo_f<T>(nv[e]) * scale;
        v[2 * e + 1] = hi_f<T>(xv[e]) * hi_f<T>(nv[e]) * scale;
    }
    u32x4 pk;
#pragma unroll
    for (int qq = 0; qq < 4; ++qq) {
        int pa, pb;
        octet_pos<FMT, T>(qq, pa, pb);
        pk[qq] = pack2<T>(v[pa], v[pb]);
    }
    return pk;
}

// Every format, for the kernels that take them all.
template <typename T, class F> bool all_fmt(int wfmt, F&& f) {
    if constexpr (__is_same(T, float)) {
        return false;
    } else {
        switch (wfmt) {
            case LSSM_W_Q4_G64: return f(FmtTag<LSSM_W_Q4_G64>{});
            case LSSM_W_Q4_B32: return f(FmtTag<LSSM_W_Q4_B32>{});
            case LSSM_W_Q8_G32: return f(FmtTag<LSSM_W_Q8_G32>{});
            case LSSM_W_DENSE: return f(FmtTag<LSSM_W_DENSE>{});
            default: return false;
        }
    }
}

}  // namespace

}  // namespace lssm
