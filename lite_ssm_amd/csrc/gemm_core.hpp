// gemm_core.hpp — pieces shared by the prefill GEMMs (gemm.hip, gemm_mid.hip):
// the MFMA, the dequantization to the activation type, the DMA into swizzled
// LDS tiles and the XCD order of the tiles.
#pragma once

#include "common.hpp"
#include "internal.hpp"

namespace lssm {

namespace {

template <typename T> struct MfmaOp;
template <> struct MfmaOp<f16> {
    using frag = half8;
    static __device__ __forceinline__ floatx16 mma(frag a, frag b, floatx16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    }
};
template <> struct MfmaOp<bf16> {
    using frag = bf16x8;
    static __device__ __forceinline__ floatx16 mma(frag a, frag b, floatx16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
};

constexpr int G2K = 64;                          // k of an LDS tile row

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// 16 consecutive quantized weights of one row: raw bits + fp16 scale bits.
template <int FMT> struct WRaw { u32x2 q; uint32_t s; };
template <> struct WRaw<LSSM_W_Q8_G32> { u32x4 q; uint32_t s; };

template <typename T> __device__ __forceinline__ uint32_t pk2(float lo, float hi) {
    if constexpr (__is_same(T, bf16)) {
        typedef __bf16 v2 __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, v2{(__bf16)lo, (__bf16)hi});
    } else {
        typedef _Float16 v2 __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, v2{from_f<f16>(lo), from_f<f16>(hi)});
    }
}

// r(q s) for 8 consecutive weights -> 4 packed pairs (k order).  The
// unsigned value u (int4: q + 8, int8: q + 128) of two weights is placed by
// one v_perm into the mantissas of two fp16 values 1024 + u (bits
// 0x6400 | u), and fma(1024 + u, s, c) with c = -(1024 + 8) s (int8:
// -(1024 + 128) s) is q s exactly: both products have at most 11 + 11
// significant bits and q s at most 15, all exact in fp32; the fp16 operands
// convert inside v_fma_mix_f32.  One rounding, at the pack.  int4: q0 holds
// the 8 nibbles (k = nibble index); int8: q0, q1 the 8 bytes.
template <int FMT, typename T>
__device__ __forceinline__ u32x4 dequant8(uint32_t q0, uint32_t q1, float s, float c) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    // bytes (b0 of v, 0x64, b1 of v, 0x64) and (b2, 0x64, b3, 0x64)
    auto pair01 = [](uint32_t v) { return __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, v, 0x04010400u)); };
    auto pair23 = [](uint32_t v) { return __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, v, 0x04030402u)); };
    auto f = [&](_Float16 e) { return __builtin_fmaf((float)e, s, c); };
    if constexpr (FMT == LSSM_W_Q8_G32) {
        const uint32_t d0 = q0 ^ 0x80808080u, d1 = q1 ^ 0x80808080u;
        const h2 a = pair01(d0), b = pair23(d0), e = pair01(d1), g = pair23(d1);
        return u32x4{pk2<T>(f(a.x), f(a.y)), pk2<T>(f(b.x), f(b.y)), pk2<T>(f(e.x), f(e.y)), pk2<T>(f(g.x), f(g.y))};
    } else {
        // u of k 0, 2, 4, 6 (low nibbles) and k 1, 3, 5, 7
        const uint32_t lo = (q0 & 0x0F0F0F0Fu) ^ 0x08080808u;
        const uint32_t hi = ((q0 >> 4) & 0x0F0F0F0Fu) ^ 0x08080808u;
        const h2 e02 = pair01(lo), e46 = pair23(lo), e13 = pair01(hi), e57 = pair23(hi);
        return u32x4{pk2<T>(f(e02.x), f(e13.x)), pk2<T>(f(e02.y), f(e13.y)),
                     pk2<T>(f(e46.x), f(e57.x)), pk2<T>(f(e46.y), f(e57.y))};
    }
}
template <int FMT> __device__ __forceinline__ float dequant_bias(float s) {
    return (FMT == LSSM_W_Q8_G32 ? -1152.0f : -1032.0f) * s;
}

// 16 weights -> 8 packed pairs
template <int FMT, typename T>
__device__ __forceinline__ void dequant16(const WRaw<FMT>& r, uint32_t out[8]) {
    const float s = fp16_bits_to_f((uint16_t)r.s), c = dequant_bias<FMT>(s);
    u32x4 a, b;
    if constexpr (FMT == LSSM_W_Q8_G32) {
        a = dequant8<FMT, T>(r.q[0], r.q[1], s, c);
        b = dequant8<FMT, T>(r.q[2], r.q[3], s, c);
    } else {
        a = dequant8<FMT, T>(r.q[0], 0u, s, c);
        b = dequant8<FMT, T>(r.q[1], 0u, s, c);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        out[i] = a[i];
        out[4 + i] = b[i];
    }
}

__device__ __forceinline__ void lds_dma16(const void* g, void* l) {
    __builtin_amdgcn_global_load_lds(g, (__attribute__((address_space(3))) void*)l, 16, 0, 0);
}
// The same DMA as inline asm, for waves that also read LDS: the compiler does
// not see it, so it does not wait for it before every LDS read (it cannot
// tell which LDS bytes a DMA writes); the issuing wave waits with an explicit
// vmcnt.  m0 (the LDS base of the 1 KiB run) is saved and restored.
__device__ __forceinline__ void lds_dma16_asm(const void* g, uint32_t lds_byte) {
    uint32_t saved;
    asm volatile(
        "s_mov_b32 %0, m0\n\t"
        "s_mov_b32 m0, %2\n\t"
        "global_load_lds_dwordx4 %1, off\n\t"
        "s_mov_b32 m0, %0"
        : "=&s"(saved)
        : "v"(g), "s"(lds_byte)
        : "memory");
}
template <typename T> __device__ __forceinline__ uint32_t lds_addr(const T* p) {
    return (uint32_t)(size_t)((const __attribute__((address_space(3))) T*)p);
}

// LDS tile rows are 128 B (64 16-bit elements, 8 slots of 16 B) and the
// banks repeat every 256 B, so rows r and r + 2 share banks.  Physical slot =
// logical slot ^ ((r / 2) % 8): 16 consecutive rows read or written at one
// logical slot then cover all 16 16-byte positions of the 256 B window (row
// parity picks the half, the XOR the position), with no bank conflict.
__device__ __forceinline__ constexpr uint32_t swz(uint32_t row) { return (row >> 1) & 7u; }

// Workgroups go to the 8 XCDs round-robin in launch order (linear id % 8),
// and each XCD has its own L2.  Give XCD x a contiguous run of the tiles in
// M-major order, so the blocks that share an X row block (all N tiles of one
// M tile) run on one XCD and read X through one L2.  A bijection for any grid.
__device__ __forceinline__ void xcd_tile(uint32_t& mt, uint32_t& nt) {
    const uint32_t nbx = gridDim.x, total = nbx * gridDim.y;
    const uint32_t lin = blockIdx.x + nbx * blockIdx.y;
    const uint32_t x = lin % 8, q = total / 8, r = total % 8;
    const uint32_t tile = x * q + min(x, r) + lin / 8;
    mt = tile / nbx;
    nt = tile % nbx;
}

// The same runs in groups of `gm` M tiles, M fastest: the tiles an XCD works on
// at once then form a block of several M by several N tiles, and each X and W
// slice is read through its L2 for more of them.
__device__ __forceinline__ void xcd_tile_grouped(uint32_t gm, uint32_t& mt, uint32_t& nt) {
    const uint32_t nbx = gridDim.x, mts = gridDim.y, total = nbx * mts;
    const uint32_t lin = blockIdx.x + nbx * blockIdx.y;
    const uint32_t x = lin % 8, q = total / 8, r = total % 8;
    const uint32_t tile = x * q + min(x, r) + lin / 8;
    const uint32_t g = tile / (gm * nbx), left = mts - g * gm, h = min(gm, left);   // this group's M tiles
    const uint32_t i = tile - g * gm * nbx;
    mt = g * gm + i % h;
    nt = i / h;
}

}  // namespace

}  // namespace lssm
