// conv_core.hpp — the causal conv of width 4 over rows held in registers: 8
// consecutive channels (16-byte loads and stores) and CT consecutive time steps
// a thread, shared by conv1d and the prefill's conv + Gram kernel.
#pragma once

#include "common.hpp"

namespace lssm {

// 8 fp16 / bf16 values in a 16-byte vector register.
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
template <typename T> __device__ __forceinline__ float el8(v4u v, int e) {
    const uint32_t d = v[e / 2];
    return f_of_bits<T>((uint16_t)((e & 1) ? (d >> 16) : (d & 0xFFFF)));
}
template <typename T> __device__ __forceinline__ uint32_t bits_t(float f) {
    return __builtin_bit_cast(uint16_t, from_f<T>(f));
}
template <typename T> __device__ __forceinline__ v4u pack8(const float (&f)[8]) {
    v4u r;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = bits_t<T>(f[2 * i]) | (bits_t<T>(f[2 * i + 1]) << 16);
    return r;
}

// The CT + 3 input rows t0 - 3 .. t0 + CT - 1 of a thread's channels (xb: row 0
// of the sequence), so every input row is read once per thread, not once per
// tap; rows outside the sequence are zero.  hist (the channels' conv state) holds
// the rows before the first: entry 4 + t for row t < 0 (read where t0 == 0).
// Vector registers, elements taken out by shifts: an element address would put
// the array in scratch memory.
template <typename T, int CT>
__device__ __forceinline__ void conv_window(const T* xb, uint32_t xs, uint32_t t0, uint32_t L, const T* hist,
                                            v4u (&win)[CT + 3]) {
#pragma unroll
    for (int i = 0; i < CT + 3; ++i) {
        const int t = (int)t0 + i - 3;
        win[i] = (t >= 0 && t < (int)L) ? *reinterpret_cast<const v4u*>(xb + (size_t)t * xs)
                                        : v4u{0, 0, 0, 0};
    }
    if (hist && t0 == 0) {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            uint32_t h[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint16_t lo = __builtin_bit_cast(uint16_t, hist[(size_t)(2 * q) * 4 + 1 + i]);
                const uint16_t hi = __builtin_bit_cast(uint16_t, hist[(size_t)(2 * q + 1) * 4 + 1 + i]);
                h[q] = (uint32_t)lo | ((uint32_t)hi << 16);
            }
            win[i] = v4u{h[0], h[1], h[2], h[3]};
        }
    }
}

// store(i, r(conv)) of row t0 + i, r(silu(r(conv))) with SILU: the sums of
// conv1d_kernel in its order.  w: the channels' taps [8][4], bias may be null.
template <typename T, int CT, bool SILU, typename F>
__device__ __forceinline__ void conv_rows(const v4u (&win)[CT + 3], const T* w, const T* bias, F store) {
    float wf[8][4], bf[8];
    const v4u* w4 = reinterpret_cast<const v4u*>(w);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const v4u v = w4[q];
#pragma unroll
        for (int e = 0; e < 8; ++e) wf[2 * q + e / 4][e % 4] = el8<T>(v, e);
    }
    const v4u bv = bias ? *reinterpret_cast<const v4u*>(bias) : v4u{0, 0, 0, 0};
#pragma unroll
    for (int c = 0; c < 8; ++c) bf[c] = el8<T>(bv, c);
#pragma unroll
    for (int i = 0; i < CT; ++i) {
        float f[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            float acc = bf[c];
#pragma unroll
            for (int tap = 0; tap < 4; ++tap) acc = fmaf(wf[c][tap], el8<T>(win[i + tap], c), acc);
            f[c] = rnd<T>(acc);
            if (SILU) f[c] = silu_fast(f[c]);
        }
        store(i, pack8<T>(f));
    }
}

// The channels' conv state [8][4] after the sequence: its last four rows (zeros
// before the first), written by the thread whose rows include the last one.
template <typename T, int CT>
__device__ __forceinline__ void conv_seed(const v4u (&win)[CT + 3], uint32_t t0, uint32_t L, T* state) {
#pragma unroll
    for (int i = 0; i < CT; ++i) {
        if (t0 + i + 1 != L) continue;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            uint32_t lo[4], hi[4];                   // channels 2 q and 2 q + 1
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                lo[k] = win[i + k][q] & 0xFFFFu;
                hi[k] = win[i + k][q] >> 16;
            }
            reinterpret_cast<v4u*>(state)[q] = v4u{lo[0] | lo[1] << 16, lo[2] | lo[3] << 16, hi[0] | hi[1] << 16, hi[2] | hi[3] << 16};
        }
    }
}

}  // namespace lssm
