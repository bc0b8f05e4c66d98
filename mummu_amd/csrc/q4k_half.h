// Q4_K weights as operands of the f16 matrix units: sc * q < 1024 of a sub-block is an exact half.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "device_utils.h"
#include "qact.h"

namespace mummu {

typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef _Float16 half4v __attribute__((ext_vector_type(4)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));  // staging registers: first-class vectors stay in VGPRs

// Codes at bits 0-3 and 16-19 (4-7 and 20-23 with HIGH) of t as halfs: the code itself, as a subnormal, is code * 2^-24
// (16 code * 2^-24), which one packed product turns into code * mul.
template <bool HIGH>
__device__ inline half2v code_pair(uint32_t t, half2v mul) {
    const uint32_t u = t & (HIGH ? 0x00F000F0u : 0x000F000Fu);
    half2v h;
    __builtin_memcpy(&h, &u, 4);
    return h * mul;
}
// Four Q6_K codes as bytes (0..63) -> halfs of code - 32, two at a time in the element order of HAct: a byte under 0x64 is the half 1024 + byte.
__device__ inline half2v q6k_code_pair(uint32_t codes, uint32_t pick) {
    const half2v bias = {(_Float16)1056.0f, (_Float16)1056.0f};
    const uint32_t u = __builtin_amdgcn_perm(0x64646464u, codes, pick);
    half2v h;
    __builtin_memcpy(&h, &u, 4);
    return h - bias;
}
// Eight Q4_K codes (the low or high nibbles of two words, in the element order of HAct) times their sub-block's scale, over
// 2^14 (exact: up to 63 * 15 in units of 2^-14): two masks, a shift and four products a word.
template <bool HIGH>
__device__ inline half8 q4k_operand(uint32_t w0, uint32_t w1, half2v mul) {
    const half2v f[4] = {code_pair<HIGH>(w0, mul), code_pair<HIGH>(w0 >> 8, mul), code_pair<HIGH>(w1, mul), code_pair<HIGH>(w1 >> 8, mul)};
    half8 o;
    __builtin_memcpy(&o, f, 16);
    return o;
}
constexpr float kQ4kUnit = 16384.0f;

// The first 16 bytes of a super-block: d | dmin, and (ggml get_scale_min_k4 for all eight sub-blocks at once) the scales and
// the offsets of sub-blocks 0-3 and 4-7 as bytes.
struct Q4kHeader {
    uint32_t dd, sc4[2], mn4[2];
    __device__ void unpack(u32x4 h) {
        dd = h[0];
        sc4[0] = h[1] & 0x3F3F3F3Fu;
        mn4[0] = h[2] & 0x3F3F3F3Fu;
        sc4[1] = (h[3] & 0x0F0F0F0Fu) | ((h[1] >> 2) & 0x30303030u);
        mn4[1] = ((h[3] >> 4) & 0x0F0F0F0Fu) | ((h[2] >> 2) & 0x30303030u);
    }
    // Bytes 0, 1 (or 2, 3) of t as halfs: a byte under 0x64 is the half 1024 + byte.
    __device__ static half2v pair(uint32_t t, bool upper) {
        const uint32_t u = __builtin_amdgcn_perm(0x64646464u, t, upper ? 0x04030402u : 0x04010400u);
        half2v h;
        __builtin_memcpy(&h, &u, 4);
        return h - half2v{(_Float16)1024.0f, (_Float16)1024.0f};
    }
    // mul of q4k_operand for step st: of sub-block 2 st (the low nibbles) sc * 2^10, of 2 st + 1 (the high ones) sc * 2^6.
    __device__ void muls(int st, half2v &low, half2v &high) const {
        const half2v m = pair(sc4[st >> 1], st & 1) * half2v{(_Float16)1024.0f, (_Float16)64.0f};
        low = half2v{m[0], m[0]};
        high = half2v{m[1], m[1]};
    }
    // The block offsets m as halfs (exact), in the order of the block sums: of four sub-blocks, of all.
    __device__ half4v offsets(int part) const {
        const half2v a = pair(mn4[part], false), b = pair(mn4[part], true);
        return half4v{a[0], a[1], b[0], b[1]};
    }
    __device__ half8 offsets() const {
        const half4v a = offsets(0), b = offsets(1);
        return half8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
    }
    __device__ float d(int lift = 0) const { return __fmul_rn(kQ4kUnit / (float)(1 << lift), half_bits_to_float((uint16_t)(dd & 0xFFFFu))); }
    __device__ float minus_dmin() const { return -half_bits_to_float((uint16_t)(dd >> 16)); }
};

struct Q4kArgs {
    const uint8_t *w0, *w1;        // gate and up, or down [experts][out_dim][in_dim]
    HAct a;                        // rows of in_dim: tokens (gate/up, through sorted / k_slots) or sorted positions
    const int32_t *sorted, *tiles, *n_tiles;
    int k_slots, in_dim, out_dim;
    HAct act_h;                    // gate/up: silu(g) * u, sorted positions, in the form the down product reads
    QAct64 act_q;
    float *y;                      // down
};

// x / (1 + e^-x) in f32: the hardware's 2^y and reciprocal (1 ulp each), with what rounding y = -x log2 e lost put back and the
// reciprocal refined once.  The exponent stops at +-87, where e^-x and its reciprocal are both normal numbers: above, the quotient
// is x as it is; below, it is x * 0 (a gate of -inf is NaN, as in det_silu).
__device__ inline float silu_of(float x) {
    const float c = __builtin_amdgcn_fmed3f(x, -87.0f, 87.0f);
    const float y = __fmul_rn(c, -1.44269504f);
    const float lost = __builtin_fmaf(c, -1.44269504f, -y);
    const float lost2 = __builtin_fmaf(c, -1.92596299e-8f, lost);   // log2 e - 1.44269504f
    float t = __builtin_amdgcn_exp2f(y);
    t = __builtin_fmaf(t, __fmul_rn(lost2, 0.693147181f), t);
    const float den = __fadd_rn(1.0f, t);
    float r = __builtin_amdgcn_rcpf(den);
    r = __builtin_fmaf(__builtin_fmaf(-den, r, 1.0f), r, r);
    return __fmul_rn(x, x < -87.0f ? 0.0f : r);
}

// The same value, computed again: what is derived from it does not keep a register through the loop.
__device__ inline int again(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

}  // namespace mummu
