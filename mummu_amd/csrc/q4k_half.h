// Q4_K weights as operands of the f16 matrix units: sc * q < 1024 of a sub-block is an exact half.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_utils.h"

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
// Eight Q4_K codes (the low or high nibbles of two words, in the element order of HAct) times their sub-block's scale, over
// 2^14 (exact: up to 63 * 15 in units of 2^-14): two masks, a shift and four products a word.
template <bool HIGH>
__device__ inline half8 q4k_operand(uint32_t w0, uint32_t w1, half2v mul) {
    const half2v f[4] = {code_pair<HIGH>(w0, mul), code_pair<HIGH>(w0 >> 8, mul), code_pair<HIGH>(w1, mul), code_pair<HIGH>(w1 >> 8, mul)};
    half8 o;
    __builtin_memcpy(&o, f, 16);
    return o;
}
// ... with mul for a sub-block scale sc: sc * 2^10 for the low nibbles, sc * 2^6 for the high ones.
template <bool HIGH>
__device__ inline half2v q4k_mul(uint32_t sc) {
    const _Float16 m = (_Float16)__fmul_rn((float)sc, HIGH ? 64.0f : 1024.0f);
    return half2v{m, m};
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
    __device__ float d() const { return __fmul_rn(kQ4kUnit, half_bits_to_float((uint16_t)(dd & 0xFFFFu))); }
    __device__ float minus_dmin() const { return -half_bits_to_float((uint16_t)(dd >> 16)); }
};

}  // namespace mummu
