// Router logits of many tokens on the f32 matrix units, in the router's fixed summation order (router.hip), and the routing of
// their tokens in the same launch.
//
// v_mfma_f32_16x16x1_4b_f32 makes four outer products of 16 by 16, each element one fused multiply-add with one rounding (six
// million of them compared with fmaf on the card, subnormal, cancelling, infinite and NaN operands among them: no difference).  So
// an accumulator that takes the elements i, i + 512, i + 1024, ... of a logit one after the other holds partial i mod 512 with the
// bits of the fmaf chain, and adding up the partials is left to the vector ALUs.
//
// What bounds it: the instructions.  A product has 32 clocks for its 1024 multiply-adds (the vector ALUs need 64); the four sums
// and the conversion that go with one follow it rather than run beside it, 53 clocks together.  The streaming form or the
// tiles (router.hip) -> here, a launch among those of its layer: 4096 tokens, 64 experts of 2048, with the routing 40 -> 26 us, 1024 tokens, 512 experts of 2560 65 -> 48
// (a kernel trace has 53 -> 35 and 82 -> 60).  A step's rows read from LDS a step ahead 5 % less; with the tokens' rows read from the caches by every wave instead
// of once into LDS a fifth and a third more.
#include "device_utils.h"
#include "kernels.h"
#include "route_common.h"

namespace mummu {

constexpr int kMatrixTokens = 16, kMatrixWaves = 8;
constexpr int kMatrixMaxHidden = 4096;   // (two quarters of 16 rows in LDS)

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// A workgroup has 16 tokens and four tiles of 16 experts (from 64 * blockIdx.y); two waves split the 512 partials of a tile.  A
// wave walks its half in groups of 32 partials: block b of a product and accumulator j have partial 32 * group + 8 * b + j, so that
// a lane's eight elements of a row are neighbours, and the order of the sums - over a lane's eight as router_logits_kernel has
// them, then b, then the groups - is the one of its adjacent lanes.  The experts' rows come from the caches straight into
// registers, kDeep steps (a group's part of one chunk of 512) ahead.
// ROUTE (one workgroup a token tile): the logits meet in LDS and the waves route two tokens each.
// (x and w are not __restrict__: the loads into LDS have to stay in front of the weights', which a wait counts.)
template <int WT, bool ROUTE>
__global__ __launch_bounds__(64 * kMatrixWaves, 2) void router_matrix_kernel(
    const float *x, const void *w, int n, int hidden, int n_experts, int k, int flavour, int norm,
    float *__restrict__ logits, int32_t *__restrict__ ids, float *__restrict__ weights, unsigned long long *__restrict__ hits,
    int32_t *__restrict__ flags) {
    constexpr int GROUPS = 8, kDeep = 4;
    __shared__ f32x4 s_part[4 * 64];
    __shared__ float s_logit[ROUTE ? kMatrixTokens * 64 : 1];
    __shared__ __attribute__((aligned(16))) RouteScratch<1> sc[ROUTE ? kMatrixWaves : 1];
    const int lane = threadIdx.x & 63, wave = uniform((int)(threadIdx.x >> 6)), tile = wave & 3, run = wave >> 2;
    const int chunks = hidden / 512, t0 = (int)blockIdx.x * kMatrixTokens, e0 = (int)blockIdx.y * 64 + tile * 16;
    const int row = lane & 15, block = lane >> 4;
    // The tokens' rows come through LDS, a quarter of each run (two groups) at a time in one of two buffers: [run][chunk][row][64 elements], the
    // 16-byte pieces of a row exchanged by its number, so that sixteen rows' equal pieces lie in different banks.  A wave's load: four rows' 256 bytes.
    // (tokens and experts past the last repeat it)
    extern __shared__ __attribute__((aligned(16))) uint8_t s_x[];
    const uint32_t quarter_bytes = 8192u * (uint32_t)chunks;
    const int lrow = 4 * tile + (lane >> 4), lt = t0 + lrow < n ? t0 + lrow : n - 1;
    const uint8_t *from_x = (const uint8_t *)(x + (size_t)lt * (size_t)hidden + 32 * GROUPS * run + 4 * ((lane & 15) ^ lrow));
    const uint32_t to_x = lds_offset(s_x) + (uint32_t)(run * chunks) * 4096u + 1024u * (uint32_t)tile;
    auto load_quarter = [&](int q) {
        const uint32_t to = to_x + (uint32_t)(q & 1) * quarter_bytes;
        for (int c = 0; c < chunks; c++) load_to_lds16(to + 4096u * (uint32_t)c, from_x + 256 * q + 2048 * c);
    };
    constexpr int kBytes = WT == T_F32 ? 4 : 2, kWords = kBytes / 2;
    const uint8_t *from_w = (const uint8_t *)w + ((size_t)(e0 + row < n_experts ? e0 + row : n_experts - 1) * (size_t)hidden + 32 * GROUPS * run + 8 * block) * kBytes;
    u32x4 raw[kDeep][kWords];
    int fg = 0, fc = 0;   // the group and chunk the next loads are for (past the last the last again)
    auto fetch = [&](int slot) {
        const u32x4 *pw = (const u32x4 *)(from_w + kBytes * (512 * fc + 32 * fg));
#pragma unroll
        for (int i = 0; i < kWords; i++) raw[slot][i] = pw[i];
        if (++fc == chunks) {
            fc = fg + 1 < GROUPS ? 0 : chunks - 1;
            fg = fg + 1 < GROUPS ? fg + 1 : fg;
        }
    };
    load_quarter(0);
    load_quarter(1);
#pragma unroll
    for (int s = 0; s < kDeep; s++) {
        fetch(s);
        MUMMU_CODE_FENCE();
    }
    // (both quarters: in front of the weights' loads)
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"i"(kDeep * kWords) : "memory");
    const f32x4 *my_x = (const f32x4 *)s_x + run * chunks * 256 + row * 16;
    const int piece0 = (2 * block) ^ row, piece1 = (2 * block + 1) ^ row;   // (of an even group; of an odd one with 8 exchanged)
    // (a step's rows are read a step ahead, but for the first of a quarter, which has to have landed)
    auto read_x = [&](int g, int c, f32x4 (&xa)[2]) {
        const f32x4 *px = my_x + (((g >> 1) & 1) * 2 * chunks + c) * 256;
        xa[0] = px[piece0 ^ (8 * (g & 1))], xa[1] = px[piece1 ^ (8 * (g & 1))];
    };
    f32x4 ahead[2];
    read_x(0, 0, ahead);
    f32x16 acc[8];
    f32x4 level[3], sum;   // level[i]: the sum of 2^i groups that waits for its neighbour
    int c = 0, g = 0;
    for (int step = 0; step < GROUPS * chunks; step += kDeep) {
#pragma unroll
        for (int s = 0; s < kDeep; s++) {
            const f32x4 xa[2] = {ahead[0], ahead[1]};
            const bool last = c + 1 == chunks;   // of the group; of the quarter: with an odd one
            if (!last || !(g & 1)) read_x(last ? g + 1 : g, last ? 0 : c + 1, ahead);
            float wv[8];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                if constexpr (WT == T_F32) {
                    wv[q] = __uint_as_float(raw[s][0][q]);
                    wv[4 + q] = __uint_as_float(raw[s][1][q]);
                } else {
                    const uint16_t lo = (uint16_t)(raw[s][0][q] & 0xFFFFu), hi = (uint16_t)(raw[s][0][q] >> 16);
                    wv[2 * q] = WT == T_F16 ? half_bits_to_float(lo) : bf16_bits_to_float(lo);
                    wv[2 * q + 1] = WT == T_F16 ? half_bits_to_float(hi) : bf16_bits_to_float(hi);
                }
            }
            if (c == 0) {
                const f32x16 zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
                for (int j = 0; j < 8; j++) acc[j] = __builtin_amdgcn_mfma_f32_16x16x1f32(xa[j / 4][j % 4], wv[j], zero, 0, 0, 0);
            } else {
#pragma unroll
                for (int j = 0; j < 8; j++) acc[j] = __builtin_amdgcn_mfma_f32_16x16x1f32(xa[j / 4][j % 4], wv[j], acc[j], 0, 0, 0);
            }
            fetch(s);
            MUMMU_CODE_FENCE();
            if (++c == chunks) {
                c = 0;
                f32x16 v;
#pragma unroll
                for (int i = 0; i < 16; i++)
                    v[i] = __fadd_rn(__fadd_rn(__fadd_rn(acc[0][i], acc[4][i]), __fadd_rn(acc[1][i], acc[5][i])),
                                     __fadd_rn(__fadd_rn(acc[2][i], acc[6][i]), __fadd_rn(acc[3][i], acc[7][i])));
#pragma unroll
                for (int i = 0; i < 4; i++) sum[i] = __fadd_rn(__fadd_rn(v[i], v[4 + i]), __fadd_rn(v[8 + i], v[12 + i]));
                // (a counter in binary: a group's sum goes up while the bits below are ones)
                bool up = true;
#pragma unroll
                for (int b = 0; b < 3; b++) {
                    if (!up) continue;
                    if ((g >> b) & 1) {
#pragma unroll
                        for (int i = 0; i < 4; i++) sum[i] = __fadd_rn(level[b][i], sum[i]);
                    } else {
                        level[b] = sum;
                        up = false;
                    }
                }
                g++;
                if ((g & 1) == 0 && g < GROUPS) {
                    // the next quarter's loads are done: they were asked for in front of the last kDeep steps' weights (with one chunk: not).  Behind
                    // the barrier nobody reads the buffer of this one any more.
                    if (chunks > 1) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"i"(kDeep * kWords) : "memory");
                    else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
                    if (g / 2 + 1 < GROUPS / 2) load_quarter(g / 2 + 1);
                    read_x(g, 0, ahead);
                }
            }
        }
    }
    // lane: expert e0 + lane % 16, tokens 4 * (lane / 16) and on
    if (run == 1) s_part[tile * 64 + lane] = sum;
    __syncthreads();
    if (run == 0) {
        const f32x4 other = s_part[tile * 64 + lane];
        const int e = e0 + row;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int t = 4 * block + i;
            sum[i] = __fadd_rn(sum[i], other[i]);
            if (t0 + t < n && e < n_experts) logits[(size_t)(t0 + t) * (size_t)n_experts + (size_t)e] = sum[i];
            if constexpr (ROUTE) s_logit[t * 64 + 16 * tile + row] = sum[i];
        }
    }
    if constexpr (ROUTE) {
        __syncthreads();
        for (int t = wave; t < kMatrixTokens && t0 + t < n; t += kMatrixWaves) {
            float l[1] = {lane < n_experts ? s_logit[t * 64 + lane] : 0.0f};
            route_token<1>(l, t0 + t, n_experts, k, flavour, norm, ids, weights, hits, flags, sc[wave]);
            wave_lds_sync();
        }
    }
}

bool router_matrix_takes(const float *x, const void *w, int hidden) { return (((uintptr_t)x | (uintptr_t)w) & 15) == 0 && hidden >= 512 && hidden % 512 == 0 && hidden <= kMatrixMaxHidden; }

// Logits alone (route false, any number of experts) or with the routing behind them (up to 64 experts).
hipError_t launch_router_matrix(const float *x, const void *w, int wtype, int n, int hidden, int n_experts, int k, int flavour, int norm, float *logits,
                                int32_t *ids, float *weights, unsigned long long *hits, int32_t *flags, bool route, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    if (!router_matrix_takes(x, w, hidden) || n_experts < 1 || (route && (n_experts > 64 || k > n_experts || k < 1))) return hipErrorInvalidValue;
    const dim3 block(64 * kMatrixWaves), grid((unsigned)((n + kMatrixTokens - 1) / kMatrixTokens), route ? 1u : (unsigned)((n_experts + 63) / 64));
    const size_t lds = (size_t)(hidden / 512) * 16384;
#define MUMMU_RM(WT)                                                                                                                             \
    do {                                                                                                                                         \
        if (route) launch_kernel(router_matrix_kernel<WT, true>, grid, block, lds, s, x, w, n, hidden, n_experts, k, flavour, norm, logits, ids, weights, hits, flags); \
        else launch_kernel(router_matrix_kernel<WT, false>, grid, block, lds, s, x, w, n, hidden, n_experts, k, flavour, norm, logits, ids, weights, hits, flags); \
        return hipGetLastError();                                                                                                                \
    } while (0)
    switch (wtype) {
    case T_F32: MUMMU_RM(T_F32);
    case T_F16: MUMMU_RM(T_F16);
    case T_BF16: MUMMU_RM(T_BF16);
    default: return hipErrorInvalidValue;
    }
#undef MUMMU_RM
}

}  // namespace mummu
