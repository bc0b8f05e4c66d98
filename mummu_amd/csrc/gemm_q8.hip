// Grouped GEMM of Q8_0 banks on the f16 units for few rows per expert (tiles of 32 rows).  Rows are pairs of halfs (HAct), a code
// is a half as it is, and a block's 32 products are summed by v_mfma_f32_32x32x16_f16 into one f32 accumulator, hi and lo
// halfs alike; what is left for the vector ALUs is one multiply-add per output and block, with the block's scale.
//
// What bounds it: the stream of the weights, if it gets into the CU.  Blocks of 34 bytes loaded by the lanes that multiply them
// (dwords of 64 rows a load) kept the address units busy: one line a lane and load, and the int8 form took 170 us for a layer whose
// bytes take 75, whatever the batch; 16 bytes a lane straight into registers took 237.  Here a row's 136 bytes of a
// stage (128 elements) come in one piece, 64 neighbouring dwords a load, straight into LDS, two stages ahead: 141 us (OLMoE layer, 19
// to 100 tokens; 150: 204 -> 153, 512: 350 -> 294; each byte is fetched once, 295 MB of 285 at 3.5 TB/s with the vector ALUs busy for 29 %
// of the cycles and the matrix units for 18, profiles/listed_work_counters.txt), 2.5e-7 off the 64-bit result where the int8 form is by 4.5e-5.
//
// x has one scale for its whole row (HAct): an element is off by at most 2^-34 of the row's largest, where the int8 form's is off
// by 2^-16 of the largest of its block of 64.  That is less for every row but one whose large elements fill blocks of their own and
// meet weights of 0: a block 2^20 (2^26) above the rest 1.0e-4 (6.4e-3) off the 64-bit result, the int8 form 4.6e-5.  A single element
// 2^20 above it, its weights 0: 5.0e-5, the int8 form, which loses its 63 neighbours, 2.4e-1; weights as they come: 3.3e-7 and 3.1e-5.
//
// A workgroup has 256 weight rows (128 of gate and 128 of up), a wave 32 of them, which it loads for itself; the activation tile is
// shared.  Lane (column c, K group g) reads 16 of a block's 32 codes, so element 16 g + 8 kk + i of the block is the K index
// 8 g + i of its product kk, and the A operands are read from the tile to match.
#include "device_utils.h"
#include "kernels.h"
#include "qact.h"

namespace mummu {

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float16v __attribute__((ext_vector_type(16)));

constexpr int kRows = 32;                    // rows of a tile
constexpr int kWaves = 8, kWCols = 32 * kWaves;
constexpr int kStep = 128, kBlocks = 4;      // K elements and blocks of a stage
constexpr int kRowW = 136;                   // bytes of a weight row's stage, in memory and in LDS
constexpr int kWLoads = 32 * kRowW / 256;    // loads of a wave's weights: 64 dwords each
constexpr int kWaveW = 32 * kRowW, kStageW = kWaves * kWaveW, kRing = 3;
constexpr int kPlane = kRows * kStep * 2, kStageA = 2 * kPlane;   // hi, lo: [row][16 pieces of 16 bytes]
constexpr int kLdsBytes = kRing * kStageW + 2 * kStageA;
constexpr int kRowC = 128 + 4;               // f32 row of the gate/up epilogue
static_assert(32 * kRowW % 256 == 0 && 2 * kRows * kRowC * 4 <= kLdsBytes, "whole loads; the epilogue fits the stages");

// Eight codes as halfs, in the element order of HAct: a byte b ^ 0x80 under 0x64 is the half 1024 + 128 + b.
__device__ inline half8 q8_codes(uint32_t w0, uint32_t w1) {
    const half2v bias = {(_Float16)1152.0f, (_Float16)1152.0f};
    auto pair = [&](uint32_t w, uint32_t pick) {
        const uint32_t u = __builtin_amdgcn_perm(0x64646464u, w ^ 0x80808080u, pick);
        half2v h;
        __builtin_memcpy(&h, &u, 4);
        return h - bias;
    };
    const half2v f[4] = {pair(w0, 0x04020400u), pair(w0, 0x04030401u), pair(w1, 0x04020400u), pair(w1, 0x04030401u)};
    half8 o;
    __builtin_memcpy(&o, f, 16);
    return o;
}

// GATE_UP: a = the token rows gathered through `sorted`, one scale per row; silu(g) * u leaves as HAct in sorted order.
// else   : a in sorted order, a scale per 128 elements; y[pos, n] = f32 sum.
template <bool GATE_UP>
__global__ __launch_bounds__(64 * kWaves, 2) void grouped_gemm_q8_kernel(const uint8_t *__restrict__ w0, const uint8_t *__restrict__ w1, HAct a,
                                                                         const int32_t *__restrict__ sorted, int k_slots,
                                                                         const int32_t *__restrict__ tiles, const int32_t *__restrict__ n_tiles,
                                                                         int in_dim, int out_dim, HAct act, float *__restrict__ y) {
    extern __shared__ __attribute__((aligned(16))) uint8_t s_lds[];   // [kRing][kStageW], then [2][kStageA]
    __shared__ __attribute__((aligned(16))) float s_as[2][64];        // row scales (gate/up: [0], else of a stage), twice
    // as xcd_tile in gemm.hip: an XCD takes neighbouring tiles, the slab running fastest
    constexpr int kCols = GATE_UP ? kWCols / 2 : kWCols;
    const int n_slabs = (out_dim + kCols - 1) / kCols;
    const int total = *n_tiles, per_xcd = (total + 7) >> 3;
    const int item = (int)(blockIdx.x >> 3), within = item / n_slabs, slab = item - within * n_slabs;
    const int tile = (int)(blockIdx.x & 7) * per_xcd + within;
    if (within >= per_xcd || tile >= total) return;
    const int e = uniform(tiles[3 * tile]), p0 = uniform(tiles[3 * tile + 1]), rows = uniform(tiles[3 * tile + 2]);
    const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6), c = lane & 31, g = lane >> 5;
    const uint32_t row_bytes = (uint32_t)(in_dim / kStep) * kRowW;
    const uint32_t lds0 = lds_offset(s_lds);
    const uint32_t lds_as = lds_offset(s_as);
    const int n_steps = in_dim / kStep;

    // this wave's weight rows: first .. first + 31 of gate (waves 0-3), up (4-7) or down
    const int first = slab * kCols + 32 * (GATE_UP ? wave & 3 : wave);
    const uint8_t *w_base = uniform((GATE_UP && wave >= 4 ? w1 : w0) + (size_t)e * (size_t)out_dim * row_bytes);
    // (columns past the matrix repeat its last, rows past the tile's end its last: multiplied, never stored)
    uint32_t w_off[kWLoads];
#pragma unroll
    for (int j = 0; j < kWLoads; j++) {
        const int d = 64 * j + lane, col = first + d / (kRowW / 4);
        w_off[j] = (uint32_t)(col < out_dim ? col : out_dim - 1) * row_bytes + (uint32_t)(d % (kRowW / 4)) * 4u;
    }
    auto source_row = [&](int r) {
        r = r < rows ? r : rows - 1;
        return (uint32_t)(GATE_UP ? sorted[p0 + r] / k_slots : p0 + r);
    };
    // Activation pieces: load `wave` of each plane holds four rows.  Piece q of row r lies at q ^ (r % 16): sixteen lanes that read
    // the same piece of neighbouring rows meet all banks.
    const int a_row = 4 * wave + (lane >> 4);
    const uint32_t a_off = source_row(a_row) * (uint32_t)in_dim * 2u + (uint32_t)((lane & 15) ^ (a_row & 15)) * 16u;
    const uint32_t s_off = source_row(c) * (uint32_t)(in_dim / 128) * 4u;
    auto load_w = [&](int step) {
        const uint32_t at = lds0 + (uint32_t)(step % kRing) * kStageW + (uint32_t)wave * kWaveW;
        const uint8_t *base = w_base + (size_t)step * kRowW;
#pragma unroll
        for (int j = 0; j < kWLoads; j++) load_to_lds4(at + 256 * j, base, w_off[j]);
    };
    auto load_a = [&](int step) {
        const uint32_t at = lds0 + kRing * kStageW + (uint32_t)(step & 1) * kStageA + (uint32_t)wave * 1024u;
        load_to_lds16(at, (const uint8_t *)a.hi + (size_t)step * (kStep * 2), a_off);
        load_to_lds16(at + kPlane, (const uint8_t *)a.lo + (size_t)step * (kStep * 2), a_off);
        if (!GATE_UP) load_to_lds4(lds_as + (uint32_t)(step & 1) * 256u, (const uint8_t *)a.scale + (size_t)step * 4, s_off);   // (every wave the same)
    };
    if (GATE_UP && tid < 64) s_as[0][tid] = *(const float *)((const uint8_t *)a.scale + s_off);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

    const float16v zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    float16v acc = zero;
    load_w(0);
    load_a(0);
    if (n_steps > 1) load_w(1);
    for (int step = 0; step < n_steps; step++) {
        // everything but the next stage's weights is there, for this wave; then, the activations, for everybody, who are also
        // done with the tile of the step before
        if (step + 1 < n_steps) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kWLoads) : "memory");
        else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (step + 1 < n_steps) load_a(step + 1);
        if (step + 2 < n_steps) load_w(step + 2);
        const uint8_t *ws = s_lds + (uint32_t)(step % kRing) * kStageW + (uint32_t)wave * kWaveW + (uint32_t)c * kRowW + 16u * (uint32_t)g;
        const uint8_t *ds = ws - 16u * (uint32_t)g;
        const uint8_t *as = s_lds + kRing * kStageW + (uint32_t)(step & 1) * kStageA + (uint32_t)c * (kStep * 2);
        float16v run = zero;
#pragma unroll
        for (int blk = 0; blk < kBlocks; blk++) {
            // 16 codes from byte 34 blk + 2 on: two bytes into a dword in every other block
            constexpr int kDwords = 5;
            uint32_t v[kDwords], q[4];
            const int at = 34 * blk + 2, off = at & ~3;
#pragma unroll
            for (int i = 0; i < ((at & 2) ? 5 : 4); i++) v[i] = *(const uint32_t *)(ws + off + 4 * i);
#pragma unroll
            for (int i = 0; i < 4; i++) q[i] = (at & 2) ? __builtin_amdgcn_alignbyte(v[i + 1], v[i], 2) : v[i];
            const float d = half_bits_to_float(*(const uint16_t *)(ds + 34 * blk));
            const half8 w[2] = {q8_codes(q[0], q[1]), q8_codes(q[2], q[3])};
            float16v s = zero;
#pragma unroll
            for (int kk = 0; kk < 2; kk++) {
                const uint8_t *piece = as + (uint32_t)(((4 * blk + 2 * g + kk) ^ (c & 15)) * 16);
                const half8 hi = *(const half8 *)piece, lo = *(const half8 *)(piece + kPlane);
                s = __builtin_amdgcn_mfma_f32_32x32x16_f16(hi, w[kk], s, 0, 0, 0);
                s = __builtin_amdgcn_mfma_f32_32x32x16_f16(lo, w[kk], s, 0, 0, 0);
            }
#pragma unroll
            for (int r = 0; r < 16; r++) {
                if (GATE_UP) acc[r] = fmaf(d, s[r], acc[r]);
                else run[r] = blk == 0 ? __fmul_rn(d, s[r]) : fmaf(d, s[r], run[r]);
            }
        }
        if (!GATE_UP) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float4 s4 = *(const float4 *)&s_as[step & 1][8 * j + 4 * g];
                const float sr[4] = {s4.x, s4.y, s4.z, s4.w};
#pragma unroll
                for (int i = 0; i < 4; i++) acc[4 * j + i] = fmaf(run[4 * j + i], sr[i], acc[4 * j + i]);
            }
        }
    }

    // element r of an accumulator: row 8 (r / 4) + 4 g + r % 4, column lane % 32
    auto acc_row = [&](int r) { return 8 * (r >> 2) + 4 * g + (r & 3); };
    if (GATE_UP) {
        __syncthreads();   // (the stages are done with)
        float *s_c = (float *)s_lds;   // [gate, up][row][kRowC]
#pragma unroll
        for (int r = 0; r < 16; r++) s_c[((wave >> 2) * kRows + acc_row(r)) * kRowC + 32 * (wave & 3) + c] = __fmul_rn(s_as[0][acc_row(r)], acc[r]);
        __syncthreads();
#pragma unroll
        for (int pass = 0; pass < kRows / 16; pass++) {
            const int row = 16 * pass + (tid >> 5), at = row * kRowC + 4 * (tid & 31);
            const float4 gv = *(const float4 *)&s_c[at], uv = *(const float4 *)&s_c[kRows * kRowC + at];
            const float4 v = make_float4(__fmul_rn(det_silu(gv.x), uv.x), __fmul_rn(det_silu(gv.y), uv.y), __fmul_rn(det_silu(gv.z), uv.z),
                                         __fmul_rn(det_silu(gv.w), uv.w));
            const bool active = row < rows;
            hact_store128(active ? v : make_float4(0.f, 0.f, 0.f, 0.f), active, act, (size_t)(p0 + row), out_dim, slab * kCols + 4 * (tid & 31));
        }
    } else if (first + c < out_dim) {
#pragma unroll
        for (int r = 0; r < 16; r++)
            if (acc_row(r) < rows) y[(size_t)(p0 + acc_row(r)) * (size_t)out_dim + (size_t)(first + c)] = acc[r];
    }
}

template <bool GATE_UP>
hipError_t launch_q8(const uint8_t *w0, const uint8_t *w1, HAct a, const int32_t *sorted, int k_slots, const int32_t *tiles,
                     const int32_t *n_tiles, int max_tiles, int in_dim, int out_dim, HAct act, float *y, hipStream_t s) {
    constexpr int kCols = GATE_UP ? kWCols / 2 : kWCols;
    const dim3 grid((unsigned)((max_tiles + 7) / 8 * 8) * (unsigned)((out_dim + kCols - 1) / kCols));
    launch_kernel(grouped_gemm_q8_kernel<GATE_UP>, grid, dim3(64 * kWaves), kLdsBytes, s, w0, w1, a, sorted, k_slots, tiles, n_tiles, in_dim,
                  out_dim, act, y);
    return hipGetLastError();
}

}  // namespace

bool q8_gemm_takes(const ExpertBanks &b) {
    // (one expert's matrix is addressed with 32-bit byte offsets; the gate/up slabs are whole)
    return b.gate_type == T_Q8_0 && b.up_type == T_Q8_0 && b.down_type == T_Q8_0 && b.hidden % kStep == 0 && b.inter % kStep == 0 &&
           (size_t)b.hidden * (size_t)b.inter / kStep * kRowW < (1ull << 32);
}

hipError_t launch_q8_gate_up(const ExpertBanks &b, HAct x, const int32_t *sorted, int k_slots, const int32_t *tiles, const int32_t *n_tiles,
                             int max_tiles, HAct act, hipStream_t s) {
    return launch_q8<true>(b.gate, b.up, x, sorted, k_slots, tiles, n_tiles, max_tiles, b.hidden, b.inter, act, nullptr, s);
}

hipError_t launch_q8_down(const ExpertBanks &b, HAct act, const int32_t *tiles, const int32_t *n_tiles, int max_tiles, float *y, hipStream_t s) {
    return launch_q8<false>(b.down, nullptr, act, nullptr, 1, tiles, n_tiles, max_tiles, b.inter, b.hidden, HAct(), y, s);
}

}  // namespace mummu
