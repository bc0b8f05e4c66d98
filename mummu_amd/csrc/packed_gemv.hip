// Packed GEMV over burn's block-32 quantized weight layout: the custom-op seam of the reference,
// Q4GemvOps::q4s_gemv (nn/packed_gemv.rs:248-260), whose CubeCL kernel is packed_gemv_kernel
// (nn/packed_gemv.rs:370-451).
//
// Layout (nn/packed_gemv.rs:26-29, pack.rs:940-985): the weight is [K, N] row-major, values two's
// complement in 4 (Q4S) or 8 (Q8S) bits, element j of a u32 word at bits j*bits, words running along
// N; one f32 scale per (k, block of 32 consecutive n).  The op is
//     y[n] = sum_k float(q(k, n)) * (x[k] * scale(k, n / 32)),
// the product x*scale rounded, the product with q rounded, then added (two roundings, as the
// reference's kernel and its dequantize-then-matmul form do).
//
// The sum over k runs on the matrix cores, in v_mfma_f32_16x16x32_bf16, without giving up precision: a code of up to 8
// bits is a bf16, and the f32 product x*scale is the exact sum of three (its first, second and third 8 significant bits),
// so three products into one f32 accumulator see every bit that the reference's arithmetic sees.  On the vector ALUs a
// weight cost ten operations at four rows and the launch was bound by them ([5120, 17408] Q4S, 4 rows 28.6 us for the
// 9.5 us its bytes take; 64 rows 327 us).
//
// Since the scale goes with x, a row of the A operand belongs to a block of 32 columns.  A operands hold R rows of x for
// 16 / R neighbouring blocks, and a product of them with 16 columns gives R x 16 results that are wanted and 16 / R - 1
// times as many that are not: R = 4 for up to 4 rows, 8 for up to 8, else 16 and up to two A operands a weight.  What the
// split of x*scale costs (6.5 operations an element of A) sinks with 16 / R, what a decoded weight costs (1.6) is shared
// by the A operands.
//
// Two waves take 256 columns (whole 128-byte lines of words: with half lines the requests are the limit, 34 against 29 us
// on [8192, 20480]) and a slice of K, the words, scales and x straight from memory into LDS, a stage of 32 k ahead.  A word
// holds 8 (or 4) columns at one k, so reading it for eight k gives a lane the B operands of as many columns without a
// transposition.  Four such pairs are a workgroup and meet in LDS in ascending order, the workgroups of a column group through
// partial sums, added in ascending order by the one that comes last, or, if they or the rows are many, by a second kernel.  Which slice a k belongs to and the order of every sum depend on the weight alone: a row's bits are the same whatever
// shares the launch.
//
// [5120, 17408] Q4S, 1 / 4 / 16 / 64 rows: 17.6 / 29.1 / 86 / 327 -> 17.5 / 17.8 / 26.9 / 88 us; Q8S 25.8 / 38.0 / 108 / 407 ->
// 22.9 / 24.4 / 37 / 102; [2048, 4096] Q4S 9.4 / 17.6 / 18.3 / 36.5 -> 7.8 / 8.2 / 10.9 / 16.5.  Nearest to
// a bound now are the vector ALUs (700 clocks of decoding and splitting per 32 x 128 weights at up to 4 rows, 1220 at 16; a launch of 4
// rows, 18.9 us or some 42 k clocks in a trace, has 17.8 k clocks of them and 8.2 k of the matrix units on each SIMD), below 10 MB the
// chain of launch, first load and meeting of the partial sums (6 us).
#include "device_utils.h"
#include "host_staging.h"
#include "kernels.h"

#include <algorithm>
#include <mutex>
#include <string>
#include <type_traits>

#include "../../include/mummu_moe.h"

MUMMU_TRACE_UNIT(packed_gemv)

namespace mummu {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr int kPgSlices = 4;      // K slices of a workgroup, each a pair of waves
constexpr int kPgCols = 128;      // columns of a wave: four scale blocks
constexpr int kPgGroup = 2 * kPgCols;   // columns of a pair, and of the workgroup
constexpr int kPgStage = 32;      // K elements of a stage
constexpr int kLastRows = 8;      // up to which the last workgroup of a column group may add the partial sums: one row group

struct PackedArgs {
    const uint32_t *words;   // [k_len][n_words]
    const float *scales;     // [k_len][n_blocks]
    const float *x;          // [m][k_len]
    int m, k_len, n_words, n_blocks;
    int stages;              // of kPgStage k, dealt evenly to the slices
    int wg_x, grid_k;        // column groups of kPgGroup, workgroups along K
    bool words16, x16;       // the words, the rows of x are 16-byte aligned
    float *out;              // y, or [grid_k][m][n] partial sums
    float *y;                // not null (one row group only): the last workgroup of a column group adds the partial sums into it
    unsigned *arrived;       // ... counted here, [wg_x], 0 between launches
};

// The four-bit code in the low half of byte `b` of w, over 16 (the sums are multiplied by 16 at the end).
template <int B>
__device__ inline float nibble(uint32_t w) {
    float f;
    if constexpr (B == 0) asm("v_cvt_off_f32_i4_sdwa %0, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_0" : "=v"(f) : "v"(w));
    if constexpr (B == 1) asm("v_cvt_off_f32_i4_sdwa %0, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_1" : "=v"(f) : "v"(w));
    if constexpr (B == 2) asm("v_cvt_off_f32_i4_sdwa %0, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_2" : "=v"(f) : "v"(w));
    if constexpr (B == 3) asm("v_cvt_off_f32_i4_sdwa %0, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_3" : "=v"(f) : "v"(w));
    return f;
}
template <int B>
__device__ inline float byte_code(uint32_t w) { return (float)(int8_t)(w >> (8 * B)); }

// bf16 pair: the upper halves of two floats (with kNoHalves: two zeros).
constexpr uint32_t kUpperHalves = 0x07060302u, kNoHalves = 0x0C0C0C0Cu;
__device__ inline uint32_t upper_halves(float lo, float hi, uint32_t pick = kUpperHalves) {
    return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), pick);
}

template <int BITS, int R, int RT>
struct PackedMap {
    static constexpr int WORDS = kPgGroup * BITS / 32;  // words of a pair's columns at one k
    static constexpr int GROUPS = R / 4;                // passes over a wave's four blocks, 4 / GROUPS blocks each
    static constexpr int SETS = 32 / R;                 // B operands of a pass: columns per lane
    static constexpr int LANE_WORDS = BITS == 8 && R == 4 ? 2 : 1;
    // bytes of a stage: words [kPgStage][WORDS], scales [kPgStage][8], x [RT * R][kPgStage]
    static constexpr int S_AT = kPgStage * WORDS * 4, X_AT = S_AT + kPgStage * 32, STAGE = X_AT + RT * R * kPgStage * 4;
    // ... of the slices' sums, rows a little longer than the columns; behind them a word per wave
    static constexpr int SUM_ROW = kPgGroup + 4, SUMS = kPgSlices * R * SUM_ROW * 4, RING = kPgSlices * 2 * STAGE;
    static constexpr int LDS = RING > SUMS + 32 ? RING : SUMS + 32;
};

// RT row tiles of R rows of workgroup `lin`'s columns and part of K, into p.out; true if a sum of this lane came out as NaN.
// lower: kUpperHalves; kNoHalves: x*scale is its first part alone, and only sums that are NaN in p.out are written.
template <int BITS, int R, int RT>
__device__ inline bool packed_tile(const PackedArgs &p, uint8_t *s_lds, int tid, int lin, uint32_t lower) {
    using Map = PackedMap<BITS, R, RT>;
    constexpr int WORDS = Map::WORDS, GROUPS = Map::GROUPS, SETS = Map::SETS, LW = Map::LANE_WORDS;
    constexpr int PIECES = WORDS / 4, KS = kPgStage;
    constexpr int S_AT = Map::S_AT, X_AT = Map::X_AT, STAGE = Map::STAGE;
    const int lane = tid & 63, wave = uniform(tid >> 6);
    const int n = lane & 15, g = lane >> 4;
    const int kpart = lin / p.wg_x, wg = lin - kpart * p.wg_x;
    const int row0 = (int)blockIdx.y * (RT * R), rows = p.m - row0;
    const int half = wave & 1, slice = kpart * kPgSlices + (wave >> 1);
    const int block0 = wg * (kPgGroup / 32);
    // (a stage more or less than the other slices: what a CU has to do is the sum over its workgroups)
    const int n_slices = p.grid_k * kPgSlices;
    const int k0 = (int)((int64_t)slice * p.stages / n_slices) * KS, k_end = (int)((int64_t)(slice + 1) * p.stages / n_slices) * KS;
    const int k1 = k_end < p.k_len ? k_end : p.k_len;
    const int most = (p.stages + n_slices - 1) / n_slices;

    // A stage in LDS.  Row rho of its 32 is k = 8 (rho % 4) + rho / 4: lane group g reads its k = 8 g + i at rho = 4 i + g.
    // Words of row rho change places with those at ^ turn(rho): the four groups' reads then meet all banks.
    auto k_of = [](int rho) { return 8 * (rho & 3) + (rho >> 2); };
    auto turn = [](int rho) { return BITS == 8 ? (rho & 1) * 32 + ((rho >> 1) & 1) * 20 : ((rho >> 1) & 1) * 16; };
    // x: 16 bytes at slot q of row r are those at q ^ x_turn(r), to the same end.  (rows past m repeat the last)
    auto x_turn = [](int row) { return row & 7; };
    auto x_row = [&](int row) { return row < rows ? row : rows - 1; };
    auto x_k = [&](int d) { return ((d % KS / 4) ^ x_turn(d / KS)) * 4 + (d & 3); };   // k of dword d
    const uint32_t row_bytes = (uint32_t)p.n_words * 4u, srow_bytes = (uint32_t)p.n_blocks * 4u;
    const uint32_t lds0 = lds_offset(s_lds) + (uint32_t)(wave >> 1) * (2 * STAGE);
    auto block = [&](int b) { return block0 + b < p.n_blocks ? block0 + b : p.n_blocks - 1; };   // (columns past the last block repeat it)
    // byte offset in a k row of the word at place w of row rho
    auto word_off = [&](int rho, int w) {
        const int src = w ^ turn(rho);
        return (uint32_t)(block(src / BITS) * (BITS * 4) + src % BITS * 4);
    };
    // Loads of a stage, half of them each wave's: of 16 bytes a lane (words; x if its rows allow) or 4.
    constexpr int W16 = KS * PIECES / 128, S4 = KS / 16, X4 = RT * R * KS / 128, X16 = RT * R * KS / 512;
    // A whole stage: lane offsets once, the rest in the base addresses.
    const uint32_t w_off = (uint32_t)k_of(lane / PIECES) * row_bytes + word_off(lane / PIECES, lane % PIECES * 4);
    const uint32_t s_off = (uint32_t)k_of(lane >> 3) * srow_bytes + 4u * (uint32_t)block(lane & 7);
    uint32_t x_off16[X16 > 0 ? X16 : 1];
#pragma unroll
    for (int j = 0; j < X16; j++)
        x_off16[j] = (uint32_t)(x_row(8 * (half * X16 + j) + (lane >> 3)) * p.k_len + x_k(256 * (half * X16 + j) + 4 * lane)) * 4u;
    const uint32_t x_lane = (uint32_t)((lane & 31) * 4) ^ (uint32_t)(x_turn(lane >> 5) << 4), x_upper = (uint32_t)(lane >> 5) * (uint32_t)p.k_len * 4u;
    auto stage = [&](int slot, int kb) {
        const uint32_t at = lds0 + (uint32_t)slot * STAGE;
        const uint8_t *wb = (const uint8_t *)p.words + (size_t)kb * row_bytes, *sb = (const uint8_t *)p.scales + (size_t)kb * srow_bytes;
        const uint8_t *xb = (const uint8_t *)(p.x + (size_t)row0 * (size_t)p.k_len + (size_t)kb);
        if (kb + KS <= p.k_len && p.words16) {
            // (load j of the words holds rows 64 / PIECES j .., which are k of load 0's rows plus 16 / PIECES j)
#pragma unroll
            for (int i = 0; i < W16; i++) {
                const int j = half * W16 + i;
                load_to_lds16(at + 1024 * j, wb + (size_t)(16 / PIECES * j) * row_bytes, w_off);
            }
#pragma unroll
            for (int i = 0; i < S4; i++) {
                const int j = half * S4 + i;
                load_to_lds4(at + S_AT + 256 * j, sb + (size_t)(2 * j) * srow_bytes, s_off);
            }
            if (X16 > 0 && p.x16) {
#pragma unroll
                for (int i = 0; i < X16; i++) load_to_lds16(at + X_AT + 1024 * (half * X16 + i), xb, x_off16[i]);
            } else {
                // load j: rows 2 j and 2 j + 1
#pragma unroll
                for (int i = 0; i < X4; i++) {
                    const int j = half * X4 + i;
                    load_to_lds4(at + X_AT + 256 * j, xb + (size_t)x_row(2 * j) * (size_t)p.k_len * 4,
                                 (x_lane ^ (uint32_t)(x_turn(2 * j) << 4)) + (2 * j + 1 < rows ? x_upper : 0u));
                }
            }
            return;
        }
        const int last = p.k_len - 1 - kb;   // (rows past the end of K repeat the last: x and scales count as 0 there)
        auto k_in = [&](int k) { return (uint32_t)(k < last ? k : last); };
        for (int i = 0; i < 4 * W16; i++) {
            const int d = 64 * (half * 4 * W16 + i) + lane, rho = d / WORDS;
            load_to_lds4(at + 256 * (half * 4 * W16 + i), wb, k_in(k_of(rho)) * row_bytes + word_off(rho, d % WORDS));
        }
        for (int j = half * S4; j < (half + 1) * S4; j++)
            load_to_lds4(at + S_AT + 256 * j, sb, k_in(k_of(8 * j + (lane >> 3))) * srow_bytes + 4u * (uint32_t)block(lane & 7));
        for (int j = half * X4; j < (half + 1) * X4; j++)
            load_to_lds4(at + X_AT + 256 * j, xb, ((uint32_t)(x_row(2 * j + (lane >> 5)) * p.k_len) + k_in(x_k(64 * j + lane))) * 4u);
    };

    // What a lane reads of a stage: of rows 4 i + g the word(s) whose columns it multiplies, in block n / R of a pass, that
    // block's scales, and its rows of x
    const int word = half * (WORDS / 2) + (BITS == 8 ? 8 * (n / R) + (R == 4 ? n & 3 : n & 7) : 4 * (n / R) + (n & 3));
    uint32_t w_lane[GROUPS];
#pragma unroll
    for (int b = 0; b < GROUPS; b++) w_lane[b] = (uint32_t)(g * WORDS + ((word + b * (WORDS / 2 / GROUPS)) ^ turn(g))) * 4u;
    const int w_second = (((word + 4) ^ turn(g)) - (word ^ turn(g))) * 4;
    const uint32_t s_lane = (uint32_t)(8 * g + 4 * half + n / R) * 4u;
    uint32_t x_lane16[2];
#pragma unroll
    for (int h = 0; h < 2; h++) x_lane16[h] = (uint32_t)(n % R * KS + ((2 * g + h) ^ x_turn(n % R)) * 4) * 4u;

    f32x4 acc[RT][GROUPS][SETS];
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
        for (int b = 0; b < GROUPS; b++)
#pragma unroll
            for (int c = 0; c < SETS; c++) acc[t][b][c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    if (k0 < k1) stage(0, k0);
    for (int i = 0, kb = k0; i < most; i++, kb += KS) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        uint8_t *st = s_lds + (size_t)(wave >> 1) * (2 * STAGE) + (size_t)(i & 1) * STAGE;
        if (kb < k1 && kb + KS > k1) {   // past the end of K
            for (int d = half * 64 * X4 + lane; d < (half + 1) * 64 * X4; d += 64)
                if (kb + x_k(d) >= k1) *(float *)(st + X_AT + 4 * d) = 0.0f;
            for (int d = half * 64 * S4 + lane; d < (half + 1) * 64 * S4; d += 64)
                if (kb + k_of(d >> 3) >= k1) *(float *)(st + S_AT + 4 * d) = 0.0f;
        }
        // the stage is there for both waves of the pair, and everybody has read the one before it
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (kb + KS < k1) stage(~i & 1, kb + KS);
        if (kb < k1) {
            const uint8_t *s_rd = st + S_AT + s_lane, *x_rd = st + X_AT;
#pragma unroll
            for (int b = 0; b < GROUPS; b++) {
                __builtin_amdgcn_sched_barrier(0);   // (one pass's operands at a time: registers)
                uint32_t wv[LW][8];
                float sv[8];
#pragma unroll
                for (int i = 0; i < 8; i++) {
#pragma unroll
                    for (int h = 0; h < LW; h++)
                        wv[h][i] = *(const uint32_t *)(st + w_lane[b] + (h == 0 ? 0 : w_second) + 16 * i * WORDS);
                    sv[i] = *(const float *)(s_rd + 128 * i + 4 * b * (4 / GROUPS));
                }
                // x * scale, in three
                bf16x8 a[RT][3];
#pragma unroll
                for (int t = 0; t < RT; t++) {
                    float r[8];
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        const f32x4 xv = *(const f32x4 *)(x_rd + x_lane16[h] + t * (R * KS * 4));
#pragma unroll
                        for (int i = 0; i < 4; i++) r[4 * h + i] = __fmul_rn(xv[i], sv[4 * h + i]);
                    }
#pragma unroll
                    for (int part = 0; part < 3; part++) {
                        u32x4 v;
#pragma unroll
                        for (int i = 0; i < 4; i++) v[i] = upper_halves(r[2 * i], r[2 * i + 1], part > 0 ? lower : kUpperHalves);
                        __builtin_memcpy(&a[t][part], &v, 16);
                        if (part < 2)
#pragma unroll
                            for (int i = 0; i < 8; i++) r[i] = __fsub_rn(r[i], __uint_as_float(__float_as_uint(r[i]) & 0xFFFF0000u));
                    }
                }
                // columns of this lane: byte c of its words (8 bits; R 16: of one shifted by its upper two bytes), or the
                // nibbles at an even or odd place of each byte (R 4: both)
                uint32_t odd[8];
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    if constexpr (BITS == 8 && R == 16) wv[0][i] >>= 16 * (n >> 3);
                    if constexpr (BITS == 4 && R == 4) odd[i] = wv[0][i] >> 4;
                    if constexpr (BITS == 4 && R > 4) wv[0][i] >>= 4 * ((n >> 2) % (R / 4));
                }
                auto operand = [&](auto dec, const uint32_t(&w)[8]) {
                    u32x4 v;
#pragma unroll
                    for (int i = 0; i < 4; i++) v[i] = upper_halves(dec(w[2 * i]), dec(w[2 * i + 1]));
                    bf16x8 o;
                    __builtin_memcpy(&o, &v, 16);
                    return o;
                };
                // (two columns at a time: a product waits for the one before it in its accumulator)
                auto multiply = [&](int c, bf16x8 w0, bf16x8 w1) {
#pragma unroll
                    for (int part = 2; part >= 0; part--)
#pragma unroll
                        for (int t = 0; t < RT; t++) {
                            acc[t][b][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t][part], w0, acc[t][b][c], 0, 0, 0);
                            acc[t][b][c + 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t][part], w1, acc[t][b][c + 1], 0, 0, 0);
                        }
                };
                if constexpr (BITS == 4 && R == 4) {
                    multiply(0, operand(nibble<0>, wv[0]), operand(nibble<0>, odd));
                    multiply(2, operand(nibble<1>, wv[0]), operand(nibble<1>, odd));
                    multiply(4, operand(nibble<2>, wv[0]), operand(nibble<2>, odd));
                    multiply(6, operand(nibble<3>, wv[0]), operand(nibble<3>, odd));
                } else if constexpr (BITS == 4 && R == 8) {
                    multiply(0, operand(nibble<0>, wv[0]), operand(nibble<1>, wv[0]));
                    multiply(2, operand(nibble<2>, wv[0]), operand(nibble<3>, wv[0]));
                } else if constexpr (BITS == 4) {
                    multiply(0, operand(nibble<0>, wv[0]), operand(nibble<2>, wv[0]));
                } else {
                    multiply(0, operand(byte_code<0>, wv[0]), operand(byte_code<1>, wv[0]));
                    if constexpr (R < 16) multiply(2, operand(byte_code<2>, wv[0]), operand(byte_code<3>, wv[0]));
                    if constexpr (R == 4) {
                        multiply(4, operand(byte_code<0>, wv[LW - 1]), operand(byte_code<1>, wv[LW - 1]));
                        multiply(6, operand(byte_code<2>, wv[LW - 1]), operand(byte_code<3>, wv[LW - 1]));
                    }
                }
            }
        }
    }

    // The slices' sums, [kPgSlices][R][kSumRow]: a wave's columns as its accumulators hold them (lane n of operand c of pass b
    // at (b SETS + c) 16 + n), the row a little longer than the columns, so that its four lane groups write side by side.
    constexpr int kSumRow = Map::SUM_ROW;
    float *s_sum = (float *)s_lds;
    const size_t out_n = (size_t)p.n_blocks * 32;
    const bool last_adds = R <= kLastRows && p.y != nullptr;
    const int place = tid % kPgGroup, pn = place & 15, pc = (place >> 4) % SETS, pb = place % kPgCols / (16 * SETS);
    const int in_block = BITS == 8 ? (R == 4 ? 4 * ((pn & 3) + 4 * (pc >> 2)) + (pc & 3) : 4 * (pn & 7) + (R == 16 ? 2 * (pn >> 3) : 0) + pc)
                                   : 8 * (pn & 3) + (R == 4 ? pc : (R == 8 ? ((pn >> 2) & 1) + 2 * pc : (pn >> 2) + 4 * pc));
    const size_t col = (size_t)wg * kPgGroup + (size_t)(place / kPgCols * kPgCols + 32 * (pb * (4 / GROUPS) + pn / R) + in_block);
    bool nan = false;
#pragma unroll
    for (int t = 0; t < RT; t++) {
        __syncthreads();
        // accumulator element e of lane (n, g) is row 4 g + e of the A operand: x row (4 g + e) % R of block (4 g + e) / R
        if (4 * g / R == n / R) {
#pragma unroll
            for (int b = 0; b < GROUPS; b++)
#pragma unroll
                for (int c = 0; c < SETS; c++)
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        s_sum[((wave >> 1) * R + 4 * g % R + e) * kSumRow + half * kPgCols + (b * SETS + c) * 16 + n] = acc[t][b][c][e];
        }
        __syncthreads();
        constexpr int EACH = R * kPgGroup / 512;   // (all reads out before the first sum is stored: 34.6 -> 33.6 us, [4096, 8192] Q8S, 32 rows)
        float sum[EACH];
#pragma unroll
        for (int i = 0; i < EACH; i++) {
            sum[i] = 0.0f;
#pragma unroll
            for (int s = 0; s < kPgSlices; s++) sum[i] = __fadd_rn(sum[i], s_sum[(s * R + tid / kPgGroup + 512 / kPgGroup * i) * kSumRow + place]);
            if (BITS == 4) sum[i] = __fmul_rn(sum[i], 16.0f);
        }
#pragma unroll
        for (int i = 0; i < EACH; i++) {
            const int r = R * t + tid / kPgGroup + 512 / kPgGroup * i;
            if (r >= rows || col >= out_n) continue;
            float *dst = p.out + ((size_t)kpart * (size_t)p.m + (size_t)(row0 + r)) * out_n + col;
            if (lower == kNoHalves) {
                const float was = __hip_atomic_load(dst, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // (this lane's own store)
                if (was == was) continue;
            }
            nan |= sum[i] != sum[i];
            if (last_adds) __hip_atomic_store(dst, sum[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // past this XCD's L2
            else *dst = sum[i];
        }
    }
    return nan;
}

// The partial sums of a column group into p.y, by the workgroup that has left the last of them.
__device__ inline void add_parts(const PackedArgs &p, int wg) {
    const size_t out_n = (size_t)p.n_blocks * 32;
    // ascending parts, 16 loads out before the first add (a missing part adds +0.0, which changes nothing)
    auto add = [&](auto items, auto parts) {
        constexpr int ITEMS = decltype(items)::value, PARTS = decltype(parts)::value;
        for (int i0 = (int)threadIdx.x; i0 < p.m * kPgGroup; i0 += 512 * ITEMS) {
            float sum[ITEMS];
            size_t at[ITEMS];
            bool in[ITEMS];
#pragma unroll
            for (int j = 0; j < ITEMS; j++) {
                const int i = i0 + 512 * j, c = wg * kPgGroup + i % kPgGroup;
                sum[j] = 0.0f;
                in[j] = i < p.m * kPgGroup && c < p.n_blocks * 32;
                at[j] = (size_t)(in[j] ? i / kPgGroup : 0) * out_n + (size_t)(in[j] ? c : 0);
            }
            for (int s0 = 0; s0 < p.grid_k; s0 += PARTS) {
                float v[ITEMS][PARTS];
#pragma unroll
                for (int u = 0; u < PARTS; u++)
#pragma unroll
                    for (int j = 0; j < ITEMS; j++) {
                        const int part = s0 + u < p.grid_k ? s0 + u : 0;
                        v[j][u] = __hip_atomic_load(p.out + (size_t)part * (size_t)p.m * out_n + at[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    }
#pragma unroll
                for (int u = 0; u < PARTS; u++)
#pragma unroll
                    for (int j = 0; j < ITEMS; j++) sum[j] = __fadd_rn(sum[j], s0 + u < p.grid_k ? v[j][u] : 0.0f);
            }
#pragma unroll
            for (int j = 0; j < ITEMS; j++)
                if (in[j]) p.y[at[j]] = sum[j];
        }
    };
    if (p.grid_k <= 4) add(std::integral_constant<int, 4>(), std::integral_constant<int, 4>());
    else if (p.grid_k <= 8) add(std::integral_constant<int, 2>(), std::integral_constant<int, 8>());
    else add(std::integral_constant<int, 1>(), std::integral_constant<int, 16>());
}

template <int BITS, int R, int RT>
__global__ __launch_bounds__(512, (PackedMap<BITS, R, RT>::STAGE > 10240 ? 2 : 4)) void packed_gemv_kernel(PackedArgs p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t s_lds[];   // [kPgSlices][2][STAGE]; then the slices' sums, and a word per wave
    // workgroups of an XCD (equal ids modulo 8) take neighbouring column groups: they share the lines of the scales
    const int total = p.wg_x * p.grid_k, per_xcd = (total + 7) >> 3;
    const int lin = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per_xcd || lin >= total) return;
    int *s_nan = (int *)(s_lds + PackedMap<BITS, R, RT>::SUMS);
    // An infinite x*scale has inf - inf in its second part, where the products themselves are infinite and their sum may well be.
    // A workgroup that finds a sum to be NaN forms its sums again of first parts alone: they hold the infinities, beside which the rest
    // does not count; what was a number stays.  (One such row among 4: [5120, 17408] Q4S 20 -> 30 us, Q8S 26 -> 37, [2048, 50304] Q4S
    // 25 -> 39.  Term by term, each row and column by a lane, it made 184, 201 and 275 of them.)
    for (uint32_t lower = kUpperHalves;; lower = kNoHalves) {
        // (nothing derived from these is kept in registers for the second time: the kernel's one argument, read again, and its ids)
        int tid = threadIdx.x, id = lin;
        const __attribute__((address_space(4))) PackedArgs *args = (const __attribute__((address_space(4))) PackedArgs *)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+v"(tid), "+s"(id), "+s"(args), "+s"(lower));
        const PackedArgs q = *(const PackedArgs *)args;
        const int nan = __ballot(packed_tile<BITS, R, RT>(q, s_lds, tid, id, lower)) != 0;
        if ((threadIdx.x & 63) == 0) s_nan[threadIdx.x >> 6] = nan;
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // (no wait for the stores of the sums)
        int any = 0;
#pragma unroll
        for (int w = 0; w < 2 * kPgSlices; w++) any |= s_nan[w];
        if (uniform(any) == 0 || lower == kNoHalves) break;
        __syncthreads();
    }
    if constexpr (R <= kLastRows) {   // (the counter and the sums are those of all rows: forms with one row group)
        if (p.y == nullptr) return;
        // the sums of this workgroup are in memory before it counts; the counter returns to 0 with the last
        const int wg = lin % p.wg_x;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        unsigned *s_last = (unsigned *)s_lds;
        if (threadIdx.x == 0) *s_last = atomicInc(p.arrived + wg, (unsigned)p.grid_k - 1);
        __syncthreads();
        if (*s_last == (unsigned)p.grid_k - 1) add_parts(p, wg);
    }
}

template <int BITS, int R, int RT>
void launch_packed(const PackedArgs &p, hipStream_t s) {
    const dim3 grid((unsigned)(p.wg_x * p.grid_k + 7) / 8 * 8, (unsigned)(p.m + RT * R - 1) / (RT * R));
    launch_kernel(packed_gemv_kernel<BITS, R, RT>, grid, dim3(512), (size_t)PackedMap<BITS, R, RT>::LDS, s, p);
}

template <int BITS>
void launch_packed_rows(const PackedArgs &p, hipStream_t s) {
    if (p.m <= 4) launch_packed<BITS, 4, 1>(p, s);
    else if (p.m <= 8) launch_packed<BITS, 8, 1>(p, s);
    // (8-bit stages leave room for one workgroup per CU at 16 rows or 32, and the decoding is shared: 64 rows of [5120, 17408]
    // 134 us with one tile, 106 with two; 4-bit: two workgroups, 92 with one tile, 99 with two)
    else if (BITS == 4 || p.m <= 16) launch_packed<BITS, 16, 1>(p, s);
    else if constexpr (BITS == 8) launch_packed<BITS, 16, 2>(p, s);
}

}  // namespace

__global__ __launch_bounds__(256) void packed_gemv_sum_kernel(const float *__restrict__ partial, int slices, size_t n,
                                                              float *__restrict__ y) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    // ascending slices, eight loads out before the first add (a missing slice adds +0.0, which changes nothing)
    float total = 0.0f;
    for (int s0 = 0; s0 < slices; s0 += 8) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = s0 + u < slices ? partial[(size_t)(s0 + u) * n + i] : 0.0f;
#pragma unroll
        for (int u = 0; u < 8; u++) total = __fadd_rn(total, v[u]);
    }
    y[i] = total;
}

}  // namespace mummu

using namespace mummu;

struct mummu_packed_weight {
    uint32_t *words = nullptr;  // device [K][n_words]
    float *scales = nullptr;    // device [K][N/32]
    float *x = nullptr, *y = nullptr, *partial = nullptr;  // staging for the host-pointer call and the K partials
    unsigned *arrived = nullptr;  // per column group: workgroups that have left their partial sums
    int k = 0, n = 0, bits = 4, wg_x = 1, grid_k = 1, stages = 1;
    bool owns_weight = true;  // false: words and scales are the caller's device buffers
    hipStream_t stream = nullptr;
    std::mutex mu;
    std::string error;
};

namespace {

constexpr int kMaxRows = 64;  // nn/packed_gemv.rs:138: row by row up to 64 rows
thread_local std::string g_packed_error;

int pfail(mummu_packed_weight *w, int code, const std::string &msg) {
    if (w) w->error = msg;
    g_packed_error = msg;
    return code;
}

// Whether the last workgroup of a column group adds the partial sums or a second launch does, for 0.3 to 0.8 us.  What the last one
// costs grows with the rows, the parts and the workgroups that end together with it; from 64 column groups on, two workgroups to a CU,
// they end one after the other (us, last workgroup / second launch, Q4S):
//   parts x column groups   3 x 16     6 x 7      6 x 16     8 x 7      8 x 16     12 x 4     16 x 4     16 x 16     16 x 32     7 x 68
//   1 row                   7.3/7.8    7.2/7.8    7.8/7.9    7.3/7.8    8.2/7.7    7.5/8.1    7.7/8.1    10.2/8.3    11.3/11.0   19.8/20.0
//   4 rows                  7.6/8.1    7.8/8.2    8.4/8.2    8.0/8.2    8.8/8.1    8.9/8.5    9.1/8.5    11.5/8.7    12.3/11.5   19.7/20.3
//   8 rows                  8.6/9.2    9.5/9.3    9.9/9.3    9.5/9.2    10.3/9.1   11.7/9.5   11.9/9.5   14.3/9.8    16.2/13.7   23.2/23.8
// (16 rows, several row groups: 2 x 16 10.9/10.8, 8 x 16 13.4/10.9, 16 x 16 20.0/11.7; 32 parts lose at any number of rows)
bool last_workgroup_adds(const mummu_packed_weight *w, int m) {
    const int parts = w->grid_k, workgroups = parts * w->wg_x;
    if (m > kLastRows) return false;
    return w->wg_x >= 64 || (m * parts <= 32 && (parts <= 6 || workgroups <= 64 || (workgroups > 256 && parts <= 16)));
}

int enqueue(mummu_packed_weight *w, const float *x_dev, int m, float *y_dev, hipStream_t s) {
    const size_t out_n = (size_t)m * (size_t)w->n;
    const bool parts = w->grid_k > 1, last_adds = parts && last_workgroup_adds(w, m);
    const PackedArgs p{w->words, w->scales, x_dev, m, w->k, w->n * w->bits / 32, w->n / 32, w->stages, w->wg_x, w->grid_k,
                       ((uintptr_t)w->words & 15) == 0, ((uintptr_t)x_dev & 15) == 0 && w->k % 4 == 0, parts ? w->partial : y_dev, last_adds ? y_dev : nullptr, w->arrived};
    if (w->bits == 4) launch_packed_rows<4>(p, s);
    else launch_packed_rows<8>(p, s);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess && parts && !last_adds) {
        launch_kernel(packed_gemv_sum_kernel, dim3((unsigned)((out_n + 255) / 256)), dim3(256), 0, s, (const float *)w->partial,
                      w->grid_k, out_n, y_dev);
        e = hipGetLastError();
    }
    if (e != hipSuccess) return pfail(w, MUMMU_ERR_DEVICE, std::string("packed gemv launch: ") + hipGetErrorString(e));
    return MUMMU_OK;
}

}  // namespace

extern "C" {

const char *mummu_packed_last_error(void) { return g_packed_error.c_str(); }

static int packed_create(const uint32_t *words, const float *scales, int k, int n, int value_bits, bool on_device,
                         mummu_packed_weight **out) {
    if (!out) return pfail(nullptr, MUMMU_ERR_ARG, "null argument");
    *out = nullptr;
    if (!words || !scales) return pfail(nullptr, MUMMU_ERR_ARG, "null weight buffer");
    if (value_bits != 4 && value_bits != 8)
        return pfail(nullptr, MUMMU_ERR_TYPE, "packed weight: " + std::to_string(value_bits) + "-bit values are not supported (Q4S and Q8S are)");
    if (k < 1 || n < 1 || n % 32 != 0)
        return pfail(nullptr, MUMMU_ERR_SHAPE, "packed weight: [" + std::to_string(k) + ", " + std::to_string(n) +
                                                   "] needs K >= 1 and N a positive multiple of the 32-value scale block");
    int devices = 0;
    if (hipGetDeviceCount(&devices) != hipSuccess || devices < 1) {
        (void)hipGetLastError();
        return pfail(nullptr, MUMMU_ERR_DEVICE, "no HIP device");
    }
    auto *w = new mummu_packed_weight();
    HostStaging::retain();
    w->k = k;
    w->n = n;
    w->bits = value_bits;
    w->owns_weight = !on_device;
    const int n_words = n * value_bits / 32;
    // K split over the grid: one round of two workgroups (16 waves) per CU, of slices of at least two stages (shorter ones only
    // make more partial sums)
    w->stages = (k + kPgStage - 1) / kPgStage;
    w->wg_x = (n + kPgGroup - 1) / kPgGroup;
    w->grid_k = std::max(1, std::min(512 / w->wg_x, (w->stages + 2 * kPgSlices - 1) / (2 * kPgSlices)));
    const size_t wb = sizeof(uint32_t) * (size_t)k * (size_t)n_words, sb = sizeof(float) * (size_t)k * (size_t)(n / 32);
    hipError_t e = hipSuccess;
    if (on_device) {
        w->words = const_cast<uint32_t *>(words);
        w->scales = const_cast<float *>(scales);
    } else {
        e = hipMalloc(&w->words, wb);
        if (e == hipSuccess) e = hipMalloc(&w->scales, sb);
    }
    if (e == hipSuccess) e = hipMalloc(&w->x, sizeof(float) * (size_t)kMaxRows * (size_t)k);
    if (e == hipSuccess) e = hipMalloc(&w->y, sizeof(float) * (size_t)kMaxRows * (size_t)n);
    if (e == hipSuccess) e = hipMalloc(&w->partial, sizeof(float) * (size_t)w->grid_k * (size_t)kMaxRows * (size_t)n);
    if (e == hipSuccess) e = hipMalloc(&w->arrived, sizeof(unsigned) * (size_t)w->wg_x);
    if (e == hipSuccess) e = hipMemset(w->arrived, 0, sizeof(unsigned) * (size_t)w->wg_x);
    if (e == hipSuccess) e = hipStreamCreate(&w->stream);
    if (e == hipSuccess && !on_device) e = hipMemcpy(w->words, words, wb, hipMemcpyHostToDevice);
    if (e == hipSuccess && !on_device) e = hipMemcpy(w->scales, scales, sb, hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        const std::string msg = std::string("packed weight: ") + hipGetErrorString(e);
        mummu_packed_weight_destroy(w);
        return pfail(nullptr, MUMMU_ERR_DEVICE, msg);
    }
    *out = w;
    return MUMMU_OK;
}

int mummu_packed_weight_create(const uint32_t *words, const float *scales, int k, int n, int value_bits,
                               mummu_packed_weight **out) {
    return packed_create(words, scales, k, n, value_bits, false, out);
}

int mummu_packed_weight_wrap_device(const uint32_t *words_dev, const float *scales_dev, int k, int n, int value_bits,
                                    mummu_packed_weight **out) {
    return packed_create(words_dev, scales_dev, k, n, value_bits, true, out);
}

void mummu_packed_weight_destroy(mummu_packed_weight *w) {
    if (!w) return;
    if (w->stream) {
        (void)hipStreamSynchronize(w->stream);
        (void)hipStreamDestroy(w->stream);
    }
    if (w->owns_weight) {
        (void)hipFree(w->words);
        (void)hipFree(w->scales);
    }
    (void)hipFree(w->x);
    (void)hipFree(w->y);
    (void)hipFree(w->partial);
    (void)hipFree(w->arrived);
    HostStaging::release();
    delete w;
}

uint64_t mummu_packed_weight_bytes(const mummu_packed_weight *w) {
    if (!w) return 0;
    return (uint64_t)w->k * (uint64_t)w->n * (uint64_t)w->bits / 8 + (uint64_t)w->k * (uint64_t)(w->n / 32) * 4;
}

int mummu_q4s_gemv(mummu_packed_weight *w, const float *x, int64_t m, int k, float *y) {
    if (!w) return pfail(nullptr, MUMMU_ERR_ARG, "null weight");
    std::lock_guard<std::mutex> lock(w->mu);
    if (k != w->k) return pfail(w, MUMMU_ERR_SHAPE, "input width " + std::to_string(k) + " does not match the weight's K " + std::to_string(w->k));
    if (m < 0 || m > kMaxRows) return pfail(w, MUMMU_ERR_TOKENS, std::to_string(m) + " rows: the packed GEMV takes 0 to 64 rows a call");
    if (m == 0) return MUMMU_OK;
    if (!x || !y) return pfail(w, MUMMU_ERR_ARG, "null buffer");
    HostStaging io;
    const size_t xb = sizeof(float) * (size_t)m * (size_t)k, yb = sizeof(float) * (size_t)m * (size_t)w->n;
    hipError_t e = io.valid() ? io.upload(w->x, x, xb, w->stream) : hipMemcpyAsync(w->x, x, xb, hipMemcpyHostToDevice, w->stream);
    if (e != hipSuccess) return pfail(w, MUMMU_ERR_DEVICE, std::string("packed gemv upload: ") + hipGetErrorString(e));
    const int rc = enqueue(w, w->x, (int)m, w->y, w->stream);
    if (rc) return rc;
    if (io.valid()) {
        const HostStaging::Piece out{y, w->y, yb};
        int status = 0;
        e = io.download(&out, 1, nullptr, 0, w->stream, [](const void *) { return 0; }, &status);
    } else {
        e = hipMemcpyAsync(y, w->y, yb, hipMemcpyDeviceToHost, w->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(w->stream);
    }
    if (e != hipSuccess) return pfail(w, MUMMU_ERR_DEVICE, std::string("packed gemv: ") + hipGetErrorString(e));
    return MUMMU_OK;
}

int mummu_q4s_gemv_device(mummu_packed_weight *w, const float *x_dev, int64_t m, int k, float *y_dev, void *stream) {
    if (!w) return pfail(nullptr, MUMMU_ERR_ARG, "null weight");
    if (k != w->k) return pfail(w, MUMMU_ERR_SHAPE, "input width " + std::to_string(k) + " does not match the weight's K " + std::to_string(w->k));
    if (m < 0 || m > kMaxRows) return pfail(w, MUMMU_ERR_TOKENS, std::to_string(m) + " rows: the packed GEMV takes 0 to 64 rows a call");
    if (m == 0) return MUMMU_OK;
    if (!x_dev || !y_dev) return pfail(w, MUMMU_ERR_ARG, "null device pointer");
    return enqueue(w, x_dev, (int)m, y_dev, (hipStream_t)stream);
}

}  // extern "C"
