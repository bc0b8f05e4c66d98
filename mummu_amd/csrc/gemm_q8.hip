// Grouped GEMM of Q8_0 banks on the f16 units for few rows per expert (tiles of 32 rows).  Rows are pairs of halfs (HAct), a code
// is a half as it is, and a block's 32 products are summed by v_mfma_f32_16x16x32_f16 into one f32 accumulator, hi and lo
// halfs alike; what is left for the vector ALUs is one multiply-add per output and block, with the block's scale.
//
// What bounds it: the stream of the weights and, not wholly beside it, the CU's own work (with every tile on one expert's weights, out
// of L2, gate/up of the layer below still takes 59 us of its 75; its bytes take 50).  Blocks of 34 bytes loaded by the lanes that
// multiply them kept the address units busy (int8 form: 170 us for a layer whose bytes take 75), 16 bytes a lane straight into
// registers took 237.  Here a stage of a row (128 elements, 136 bytes) comes as the aligned pieces of 16 bytes that hold it, straight into LDS,
// two stages ahead, the loads dealt over the products of a stage: a burst behind the barrier stalls all waves at the address units.
// A workgroup fills a CU's LDS, so what it does outside the loop is not hidden by another: it takes several items, and loads for the
// next while it stores the last.  OLMoE layer, 150 tokens, gate/up + down, us: dwords loaded in a burst 86 + 47; pieces, dealt 80.5 + 45.5; several items 75.2 +
// 42.5; codes read from LDS by whole pieces, 16 lanes of which meet all banks (so do the dwords of two K groups here), 74 + 41 (the layer: 152, 147, 142,
// 139.5; 16 tokens 134 -> 117, 512: 296 -> 255, 1000: 491 -> 412).
// Fetched once: 296 MB of 285.  Tried: half the rows of a stage and two workgroups a CU (84.7 + 60.2: more streams than L2 holds lines
// for, 385 MB); a wave for one block of a stage and 128 columns, a quarter of the reads of rows (81.1 + 54.8: sums exchanged at the end).
// Products of 16 x 16 and 32 of K instead of 32 x 32 and 16, which pass through the accumulators half as often: less power, a higher clock, at four operands a
// block instead of two.  Layers among others, us, 16 / 64 / 150 / 260 / 512 / 1000 / 2000 tokens 86.8 / 101.8 / 110.9 / 149.8 / 229.8 / 391.5 / 708 -> 85.8 / 100.2 / 108.3 / 146.4 /
// 224.9 / 379.8 / 689.5.
// Off the 64-bit result by 2.5e-7 where the int8 form is by 4.5e-5 (four shapes 2.51, 2.49, 2.42, 2.64 e-7 with the larger products, whose high halfs came first; 2.48, 2.47, 2.41,
// 2.63 here).
//
// x has one scale for its whole row (HAct, the largest element lifted to 2^15): an element is off by at most 2^-39 of the row's largest, where
// the int8 form's is off by 2^-16 of the largest of its block of 64.  That is less for every row but one whose large elements fill blocks of
// their own, more than 2^24 above the rest, and meet weights of 0: such a block 2^20 / 2^23 / 2^24 / 2^26 above 3.1e-6 / 2.5e-5 / 4.9e-5 / 2.0e-4
// off the 64-bit result, the int8 form 4.8e-5 each time (with the largest at 2^10, as Q4_K rows have it for their sums' sake, 9.9e-5 / 7.9e-4 / 1.6e-3 /
// 6.4e-3).  A single element 2^20 above, its weights 0: 1.6e-6, the int8 form, which loses its 63 neighbours, 4.7e-1; no element above: 1.7e-7
// and 4.8e-5.
//
// An item is a tile by 256 weight rows (128 of gate and 128 of up), a wave has 32 of them, which it loads for itself; the activation tile
// is shared.  Lane (column c, K group g) reads 8 of the 32 codes of a block of columns c and c + 16 each: elements 8 g + i of the block are the K index
// 8 g + i of its product, and the A operands, rows c and c + 16, are read from the tile to match.
#include <type_traits>

#include "device_utils.h"
#include "gemm_q8_lds.h"
#include "kernels.h"
#include "qact.h"

namespace mummu {

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

using namespace q8;

constexpr int kCusOfXcd = 32;               // (a workgroup fills a CU)
constexpr int kRowC = 128 + 4;               // f32 row of the gate/up epilogue
static_assert(2 * kRows * kRowC * 4 <= kStageW, "the epilogue fits a stage's weights");

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
// PIECES: the aligned pieces of 16 bytes that hold a row's 136 of a stage: nine where rows begin at a multiple of 16 (stages then begin
// there or 8 past it), else ten.
template <bool GATE_UP, int PIECES>
__global__ __launch_bounds__(64 * kWaves, 2) void grouped_gemm_q8_kernel(const uint8_t *__restrict__ w0, const uint8_t *__restrict__ w1, HAct a,
                                                                         const int32_t *__restrict__ sorted, int k_slots,
                                                                         const int32_t *__restrict__ tiles, const int32_t *__restrict__ n_tiles,
                                                                         int in_dim, int out_dim, HAct act, float *__restrict__ y) {
    extern __shared__ __attribute__((aligned(16))) uint8_t s_lds[];   // (gemm_q8_lds.h)
    __shared__ __attribute__((aligned(16))) float s_as[2][64];        // row scales (gate/up: of an item, else of a stage), twice
    __shared__ int32_t s_idx[2][64];                                  // an item's entries of `sorted`, twice
    // as xcd_tile in gemm.hip: an XCD takes neighbouring tiles, the slab running fastest; here a workgroup takes every
    // gridDim.x / 8 -th of its XCD's items, and its loads run on from one into the next
    constexpr int kCols = GATE_UP ? kWCols / 2 : kWCols;
    const int n_slabs = (out_dim + kCols - 1) / kCols;
    const int total = *n_tiles, per_xcd = (total + 7) >> 3, tile0 = (int)(blockIdx.x & 7) * per_xcd;
    const int n_items = n_slabs * (total - tile0 < per_xcd ? total - tile0 : per_xcd), apart = (int)(gridDim.x >> 3);
    const int first_item = (int)(blockIdx.x >> 3);
    if (first_item >= n_items) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6), c = lane & 15, g = lane >> 4, row32 = lane & 31;
    const uint32_t row_bytes = (uint32_t)(in_dim / kStep) * kRowW;
    const uint32_t lds0 = lds_offset(s_lds);
    const uint32_t lds_as = lds_offset(s_as), lds_idx = lds_offset(s_idx);
    const int n_steps = in_dim / kStep;
    auto expert_of = [&](int item) { return uniform(tiles[3 * (tile0 + item / n_slabs)]); };
    auto start_of = [&](int item) { return uniform(tiles[3 * (tile0 + item / n_slabs) + 1]); };
    auto rows_of = [&](int item) { return uniform(tiles[3 * (tile0 + item / n_slabs) + 2]); };
    // this wave's weight rows: first .. first + 31 of gate (waves 0-3), up (4-7) or down
    auto first_of = [&](int item) { return item % n_slabs * kCols + 32 * (GATE_UP ? wave & 3 : wave); };

    // Where the loads stand: an item and its stage, for the weights (two stages ahead of the products) and for the rows (one).
    // Past the last item they stay at its last stage, never multiplied.
    int w_item = first_item, w_step = 0, a_item = first_item, a_step = 0, w_flip = 0, a_flip = 0;
    const uint8_t *w_base = nullptr;
    uint32_t w_off[kWLoads], a_off = 0, s_off = 0;
    // (columns past the matrix repeat its last, rows past the tile's end its last: multiplied, never stored; the lanes past the
    // last piece repeat it)
    auto set_w = [&]() {
        const int first = first_of(w_item);
        w_base = uniform((GATE_UP && wave >= 4 ? w1 : w0) + (size_t)expert_of(w_item) * (size_t)out_dim * row_bytes);
#pragma unroll
        for (int j = 0; j < kWLoads; j++) {
            const int piece = 64 * j + lane < 32 * PIECES ? 64 * j + lane : 32 * PIECES - 1, col = first + piece / PIECES;
            w_off[j] = ((uint32_t)(col < out_dim ? col : out_dim - 1) * row_bytes & ~15u) + (uint32_t)(piece % PIECES) * 16u;
        }
        if (GATE_UP) {
            const int rows = rows_of(w_item);
            load_to_lds4(lds_idx + (uint32_t)w_flip * 256u, (const uint8_t *)(sorted + start_of(w_item)), (uint32_t)(row32 < rows ? row32 : rows - 1) * 4u);
        }
    };
    // Activation pieces: load `wave` of each plane holds four rows.
    const int a_row = 4 * wave + (lane >> 4);
    // An item of up to 16 rows has its low halfs' rows behind its high halfs' in one A operand: half the products and row reads, a row's
    // two parts summed at the end.  OLMoE layer, three streams, 16 / 64 / 100 tokens 89.0 / 103.2 / 105.9 -> 86.3 / 100.8 / 104.1 us, 150 (a third of
    // the tiles) the same; off the 64-bit result by 2.43e-7 where one sum for both is by 2.52e-7.
    const uint32_t a_rd0 = row_read(c, false), a_full = row_read(c + 16, false), a_half = row_read(c + 16, true);
    uint32_t a_rd = a_full, a_low = row_low(false);   // of the item whose rows are being loaded (the first sixteen rows lie where they do either way)
    auto set_a = [&]() {
        const bool few = rows_of(a_item) <= 16;
        a_rd = few ? a_half : a_full, a_low = row_low(few);
        auto source_row = [&](int r) {
            if (GATE_UP) return (uint32_t)(s_idx[a_flip][r] / k_slots);
            const int rows = rows_of(a_item);
            return (uint32_t)(start_of(a_item) + (r < rows ? r : rows - 1));
        };
        a_off = source_row(a_row) * (uint32_t)in_dim * 2u + (uint32_t)((lane & 15) ^ (a_row & 15)) * 16u;
        s_off = source_row(row32) * (uint32_t)(in_dim / 128) * 4u;
        if (GATE_UP) load_to_lds4(lds_as + (uint32_t)a_flip * 256u, (const uint8_t *)a.scale, s_off);
    };
    auto next_w = [&]() {
        if (++w_step < n_steps) return;
        if (w_item + apart < n_items) {
            w_item += apart, w_step = 0, w_flip ^= 1;
            set_w();
        } else {
            w_step = n_steps - 1;
        }
    };
    auto next_a = [&]() {
        if (++a_step < n_steps) return;
        if (a_item + apart < n_items) {
            a_item += apart, a_step = 0, a_flip ^= 1;
            set_a();
        } else {
            a_step = n_steps - 1;
        }
    };
    // one load each
    auto load_w = [&](uint32_t slot, int j) {
        load_to_lds16(lds0 + slot + (uint32_t)wave * kWaveW + 1024 * j, w_base + ((size_t)(w_step >> 1) * (2 * kRowW) + (size_t)(w_step & 1) * (kRowW - 8)),
                      w_off[j]);
    };
    auto load_a = [&](int which, int i) {
        const uint32_t at = lds0 + rows_at(which) + (uint32_t)wave * 1024u;
        if (i == 0) load_to_lds16(at, (const uint8_t *)a.hi + (size_t)a_step * (kStep * 2), a_off);
        else if (i == 1) load_to_lds16(at + kPlane, (const uint8_t *)a.lo + (size_t)a_step * (kStep * 2), a_off);
        else load_to_lds4(lds_as + (uint32_t)which * 256u, (const uint8_t *)a.scale + (size_t)a_step * 4, s_off);   // (every wave the same)
    };
    constexpr int kALoads = GATE_UP ? 2 : 3;
    set_w();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    set_a();
#pragma unroll
    for (int j = 0; j < kWLoads; j++) load_w(0, j);
#pragma unroll
    for (int i = 0; i < kALoads; i++) load_a(0, i);
    next_w();
#pragma unroll
    for (int j = 0; j < kWLoads; j++) load_w(kStageW, j);

    const f32x4 zero = {0, 0, 0, 0};
    // what a block's products take: 8 codes and the scale of either column, the rows' pieces; of this block and of the next
    uint32_t v[2][2][3];
    float d[2][2];
    half8 hi[2][2], lo[2][2];
    uint32_t w_rd[2];
#pragma unroll
    for (int j = 0; j < 2; j++) w_rd[j] = (uint32_t)wave * kWaveW + (uint32_t)(c + 16 * j) * (16 * PIECES) + (PIECES == 9 ? 0u : (uint32_t)c * row_bytes & 8u);
    auto read = [&](uint32_t slot, int odd, int which, int blk, uint32_t rd, uint32_t low, bool both) {   // (odd: of the stage, known where PIECES is 9)
        const int at = 34 * blk + 2, n = blk & 1;
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const uint8_t *ds = s_lds + slot + w_rd[j] + 8u * (uint32_t)odd;
            // (the dwords of sixteen columns, 9 pieces apart, and two K groups lie in all banks)
#pragma unroll
            for (int i = 0; i < ((at & 2) ? 3 : 2); i++) v[n][j][i] = *(const uint32_t *)(ds + 8u * (uint32_t)g + (at & ~3) + 4 * i);
            d[n][j] = half_bits_to_float(*(const uint16_t *)(ds + 34 * blk));
        }
        const uint8_t *as = s_lds + rows_at(which);
        const uint32_t piece = row_piece(c, g >> 1, blk, g & 1);
#pragma unroll
        for (int m = 0; m < 2; m++) {
            const uint8_t *from = as + (m == 0 ? a_rd0 : rd) + piece;
            hi[n][m] = *(const half8 *)from;
            if (both) lo[n][m] = *(const half8 *)(from + low);
        }
    };
    // a block's sum -> acc, or (down) the 128 elements' sum
    f32x4 acc[2][2], run[2][2], s[2][2][2];   // [16 rows][16 columns]; s of this block and of the one before
    float fd[2] = {0.0f, 0.0f};
    auto clear = [&]() {
#pragma unroll
        for (int m = 0; m < 4; m++) acc[m >> 1][m & 1] = run[m >> 1][m & 1] = s[1][m >> 1][m & 1] = zero;
    };
    clear();
    auto fold = [&](int n, int blk) {
#pragma unroll
        for (int m = 0; m < 2; m++)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    if (GATE_UP) acc[m][j][r] = fmaf(fd[j], s[n][m][j][r], acc[m][j][r]);
                    else run[m][j][r] = blk == 0 ? __fmul_rn(fd[j], s[n][m][j][r]) : fmaf(fd[j], s[n][m][j][r], run[m][j][r]);
                }
    };
    // the stage's row scales, read in front of its last barrier: the stage after the next lands in their place
    float4 sr[2] = {};
    auto read_scales = [&](int which, bool half) {
#pragma unroll
        for (int m = 0; m < 2; m++) sr[m] = *(const float4 *)&s_as[which][(half ? 0 : 16 * m) + 4 * g];
    };
    auto fold_run = [&]() {
#pragma unroll
        for (int m = 0; m < 2; m++) {
            const float f[4] = {sr[m].x, sr[m].y, sr[m].z, sr[m].w};
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int r = 0; r < 4; r++) acc[m][j][r] = fmaf(run[m][j][r], f[r], acc[m][j][r]);
        }
    };
    // element r of acc[m][j]: row 16 m + 4 g + r, column 16 j + c of the wave's
    auto acc_row = [&](int m, int r) { return 16 * m + 4 * g + r; };

    // the first stage is there; its first block
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kWLoads) : "memory");
    read(0, 0, 0, 0, a_rd, a_low, true);
    uint32_t slot = 0;   // of the stage's weights
    int which = 0;       // of its rows
    for (int item = first_item, flip = 0; item < n_items; item += apart, flip ^= 1) {
        auto stage = [&](int step, auto odd, auto half) {
            const uint32_t rd = half ? a_half : a_full;
            const uint32_t slot1 = slot == (kRing - 1) * kStageW ? 0 : slot + kStageW, slot2 = slot1 == (kRing - 1) * kStageW ? 0 : slot1 + kStageW;
            next_a();
            next_w();
#pragma unroll
            for (int blk = 0; blk < kBlocks; blk++) {
                const int n = blk & 1;
                // In front of a stage's last products: everything but the weights of the stage after the next is there, for this
                // wave; then, the activations, for everybody, who have also read this stage's.
                if (blk == 3) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kWLoads) : "memory");
                // beside the first three, a few at a time: the next step's rows, then the weights of the one after
                if (blk == 0) {
#pragma unroll
                    for (int i = 0; i < kALoads; i++) load_a(which ^ 1, i);
                } else if (blk < 3) {
#pragma unroll
                    for (int j = 3 * blk - 3; j < 3 * blk && j < kWLoads; j++) load_w(slot2, j);
                }
                const float now[2] = {d[n][0], d[n][1]};
                half8 w[2];
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    // (codes begin two bytes into a dword in every other block)
                    const uint32_t *q = v[n][j];
                    w[j] = ((34 * blk + 2) & 2) ? q8_codes(__builtin_amdgcn_alignbyte(q[1], q[0], 2), __builtin_amdgcn_alignbyte(q[2], q[1], 2))
                                                : q8_codes(q[0], q[1]);
                }
                const half8 h[2] = {hi[n][0], hi[n][1]}, l[2] = {lo[n][0], lo[n][1]};
                if (blk < 3) read(slot, PIECES == 9 ? odd : step & 1, which, blk + 1, rd, row_low(half), !half);
                else read(slot1, PIECES == 9 ? !odd : step + 1 < n_steps ? (step + 1) & 1 : 0, which ^ 1, 0, a_rd, a_low, true);
#pragma unroll
                for (int part = half ? 1 : 0; part < 2; part++)   // (the low halfs first: the smaller sum is rounded less often at the size of the larger)
#pragma unroll
                    for (int m = 0; m < 2; m++)
#pragma unroll
                        for (int j = 0; j < 2; j++)
                            s[n][m][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(part ? h[m] : l[m], w[j], part == (half ? 1 : 0) ? zero : s[n][m][j], 0, 0, 0);
                // the block before this one, while these are multiplied
                fold(n ^ 1, (blk + 3) & 3);
                if (!GATE_UP && blk == 0) fold_run();
                if (!GATE_UP && blk == 2) read_scales(which, half);
                fd[0] = now[0], fd[1] = now[1];
            }
            slot = slot1;
            which ^= 1;
        };
        const int p0 = start_of(item), rows = rows_of(item);
        auto stages = [&](auto half) {
            for (int step = 0; step < n_steps;) {
                stage(step++, std::integral_constant<int, 0>(), half);
                if (PIECES == 9) stage(step++, std::integral_constant<int, 1>(), half);   // (stages come in pairs)
            }
        };
        if (rows > 16) stages(std::integral_constant<bool, false>());
        else stages(std::integral_constant<bool, true>());
        fold(1, 3);
        if (!GATE_UP) fold_run();
        if (rows <= 16) {
#pragma unroll
            for (int j = 0; j < 2; j++) acc[0][j] += acc[1][j];
        }
        if (GATE_UP) {
            // (the last stage's weights are read: their place is free until the loads beside the next item's products)
            float *s_c = (float *)(s_lds + (slot == 0 ? (kRing - 1) * kStageW : slot - kStageW));   // [gate, up][row][kRowC]
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int m = i >> 3, j = i >> 2 & 1, row = acc_row(m, i & 3);
                s_c[((wave >> 2) * kRows + row) * kRowC + 32 * (wave & 3) + 16 * j + c] = __fmul_rn(s_as[flip][row], acc[m][j][i & 3]);
            }
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
            for (int pass = 0; pass < kRows / 16; pass++) {
                const int row = 16 * pass + (tid >> 5), at = row * kRowC + 4 * (tid & 31);
                const float4 gv = *(const float4 *)&s_c[at], uv = *(const float4 *)&s_c[kRows * kRowC + at];
                const float4 r = make_float4(__fmul_rn(det_silu(gv.x), uv.x), __fmul_rn(det_silu(gv.y), uv.y), __fmul_rn(det_silu(gv.z), uv.z),
                                             __fmul_rn(det_silu(gv.w), uv.w));
                const bool active = row < rows;
                hact_store128(active ? r : make_float4(0.f, 0.f, 0.f, 0.f), active, act, (size_t)(p0 + row), out_dim,
                              item % n_slabs * kCols + 4 * (tid & 31), kHActLift);
            }
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        } else {
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int m = i >> 3, j = i & 1, r = i >> 1 & 3, row = acc_row(m, r), col = first_of(item) + 16 * j + c;
                if (col < out_dim && row < rows) y[(size_t)(p0 + row) * (size_t)out_dim + (size_t)col] = acc[m][j][r];
            }
        }
        clear();
        fd[0] = fd[1] = 0.0f;
#pragma unroll
        for (int m = 0; m < 2; m++) sr[m] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (no load into LDS is under way when the workgroup ends)
}

template <bool GATE_UP>
hipError_t launch_q8(const uint8_t *w0, const uint8_t *w1, HAct a, const int32_t *sorted, int k_slots, const int32_t *tiles,
                     const int32_t *n_tiles, int max_tiles, int in_dim, int out_dim, HAct act, float *y, hipStream_t s) {
    constexpr int kCols = GATE_UP ? kWCols / 2 : kWCols;
    const int per_xcd = (max_tiles + 7) / 8 * ((out_dim + kCols - 1) / kCols);
    const dim3 grid(8u * (unsigned)(per_xcd < kCusOfXcd ? per_xcd : kCusOfXcd));
    if (in_dim % (2 * kStep) == 0)
        launch_kernel(grouped_gemm_q8_kernel<GATE_UP, 9>, grid, dim3(64 * kWaves), kLdsBytes, s, w0, w1, a, sorted, k_slots, tiles, n_tiles,
                      in_dim, out_dim, act, y);
    else
        launch_kernel(grouped_gemm_q8_kernel<GATE_UP, 10>, grid, dim3(64 * kWaves), kLdsBytes, s, w0, w1, a, sorted, k_slots, tiles, n_tiles,
                      in_dim, out_dim, act, y);
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
