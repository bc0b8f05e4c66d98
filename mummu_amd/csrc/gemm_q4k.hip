// Grouped GEMM of Q4_K banks on the f16 units: rows as pairs of halfs (HAct), sc * q < 1024 as exact halfs, so that the matrix units
// sum x * (sc * q) over a whole super-block (down: 128 elements of it) before d and dmin are applied; the offset term is one
// more instruction per fold, the sums of the blocks (hi and lo halfs) against the m.  Tiles of up to 64 rows by 256 weight rows (128 of
// gate and 128 of up, or 256 of down).
//
// What bounds it: the card's power (with weights of zeros a layer of 1000 tokens takes 211 us instead of 275), and next to it the issue of the vector
// instructions, 4.3 to 32 k operations.  So:
//   - v_mfma_f32_16x16x32_f16, which passes through the accumulators half as often as 32x32x16: 1.93 -> 2.14 GHz.  It takes four operands of
//     columns where that took two, with twice the scales to a lane, so the clocks are 11 % more, dealt as they are below; but a tile costs
//     what its rows are in steps of 16, where it was 32.
//   - The operand of the next columns is made beside this one's products, by all rows and both halfs; what a fold takes of the header, and the next
//     step's scales, beside an operand's last products; the fold itself beside the next ones'.  (Folds of four operands in a row, behind the
//     products: 1000 tokens 259 us, 4096 953.)  s_setprio around the products: 947 against 930.
//   - two workgroups of four waves to a CU (80 KB of LDS, 256 registers), which drift apart: one folds, ends or begins while the
//     other multiplies.  One of eight waves in step, with 128 rows by 512 columns and each code expanded once for all, was slower
//     (the form before: 4096 rows x 8 gate/up 600 us against 561).
//   - everything from memory straight into LDS: activations two stages ahead of three, the codes a wave multiplies itself half a
//     super-block ahead, no register or vector instruction between.
//   - silu in 17 instructions instead of 60.
// OLMoE layers among others, 32x32x16 with tiles in steps of 32 -> this, us: 150 tokens 84 -> 80.6, 300: 114.5 -> 104.6, 600: 181.7 -> 177.6, 1000: 259 ->
// 257, 4096: 931 / 932; 1000 of 128 experts of 2048 x 768 242.7 -> 238.3, of the 512-expert shape 593 -> 553.
#include "device_utils.h"
#include "kernels.h"
#include "q4k_half.h"
#include "qact.h"

namespace mummu {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kWaves = 4, kWCols = 64 * kWaves;  // weight rows of a tile, 64 to a wave
constexpr int kWaveW = 64 * 64;                  // the codes of 128 elements, 64 bytes a row
constexpr int kRing = 3;                         // stages of 64 elements of the activations
constexpr int kRowC = 128 + 4;                   // f32 row of the gate/up epilogue

// Where things lie in LDS.
constexpr int kRows = kQ4kRows;
constexpr int kPlane = kRows * 128;               // a stage's half plane: 64 elements a row
constexpr int kSlotA = 2 * kPlane;                // hi, lo
constexpr int kAtW = kRing * kSlotA;              // codes: [wave][64 rows][64 bytes]
constexpr int kAtH = kAtW + kWaves * kWaveW;      // headers, two super-blocks: [2][wave][64 rows][16 bytes]
constexpr int kAtF = kAtH + 2 * kWaves * 1024;    // sums of 32 elements of x / scale, as they come: [row][8] f32
constexpr int kAtS = kAtF + kRows * 32;           // ... as pairs of halfs, two super-blocks: [2][row][16]
constexpr int kAtC = kAtS + 2 * kRows * 32;       // scales: down [2][row / 32][run of 128][32], gate/up one a row
constexpr int kLdsBytes = kAtC + 4 * kRows * 4;
static_assert(kRows == 64 && kRows * kRowC * 4 <= kAtC && kLdsBytes <= 80 * 1024,
              "a lane per row; the epilogue leaves the scales alone; two workgroups share a CU");

// A tile of up to 16 MB rows by one slab.  Wave w multiplies all rows by its 64 weight rows, four operands of 16: lane (c, kg) holds eight
// elements of row c of operand j.  Gate/up: operands 0 and 1 are columns 32 w .. of gate, 2 and 3 of up; down: operand j is columns 4 c + j, so
// that a lane's results are four neighbours.
template <bool GATE_UP, int MB, bool OUT_H>
__device__ inline void q4k_tile(const Q4kArgs &p, int e, int p0, int rows, int slab, uint8_t *s_lds) {
    constexpr bool ROW = GATE_UP;   // one scale per row, applied at the end: a fold takes a whole super-block; else 128 elements
    const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6), c = lane & 15, kg = lane >> 4;
    const uint32_t row_bytes = (uint32_t)(p.in_dim / 256) * 144u;
    const uint32_t lds0 = lds_offset(s_lds);
    const int n_steps = p.in_dim / 64, n_sb = p.in_dim / 256;

    // weights: row r of the wave's 64 in LDS (16 j + c) has its 64 code bytes of a half super-block as pieces q at q ^ (r / 4 % 4)
    const uint8_t *w_base[2];
    uint32_t w_off;
    {
        const uint8_t *m0 = p.w0 + (size_t)e * (size_t)p.out_dim * row_bytes;
        const uint8_t *m1 = (GATE_UP ? p.w1 : p.w0) + (size_t)e * (size_t)p.out_dim * row_bytes;
        const int first = GATE_UP ? slab * (kWCols / 2) + 32 * wave : slab * kWCols + 64 * wave;
        w_base[0] = uniform(m0 + (size_t)first * row_bytes);
        w_base[1] = uniform(m1 + (size_t)(first + (GATE_UP ? 0 : 2)) * row_bytes);
        w_off = (uint32_t)((GATE_UP ? 1 : 4) * (lane >> 2)) * row_bytes + 16u + (uint32_t)((lane & 3) ^ ((lane >> 4) & 3)) * 16u;
    }
    // one load each (past the end: the last again, never multiplied)
    auto load_w = [&](int half, int j) {
        const int h = half < 2 * n_sb ? half : 2 * n_sb - 1;
        load_to_lds16(lds0 + kAtW + (uint32_t)wave * kWaveW + 1024u * j,
                      w_base[j >> 1] + ((size_t)(h >> 1) * 144 + 64 * (size_t)(h & 1) + (size_t)((j & 1) * (GATE_UP ? 16 : 1)) * row_bytes), w_off);
    };
    auto load_header = [&](int sb) {
        const int l = again(lane), r = GATE_UP ? l & 31 : 4 * (l & 15) + (l >> 4 & 1);
        load_to_lds16(lds0 + kAtH + (uint32_t)((sb & 1) * kWaves + wave) * 1024u,
                      ((l >> 5) ? w_base[1] : w_base[0]) + ((size_t)(sb < n_sb ? sb : n_sb - 1) * 144 + (uint32_t)r * row_bytes));
    };
    // the rows of the tile (past its end its last: multiplied, never stored): lane r looks row r up.  (By way of LDS, like all the
    // others: the wait for an ordinary load would be one for the codes behind it as well.)
    const int my_row = lane < rows ? lane : rows - 1;
    const uint32_t at_rows = kAtS + (uint32_t)wave * 256u;
    if (GATE_UP) load_to_lds4(lds0 + at_rows, (const uint8_t *)(p.sorted + p0), (uint32_t)my_row * 4u);
#pragma unroll
    for (int j = 0; j < 4; j++) load_w(0, j);
    load_header(0);
    uint32_t my_source = (uint32_t)(p0 + my_row);
    if (GATE_UP) {
        asm volatile("s_waitcnt vmcnt(5)" ::: "memory");
        my_source = *(const uint32_t *)(s_lds + at_rows + lane * 4) / (uint32_t)p.k_slots;
    }
    auto source_row = [&](int r) { return (uint32_t)__shfl((int)my_source, r, 64); };
    // activations: load i of the 4 MB of a stage (MB to a wave: hi planes of waves 0 and 1, lo of 2 and 3) holds eight rows, eight
    // pieces of 16 bytes each; piece q of row r lies at q ^ (r / 2 % 8), so that sixteen lanes reading the same piece of
    // neighbouring rows meet all 64 banks
    uint32_t a_off[MB];
    const uint8_t *a_base = uniform((const uint8_t *)(wave & 2 ? p.a.lo : p.a.hi));
    const uint32_t a_to = lds0 + (uint32_t)((wave >> 1) * kPlane + (wave & 1) * (MB * 1024));
#pragma unroll
    for (int i = 0; i < MB; i++) {
        const int eight = MB * (wave & 1) + i;
        a_off[i] = source_row(8 * eight + (lane >> 3)) * (uint32_t)p.in_dim * 2u + (uint32_t)((lane & 7) ^ (lane >> 4) ^ (4 * (eight & 1))) * 16u;
    }
    // sums: a wave's load holds 32 rows, of 8 f32 a super-block (waves past the tile's rows load the last ones' again); scales:
    // two a super-block, or (gate/up) the row's
    const int f_wave = wave & 1;
    const uint32_t f_off = source_row(32 * f_wave + (lane >> 1)) * (uint32_t)(p.in_dim / 32) * 4u + (uint32_t)(lane & 1) * 16u;
    const uint32_t c_off = (ROW ? my_source : source_row(32 * f_wave + (lane & 31))) * (uint32_t)(p.in_dim / 128) * 4u + (ROW ? 0u : (uint32_t)(lane >> 5) * 4u);

    auto load_a = [&](int step, uint32_t slot, int i) {
        load_to_lds16(a_to + slot + 1024u * i, a_base + (size_t)(step < n_steps ? step : n_steps - 1) * 128, a_off[i]);
    };
    auto load_sums = [&](int sb) {
        load_to_lds16(lds0 + kAtF + (uint32_t)f_wave * 1024u, (const uint8_t *)p.a.ssum + (size_t)(sb < n_sb ? sb : n_sb - 1) * 32, f_off);
    };
    auto load_scales = [&](int sb) {
        load_to_lds4(lds0 + kAtC + (uint32_t)(sb & 1) * (kRows * 8) + (uint32_t)f_wave * 256u,
                     (const uint8_t *)p.a.scale + (size_t)(sb < n_sb ? sb : n_sb - 1) * 8, c_off);
    };
    constexpr int kLoadsA = MB, kLoadsW = 4, kLoadsH = ROW ? 2 : 3;

    // sums of super-block sb as pairs of halfs: a thread takes four of a row (threads past them the same as others)
    auto split_sums = [&](int sb) {
        const int t = again(tid) & (2 * kRows - 1);
        const float4 v = *(const float4 *)(s_lds + kAtF + t * 16);
        const float f[4] = {v.x, v.y, v.z, v.w};
        half4v hi, lo;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            hi[j] = (_Float16)f[j];
            lo[j] = (_Float16)__fsub_rn(f[j], (float)hi[j]);
        }
        uint8_t *to = s_lds + kAtS + (uint32_t)(sb & 1) * (kRows * 32) + (t >> 1) * 32 + (t & 1) * (ROW ? 8 : 16);
        *(half4v *)to = hi;
        *(half4v *)(to + (ROW ? 16 : 8)) = lo;
    };

    const f32x4 zero = {0, 0, 0, 0};
    f32x4 acc[4][MB], c1[4][MB];
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
        for (int m = 0; m < MB; m++) acc[j][m] = c1[j][m] = zero;

    uint32_t sc4[4][2];   // of the super-block, by sub-blocks: the scales
    uint2 raw[2][4];   // of the half super-block: [step][operand], elements 8 kg .. of either sub-block
    half8 ah[MB], al[MB], bf[2];
    half2v mul[4];   // of the step: of the low, the high codes
    // (piece 4 half + kg of a row)
    const uint32_t a_rd = (uint32_t)c * 128u + (uint32_t)(kg ^ (c >> 1 & 7)) * 16u;
    auto read_hi = [&](uint32_t slot, int half, int m) { ah[m] = *(const half8 *)(s_lds + (a_rd ^ (uint32_t)(half * 64)) + slot + m * 2048); };
    auto read_lo = [&](uint32_t slot, int half, int m) { al[m] = *(const half8 *)(s_lds + (a_rd ^ (uint32_t)(half * 64)) + slot + kPlane + m * 2048); };
    const uint32_t w_rd = kAtW + (uint32_t)wave * kWaveW + (uint32_t)c * 64u + (uint32_t)((kg >> 1) ^ ((c >> 2) & 3)) * 16u + (uint32_t)(kg & 1) * 8u;
    auto read_w = [&]() {
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) raw[i][j] = *(const uint2 *)(s_lds + (w_rd ^ (uint32_t)(i * 32)) + j * 1024);
    };
    auto read_head = [&](int sb, int j) { return *(const u32x4 *)(s_lds + kAtH + (uint32_t)((sb & 1) * kWaves + wave) * 1024u + j * 256 + c * 16); };
    auto scales_of = [&](u32x4 hd, int j) {
        Q4kHeader h;
        h.unpack(hd);
        sc4[j][0] = h.sc4[0], sc4[j][1] = h.sc4[1];
    };
    auto scales = [&](int st, int j) { mul[j] = Q4kHeader::pair(sc4[j][st >> 1], st & 1) * half2v{(_Float16)1024.0f, (_Float16)64.0f}; };
    // operand g % 4 of step st's low (g < 4) or high codes
    auto decode = [&](int st, int g) {
        const uint2 w = raw[st & 1][g & 3];
        const half2v mu = mul[g & 3];
        bf[g & 1] = g < 4 ? q4k_operand<false>(w.x, w.y, half2v{mu[0], mu[0]}) : q4k_operand<true>(w.x, w.y, half2v{mu[1], mu[1]});
    };
    // what has been summed into c1 of operand j -> acc.  part: which 128 elements of super-block sb (all of it with one scale per row)
    half4v bm[2];   // of operand j: [j % 2]
    float fd[2], fm[2];
    half4v am[MB];   // the rows' sums
    float4 sr[2];    // (down) their scales: [m % 2]
    auto fold_begin = [&](u32x4 hd, int part, int j) {
        Q4kHeader h;
        h.unpack(hd);
        if (ROW) h.mn4[0] = kg & 1 ? h.mn4[1] : h.mn4[0];
        bm[j & 1] = h.offsets(ROW ? 0 : part);
        fd[j & 1] = h.d(), fm[j & 1] = h.minus_dmin();
    };
    auto read_sums = [&](int sb, int part) {
#pragma unroll
        for (int m = 0; m < MB; m++) {
            uint2 s2 = *(const uint2 *)(s_lds + kAtS + (uint32_t)(sb & 1) * (kRows * 32) + (16 * m + c) * 32 + (ROW ? 8 * kg : 16 * part + 8 * (kg & 1)));
            if (!ROW && kg >= 2) s2.x = s2.y = 0u;   // (K = 8 of the instruction's 16)
            __builtin_memcpy(&am[m], &s2, 8);
        }
    };
    auto read_row_scales = [&](int sb, int part, int m) {
        if (!ROW) sr[m & 1] = *(const float4 *)(s_lds + kAtC + (uint32_t)(sb & 1) * (kRows * 8) + (m >> 1) * 256 + part * 128 + (16 * (m & 1) + 4 * kg) * 4);
    };
    auto fold = [&](int j, int m) {
        const f32x4 c2 = __builtin_amdgcn_mfma_f32_16x16x16f16(am[m], bm[j & 1], zero, 0, 0, 0);
        const float f[4] = {sr[m & 1].x, sr[m & 1].y, sr[m & 1].z, sr[m & 1].w};
#pragma unroll
        for (int r = 0; r < 4; r++) {
            if constexpr (ROW) acc[j][m][r] = fmaf(fm[j & 1], c2[r], fmaf(fd[j & 1], c1[j][m][r], acc[j][m][r]));
            else acc[j][m][r] = fmaf(fmaf(fm[j & 1], c2[r], __fmul_rn(fd[j & 1], c1[j][m][r])), f[r], acc[j][m][r]);
        }
    };

    // prologue (the codes and headers are under way)
#pragma unroll
    for (int i = 0; i < kLoadsA; i++) load_a(0, 0, i);
    load_sums(0);
    if (ROW) load_to_lds4(lds0 + kAtC, (const uint8_t *)p.a.scale, c_off);   // (64 rows' worth from each wave, the same)
    else load_scales(0);
#pragma unroll
    for (int i = 0; i < kLoadsA; i++) load_a(1, kSlotA, i);
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kLoadsA) : "memory");
    split_sums(0);
#pragma unroll
    for (int j = 0; j < 4; j++) {
        scales_of(read_head(0, j), j);
        scales(0, j);
    }
    read_w();
    decode(0, 0);
#pragma unroll
    for (int m = 0; m < MB; m++) {
        read_hi(0, 0, m);
        read_lo(0, 0, m);
    }
    // (the first step begins by folding nothing)
    bm[1] = half4v{(_Float16)0.0f, (_Float16)0.0f, (_Float16)0.0f, (_Float16)0.0f};
    fd[1] = fm[1] = 0.0f;
#pragma unroll
    for (int m = 0; m < MB; m++) am[m] = bm[1];
    read_row_scales(0, 0, 0);
    uint32_t slot = 0, free_slot = 2 * kSlotA;   // of this step's activations; of those two steps on

    // What a step asks for, a few loads beside each group of products: the activations of two steps on; in even steps the codes
    // of the next half super-block (this one's are in registers: read behind the last barrier, waited for in front of the load); in
    // a super-block's second step the next one's header, sums and scales (everybody has folded the one before, whose scales' place
    // they take).
    constexpr int kLoads[4] = {kLoadsA + kLoadsW, kLoadsA + kLoadsH, kLoadsA + kLoadsW, kLoadsA};
    auto step = [&](int sb, auto st_c) {
        constexpr int st = decltype(st_c)::value;
        constexpr bool begins = ROW ? st == 0 : (st & 1) == 0, ends = ROW ? st == 3 : (st & 1) == 1;   // this step starts, ends a sum
        const int s = 4 * sb + st;
        const uint32_t next_slot = slot == 2 * kSlotA ? 0u : slot + kSlotA;
        // Group g: operand g % 4 of the low (g < 4) or high codes by all rows, lo and hi (1000 rows x 8 8.98e-8 off the 64-bit result, hi and lo
        // 9.10e-8, 32x32x16 9.04e-8).  Beside its products: the next group's operand; of an
        // operand's last ones what the fold takes of its header, the next step's scales (and super-block's header); then, beside the next
        // group's, the fold.
#pragma unroll
        for (int g = 0; g < 8; g++) {
            const int j = g & 3;
            if (g == 0) {
#pragma unroll
                for (int i = 0; i < kLoadsA; i++) load_a(s + 2, free_slot, i);
                if (st == 3) split_sums(sb + 1);
            }
            if (g == 1 && (st & 1) == 0) {
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
                for (int i = 0; i < kLoadsW; i++) load_w(2 * sb + (st >> 1) + 1, i);
            }
            if (g == 4 && st == 1) {
                load_header(sb + 1);
                load_sums(sb + 1);
                if (!ROW) load_scales(sb + 1);
            }
            if (g == 7) {
                // the next step's activations have landed, and this one's have been read by everybody
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kLoads[st]) : "memory");
                if (st & 1) read_w();
            }
            u32x4 hd, next_hd;
            if (g > 3 && ends) hd = read_head(sb, j);
            if (g > 3 && st == 3) next_hd = read_head(sb + 1, j);
            if (g == 4 && ends) read_sums(sb, st >> 1);
            // (operand 3's of the sum before: in the first step)
            const bool folds = g == 0 ? begins : (ends && g > 4);
            const int fold_sb = g > 0 || st > 0 ? sb : (sb > 0 ? sb - 1 : 0), fold_part = g > 0 ? st >> 1 : (st >> 1) ^ 1;
#pragma unroll
            for (int m = 0; m < MB; m++) {
                if (folds) {
                    if (m + 1 < MB) read_row_scales(fold_sb, fold_part, m + 1);
                    fold((j + 3) & 3, m);
                }
                c1[j][m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[m], bf[g & 1], begins && g < 4 ? zero : c1[j][m], 0, 0, 0);
                if (g == 3) read_lo(slot, 1, m);
                if (g == 7) read_lo(next_slot, 0, m);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (ends && g > 3) {
                fold_begin(hd, st >> 1, j);
                read_row_scales(sb, st >> 1, 0);
            }
            if (g < 7) decode(st, g + 1);
            if (g > 3) {
                if (st == 3) scales_of(next_hd, j);
                scales((st + 1) & 3, j);
            }
            if (g == 7) decode((st + 1) & 3, 0);
#pragma unroll
            for (int m = 0; m < MB; m++) {
                c1[j][m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[m], bf[g & 1], c1[j][m], 0, 0, 0);
                if (g == 3) read_hi(slot, 1, m);
                if (g == 7) read_hi(next_slot, 0, m);
            }
#pragma unroll
            for (int m = 0; m < MB; m++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 16 / MB, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        free_slot = slot;
        slot = next_slot;
    };
    for (int sb = 0; sb < n_sb; sb++) {
        step(sb, std::integral_constant<int, 0>{});
        step(sb, std::integral_constant<int, 1>{});
        step(sb, std::integral_constant<int, 2>{});
        step(sb, std::integral_constant<int, 3>{});
    }
#pragma unroll
    for (int m = 0; m < MB; m++) {
        if (m + 1 < MB) read_row_scales(n_sb - 1, 1, m + 1);
        fold(3, m);
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");   // (no load into LDS is under way any more)

    // element r of an accumulator: row 4 kg + r, column lane % 16
    if (GATE_UP) {
        // silu(g) * u as f32 over the stages, then in the form the down product reads
        float *s_c = (float *)s_lds;
#pragma unroll
        for (int m = 0; m < MB; m++) {
            const int row = 16 * m + 4 * kg;
            const float4 s4 = *(const float4 *)(s_lds + kAtC + row * 4);
            const float sr[4] = {s4.x, s4.y, s4.z, s4.w};
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int i = 0; i < 4; i++)
                    s_c[(row + i) * kRowC + 32 * wave + 16 * j + c] = __fmul_rn(silu_of(__fmul_rn(sr[i], acc[j][m][i])), __fmul_rn(sr[i], acc[j + 2][m][i]));
        }
        __syncthreads();
        // (eight rows at once by the four waves, two passes side by side)
        if constexpr (OUT_H) {
#pragma unroll 2
            for (int pass = 0; pass < 2 * MB; pass++) {
                const int row = 8 * pass + (tid >> 5);
                const float4 v = *(const float4 *)&s_c[row * kRowC + 4 * (tid & 31)];
                const bool active = row < rows;
                hact_store128(active ? v : make_float4(0.f, 0.f, 0.f, 0.f), active, p.act_h, (size_t)(p0 + row), p.out_dim, slab * 128 + 4 * (tid & 31));
            }
        } else {
            const int l16 = tid & 15;
#pragma unroll 2
            for (int pass = 0; pass < 2 * MB; pass++) {
                const int task = 16 * pass + (tid >> 4), row = task >> 1, cb = task & 1;
                const float4 v = *(const float4 *)&s_c[row * kRowC + cb * 64 + 4 * l16];
                const bool active = row < rows;
                quantize_store64(active ? v : make_float4(0.f, 0.f, 0.f, 0.f), active, p.act_q, (size_t)(p0 + row), p.out_dim,
                                 slab * 128 + cb * 64 + 4 * l16);
            }
        }
    } else {
#pragma unroll
        for (int m = 0; m < MB; m++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int row = 16 * m + 4 * kg + r;
                if (row >= rows) continue;
                *(float4 *)(p.y + (size_t)(p0 + row) * (size_t)p.out_dim + (size_t)(slab * kWCols + 64 * wave + 4 * c)) =
                    make_float4(acc[0][m][r], acc[1][m][r], acc[2][m][r], acc[3][m][r]);
            }
    }
}

template <bool GATE_UP, bool OUT_H>
__global__ __launch_bounds__(64 * kWaves, 2) void q4k_gemm_kernel(Q4kArgs p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t s_lds[];
    // As xcd_tile in gemm.hip: an XCD takes neighbouring tiles with the slab running fastest.
    constexpr int kCols = GATE_UP ? kWCols / 2 : kWCols;
    const int n_slabs = p.out_dim / kCols;   // (whole: grouped_gemm_q4k_f16)
    const int total = *p.n_tiles, per_xcd = (total + 7) >> 3;
    const int item = (int)(blockIdx.x >> 3);
    const int within = item / n_slabs, slab = item - within * n_slabs;
    const int tile = (int)(blockIdx.x & 7) * per_xcd + within;
    if (within >= per_xcd || tile >= total) return;
    const int e = uniform(p.tiles[3 * tile]), p0 = uniform(p.tiles[3 * tile + 1]), rows = uniform(p.tiles[3 * tile + 2]);
    switch ((rows + 15) / 16) {
    case 1: q4k_tile<GATE_UP, 1, OUT_H>(p, e, p0, rows, slab, s_lds); break;
    case 2: q4k_tile<GATE_UP, 2, OUT_H>(p, e, p0, rows, slab, s_lds); break;
    case 3: q4k_tile<GATE_UP, 3, OUT_H>(p, e, p0, rows, slab, s_lds); break;
    default: q4k_tile<GATE_UP, 4, OUT_H>(p, e, p0, rows, slab, s_lds); break;
    }
}

template <bool GATE_UP, bool OUT_H>
hipError_t launch_q4k(const Q4kArgs &p, int max_tiles, hipStream_t s) {
    constexpr int kCols = GATE_UP ? kWCols / 2 : kWCols;
    const dim3 grid((unsigned)(max_tiles + 7) / 8 * 8 * (unsigned)(p.out_dim / kCols));
    launch_kernel(q4k_gemm_kernel<GATE_UP, OUT_H>, grid, dim3(64 * kWaves), kLdsBytes, s, p);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_q4k_gate_up(const ExpertBanks &b, HAct x, const int32_t *sorted, int k_slots, const int32_t *tiles, const int32_t *n_tiles,
                              int max_tiles, HAct act_h, QAct64 act_q, hipStream_t s) {
    const Q4kArgs p{b.gate, b.up, x, sorted, tiles, n_tiles, k_slots, b.hidden, b.inter, act_h, act_q, nullptr};
    return act_h.hi != nullptr ? launch_q4k<true, true>(p, max_tiles, s) : launch_q4k<true, false>(p, max_tiles, s);
}

hipError_t launch_q4k_down(const ExpertBanks &b, HAct act, const int32_t *tiles, const int32_t *n_tiles, int max_tiles, float *y, hipStream_t s) {
    const Q4kArgs p{b.down, nullptr, act, nullptr, tiles, n_tiles, 1, b.inter, b.hidden, HAct(), QAct64(), y};
    return launch_q4k<false, true>(p, max_tiles, s);
}

}  // namespace mummu
