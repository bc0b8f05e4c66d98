// Grouped GEMM of Q4_K banks on the f16 units: rows as pairs of halfs (HAct), sc * q < 1024 as exact halfs, so that the matrix units
// sum x * (sc * q) over a whole super-block (down: 128 elements of it) before d and dmin are applied; the offset term is one
// more instruction per fold, the sums of the blocks (hi and lo halfs) against the m.  Tiles of up to 64 rows by 256 weight rows (128 of
// gate and 128 of up, or 256 of down).
//
// What bounds it: the vector ALUs' port, which a product of 32 cycles takes for about 11 (two waves of a SIMD, each a product and n
// independent instructions: 33 cycles a product up to n = 5, 4 n + 11 from there; one wave alone issues one every 8 cycles, so
// two it has to be).  A wave that holds 64 rows by 32 + 32 columns has 4.5 beside each product, half of them the expansion of the
// codes, and the epilogue a fifth again.  So:
//   - two workgroups of four waves to a CU (80 KB of LDS, 256 registers), which drift apart: one folds, ends or begins while the
//     other multiplies.  One of eight waves in step, with 128 rows by 512 columns and each code expanded once for all, was slower:
//     65 % more vector work meets in the same place (4096 rows x 8: gate/up 600 us against 561).
//   - everything from memory straight into LDS: activations two stages ahead of three, the codes a wave multiplies itself half a
//     super-block ahead, no register or vector instruction between.
//   - silu in 17 instructions instead of 60.
// With rows by way of registers and codes straight into them (the form before), OLMoE layers, us: 192 tokens 122 -> 113, 400: 169 ->
// 150, 600: 250 -> 231, 1000: 352 -> 302, 2000: 582 -> 507; 4096: gate/up 1135 -> 940 k cycles, down 750 -> 593, with the matrix units
// busy for 59 / 48 % of them (51 / 40) at the 1.7 GHz that the card then holds.
#include "device_utils.h"
#include "kernels.h"
#include "q4k_half.h"
#include "qact.h"

namespace mummu {

namespace {

constexpr int kWaves = 4, kWCols = 64 * kWaves;  // weight rows of a tile, 64 to a wave
constexpr int kWaveW = 64 * 64;                  // the codes of 128 elements, 64 bytes a row
constexpr int kRing = 3;                         // stages of 64 elements of the activations
constexpr int kRowC = 128 + 4;                   // f32 row of the gate/up epilogue

// Where things lie in LDS.
constexpr int kRows = kQ4kRows;
constexpr int kPlane = kRows * 128;               // a stage's half plane: 64 elements a row
constexpr int kSlotA = 2 * kPlane;                // hi, lo
constexpr int kAtW = kRing * kSlotA;              // codes: [wave][64 rows][64 bytes]
constexpr int kAtH = kAtW + kWaves * kWaveW;      // headers: [wave][64 rows][16 bytes]
constexpr int kAtF = kAtH + kWaves * 1024;        // sums of 32 elements of x / scale, as they come: [row][8] f32
constexpr int kAtS = kAtF + kRows * 32;           // ... as pairs of halfs, two super-blocks: [2][row][16]
constexpr int kAtC = kAtS + 2 * kRows * 32;       // scales: down [2][row / 32][run of 128][32], gate/up one a row
constexpr int kLdsBytes = kAtC + 4 * kRows * 4;
static_assert(kRows == 64 && kRows * kRowC * 4 <= kAtC && kLdsBytes <= 80 * 1024,
              "a lane per row; the epilogue leaves the scales alone; two workgroups share a CU");

// A tile of up to 32 MW rows by one slab.  Wave w multiplies all rows by its 64 weight rows: columns c and 32 + c of lane
// (c, g) (gate/up: column 32 w + c of gate and of up).
template <bool GATE_UP, int MW, bool OUT_H>
__device__ inline void q4k_tile(const Q4kArgs &p, int e, int p0, int rows, int slab, uint8_t *s_lds) {
    constexpr bool ROW = GATE_UP;   // one scale per row, applied at the end: a fold takes a whole super-block; else 128 elements
    const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6), c = lane & 31, g = lane >> 5;
    const uint32_t row_bytes = (uint32_t)(p.in_dim / 256) * 144u;
    const uint32_t lds0 = lds_offset(s_lds);
    const int n_steps = p.in_dim / 64, n_sb = p.in_dim / 256;

    // weights: row r of the wave's 64 has its 64 code bytes of a half super-block as pieces q at q ^ (r / 4 % 4)
    const uint8_t *w_base[2];
    uint32_t w_off[2];
    {
        const uint8_t *m0 = p.w0 + (size_t)e * (size_t)p.out_dim * row_bytes;
        const uint8_t *m1 = (GATE_UP ? p.w1 : p.w0) + (size_t)e * (size_t)p.out_dim * row_bytes;
        const int first = GATE_UP ? slab * (kWCols / 2) + 32 * wave : slab * kWCols + 64 * wave;
        w_base[0] = uniform(m0 + (size_t)first * row_bytes);
        w_base[1] = uniform(m1 + (size_t)(first + (GATE_UP ? 0 : 32)) * row_bytes);
        const uint32_t piece = (uint32_t)((lane & 3) ^ ((lane >> 4) & 3)) * 16u;
#pragma unroll
        for (int j = 0; j < 2; j++) w_off[j] = (uint32_t)(16 * j + (lane >> 2)) * row_bytes + 16u + piece;
    }
    // one load each (past the end: the last again, never multiplied)
    auto load_w = [&](int half, int j) {
        const int h = half < 2 * n_sb ? half : 2 * n_sb - 1;
        load_to_lds16(lds0 + kAtW + (uint32_t)wave * kWaveW + 1024u * j, w_base[j >> 1] + ((size_t)(h >> 1) * 144 + 64 * (size_t)(h & 1)), w_off[j & 1]);
    };
    auto load_header = [&](int sb) {
        const int l = again(lane);
        load_to_lds16(lds0 + kAtH + (uint32_t)wave * 1024u,
                      ((l >> 5) ? w_base[1] : w_base[0]) + ((size_t)(sb < n_sb ? sb : n_sb - 1) * 144 + (uint32_t)(l & 31) * row_bytes));
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
    // activations: load i of the 8 MW of a stage (2 MW to a wave: hi planes of waves 0 and 1, lo of 2 and 3) holds eight rows, eight
    // pieces of 16 bytes each; piece q of row r lies at q ^ (r % 8), so that eight lanes reading the same piece of
    // neighbouring rows meet all banks
    uint32_t a_off[2 * MW];
    const uint8_t *a_base = uniform((const uint8_t *)(wave & 2 ? p.a.lo : p.a.hi));
    const uint32_t a_to = lds0 + (uint32_t)((wave >> 1) * kPlane + (wave & 1) * (2 * MW * 1024));
#pragma unroll
    for (int i = 0; i < 2 * MW; i++)
        a_off[i] = source_row(8 * (2 * MW * (wave & 1) + i) + (lane >> 3)) * (uint32_t)p.in_dim * 2u + (uint32_t)((lane & 7) ^ (lane >> 3)) * 16u;
    // sums: a wave's load holds 32 rows, of 8 f32 a super-block (waves past the tile's rows load the last ones' again); scales:
    // two a super-block, or (gate/up) the row's
    const int f_wave = wave & 1;
    const uint32_t f_off = source_row(32 * f_wave + (lane >> 1)) * (uint32_t)(p.in_dim / 32) * 4u + (uint32_t)(lane & 1) * 16u;
    const uint32_t c_off = (ROW ? my_source : source_row(32 * f_wave + c)) * (uint32_t)(p.in_dim / 128) * 4u + (ROW ? 0u : (uint32_t)g * 4u);

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
    constexpr int kLoadsA = 2 * MW, kLoadsW = 4, kLoadsH = ROW ? 2 : 3;

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

    const float16v zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    float16v acc[2][MW], c1[2][MW];
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
        for (int m = 0; m < MW; m++) acc[b][m] = c1[b][m] = zero;

    Q4kHeader head[2];
    u32x4 raw[2][2];   // of the half super-block: [step][b]
    half8 ah[2][MW], al[2][MW], bf[2][2];
    half2v ml[2], mh[2];
    // (the piece of K group kk: 4 (kk / 2) + 2 g + kk % 2)
    const uint32_t a_rd = (uint32_t)c * 128u + (uint32_t)((2 * g) ^ (c & 7)) * 16u;
    auto read_a = [&](uint32_t slot, int kk) {
        const uint8_t *at = s_lds + (a_rd ^ (uint32_t)((kk >> 1) * 64 + (kk & 1) * 16)) + slot;
#pragma unroll
        for (int m = 0; m < MW; m++) {
            ah[kk & 1][m] = *(const half8 *)(at + m * 4096);
            al[kk & 1][m] = *(const half8 *)(at + kPlane + m * 4096);
        }
    };
    const uint32_t w_rd = kAtW + (uint32_t)wave * kWaveW + (uint32_t)c * 64u + (uint32_t)(g ^ ((c >> 2) & 3)) * 16u;
    auto read_w = [&]() {
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int b = 0; b < 2; b++) raw[i][b] = *(const u32x4 *)(s_lds + (w_rd ^ (uint32_t)(i * 32)) + b * 2048);
    };
    auto read_head = [&]() {
#pragma unroll
        for (int b = 0; b < 2; b++) head[b].unpack(*(const u32x4 *)(s_lds + kAtH + (uint32_t)wave * 1024u + b * 512 + c * 16));
    };
    auto scales = [&](int st) {
#pragma unroll
        for (int b = 0; b < 2; b++) {
            head[b].muls(st, ml[b], mh[b]);
        }
    };
    auto decode = [&](int st, int kk) {
#pragma unroll
        for (int b = 0; b < 2; b++) {
            const u32x4 w = raw[st & 1][b];
            const uint32_t w_a = (kk & 1) ? w[2] : w[0], w_b = (kk & 1) ? w[3] : w[1];
            bf[kk & 1][b] = kk < 2 ? q4k_operand<false>(w_a, w_b, ml[b]) : q4k_operand<true>(w_a, w_b, mh[b]);
        }
    };
    // what has been summed into c1 -> acc.  part: which 128 elements of super-block sb (all of it with one scale per row)
    float fd[2], fm[2];
    std::conditional_t<ROW, half8, half4v> bm[2];
    auto fold_begin = [&](int part) {
#pragma unroll
        for (int b = 0; b < 2; b++) {
            fd[b] = head[b].d();
            fm[b] = head[b].minus_dmin();
            if constexpr (ROW) bm[b] = head[b].offsets();
            else bm[b] = head[b].offsets(part);
        }
    };
    auto fold = [&](int sb, int part) {
#pragma unroll
        for (int m = 0; m < MW; m++) {
            const uint8_t *at = s_lds + kAtS + (uint32_t)(sb & 1) * (kRows * 32) + (32 * m + c) * 32;
#pragma unroll
            for (int b = 0; b < 2; b++) {
                float16v c2;
                if constexpr (ROW) c2 = __builtin_amdgcn_mfma_f32_32x32x16_f16(*(const half8 *)(at + 16 * g), bm[b], zero, 0, 0, 0);
                else {
                    c2 = __builtin_amdgcn_mfma_f32_32x32x8f16(*(const half4v *)(at + 16 * part + 8 * g), bm[b], zero, 0, 0, 0);
                }
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    float sr[4];
                    if constexpr (!ROW) {
                        const float4 s4 = *(const float4 *)(s_lds + kAtC + (uint32_t)(sb & 1) * (kRows * 8) + m * 256 + part * 128 + (8 * j + 4 * g) * 4);
                        sr[0] = s4.x, sr[1] = s4.y, sr[2] = s4.z, sr[3] = s4.w;
                    }
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const int r = 4 * j + i;
                        if constexpr (ROW) acc[b][m][r] = fmaf(fm[b], c2[r], fmaf(fd[b], c1[b][m][r], acc[b][m][r]));
                        else acc[b][m][r] = fmaf(fmaf(fm[b], c2[r], __fmul_rn(fd[b], c1[b][m][r])), sr[i], acc[b][m][r]);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);   // (one at a time: together they do not fit the registers)
            }
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
    read_head();
    read_w();
    scales(0);
    decode(0, 0);
    read_a(0, 0);
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
#pragma unroll
        for (int kk = 0; kk < 4; kk++) {
            if (kk == 1 && (st & 1) == 0) {
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
                for (int j = 0; j < kLoadsW; j++) load_w(2 * sb + (st >> 1) + 1, j);
            }
            if (kk == 0) {
#pragma unroll
                for (int i = 0; i < kLoadsA; i++) load_a(s + 2, free_slot, i);
            }
            if (kk == 2 && st == 1) {
                load_header(sb + 1);
                load_sums(sb + 1);
                if (!ROW) load_scales(sb + 1);
            }
            if (ends && kk == 2) fold_begin(st >> 1);
            if (kk == 3) {
                // the next step's activations have landed, and this one's have been read by everybody
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kLoads[st]) : "memory");
                if (st == 3) read_head();
                if (st & 1) read_w();
                scales((st + 1) & 3);
            }
            if (kk == 0 && st == 3) split_sums(sb + 1);
            read_a(kk == 3 ? next_slot : slot, (kk + 1) & 3);
            if (kk < 3) decode(st, kk + 1);
            constexpr int NB = 2;
#pragma unroll
            for (int m = 0; m < MW; m++)
#pragma unroll
                for (int b = 0; b < NB; b++)
                    c1[b][m] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[kk & 1][m], bf[kk & 1][b], begins && kk == 0 ? zero : c1[b][m], 0, 0, 0);
#pragma unroll
            for (int m = 0; m < MW; m++)
#pragma unroll
                for (int b = 0; b < NB; b++) c1[b][m] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[kk & 1][m], bf[kk & 1][b], c1[b][m], 0, 0, 0);
            if (kk == 3) decode((st + 1) & 3, 0);
#pragma unroll
            for (int i = 0; i < 4 * MW; i++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, MW == 1 ? 8 : 4, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        free_slot = slot;
        slot = next_slot;
    };
    for (int sb = 0; sb < n_sb; sb++) {
        step(sb, std::integral_constant<int, 0>{});
        step(sb, std::integral_constant<int, 1>{});
        if (!ROW) fold(sb, 0);
        step(sb, std::integral_constant<int, 2>{});
        step(sb, std::integral_constant<int, 3>{});
        fold(sb, ROW ? 0 : 1);
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");   // (no load into LDS is under way any more)

    // element r of an accumulator: row 8 (r / 4) + 4 g + r % 4, column lane % 32
    if (GATE_UP) {
        // silu(g) * u as f32 over the stages, then in the form the down product reads
        float *s_c = (float *)s_lds;
#pragma unroll
        for (int m = 0; m < MW; m++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int row = 32 * m + 8 * j + 4 * g;
                const float4 s4 = *(const float4 *)(s_lds + kAtC + row * 4);
                const float sr[4] = {s4.x, s4.y, s4.z, s4.w};
#pragma unroll
                for (int i = 0; i < 4; i++)
                    s_c[(row + i) * kRowC + 32 * wave + c] =
                        __fmul_rn(silu_of(__fmul_rn(sr[i], acc[0][m][4 * j + i])), __fmul_rn(sr[i], acc[1][m][4 * j + i]));
            }
        __syncthreads();
        // (eight rows at once by the four waves, two passes side by side)
        if constexpr (OUT_H) {
#pragma unroll 2
            for (int pass = 0; pass < 4 * MW; pass++) {
                const int row = 8 * pass + (tid >> 5);
                const float4 v = *(const float4 *)&s_c[row * kRowC + 4 * c];
                const bool active = row < rows;
                hact_store128(active ? v : make_float4(0.f, 0.f, 0.f, 0.f), active, p.act_h, (size_t)(p0 + row), p.out_dim, slab * 128 + 4 * c);
            }
        } else {
            const int l16 = tid & 15;
#pragma unroll 2
            for (int pass = 0; pass < 4 * MW; pass++) {
                const int task = 16 * pass + (tid >> 4), row = task >> 1, cb = task & 1;
                const float4 v = *(const float4 *)&s_c[row * kRowC + cb * 64 + 4 * l16];
                const bool active = row < rows;
                quantize_store64(active ? v : make_float4(0.f, 0.f, 0.f, 0.f), active, p.act_q, (size_t)(p0 + row), p.out_dim,
                                 slab * 128 + cb * 64 + 4 * l16);
            }
        }
    } else {
#pragma unroll
        for (int m = 0; m < MW; m++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int row = 32 * m + 8 * (r >> 2) + 4 * g + (r & 3);
                if (row >= rows) continue;
                float *to = p.y + (size_t)(p0 + row) * (size_t)p.out_dim + (size_t)(slab * kWCols + 64 * wave + c);
                to[0] = acc[0][m][r];
                to[32] = acc[1][m][r];
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
    if (rows <= 32) q4k_tile<GATE_UP, 1, OUT_H>(p, e, p0, rows, slab, s_lds);
    else q4k_tile<GATE_UP, 2, OUT_H>(p, e, p0, rows, slab, s_lds);
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
