// Grouped GEMM of Q4_K banks on the f16 units for few rows per expert: the operands and arithmetic of gemm_q4k.hip on tiles of up to 16
// rows (v_mfma_f32_16x16x32_f16) by 256 weight rows, 64 to a wave.
//
// What bounds it: the stream of the weights past the L2.  Thousands of rows are read side by side, each in pieces that end inside a line
// of 128 bytes, and lines leave the L2 (4 MB for an XCD's 128 KB and more of rows in flight per CU) before their second piece is
// asked for.  512-expert shape, 64 tokens, gate/up, 682 MB of weights: a piece of 64 bytes at a time by four workgroups to a CU 1266 MB and
// 214 us, by two 840 MB and 206 (too little in flight), straight into registers (the form before) 871 MB and 200; a whole super-block
// of 144 at a time 940 MB and 173 us, 5.4 TB/s.  So a stage is a super-block, of the activations too: its weights go from LDS into
// registers as soon as they are there, the next ones into the same place, and there is one barrier to 256 elements.
// 128 experts of 2048 x 768, 27 tokens: gate/up 60.8 -> 50.6 us; layers, 27 / 128 tokens 116 -> 107, 139 -> 127; OLMoE 48 tokens 79.6 -> 76.3;
// the 512-expert shape, 64 tokens 360 -> 331.
#include "device_utils.h"
#include "kernels.h"
#include "q4k_half.h"
#include "qact.h"

namespace mummu {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kWaves = 4, kWCols = 64 * kWaves;  // weight rows of a tile
constexpr int kBlock = 144;                      // bytes of a super-block, in memory and in LDS
constexpr int kLoadsW = 64 * kBlock / 1024;      // loads of a wave's super-blocks
constexpr int kRowC = 128 + 4;                   // f32 row of the gate/up epilogue
constexpr int kRows = kQ4kFewRows;
// Where things lie in LDS.
constexpr int kPlane = kRows * 512;               // a stage's half plane: 256 elements a row
constexpr int kSlotA = 2 * kPlane;                // hi, lo; two slots
constexpr int kAtW = 2 * kSlotA;                  // super-blocks: [wave][64 rows]
constexpr int kAtF = kAtW + kWaves * 64 * kBlock; // sums of 32 elements of x / scale, as they come: [wave][row][8] f32 (and again)
constexpr int kAtS = kAtF + kWaves * 1024;        // ... as pairs of halfs: [row][16]
constexpr int kAtC = kAtS + kRows * 32;           // scales: [wave]: down [run of 128][row], gate/up one a row (and again)
constexpr int kLdsBytes = kAtC + kWaves * 256;
static_assert(kRows == 16 && 64 * kBlock % 1024 == 0 && kRows * kRowC * 4 <= kAtC && kLdsBytes <= 80 * 1024,
              "whole loads; the epilogue leaves the scales alone; two workgroups share a CU");

// Wave w multiplies the rows by its 64 weight rows, four blocks of 16: column 16 j + c of lane (c, kg) (gate/up: blocks 0 and 1 columns
// 32 w .. + 31 of gate, 2 and 3 of up).
template <bool GATE_UP, bool OUT_H>
__device__ inline void q4k_few_tile(const Q4kArgs &p, int e, int p0, int rows, int slab, uint8_t *s_lds) {
    constexpr bool ROW = GATE_UP;   // one scale per row, applied at the end: a fold takes a whole super-block; else 128 elements
    const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6), c = lane & 15, kg = lane >> 4;
    const int n_sb = p.in_dim / 256;
    const uint32_t row_bytes = (uint32_t)n_sb * kBlock;
    const uint32_t lds0 = lds_offset(s_lds);

    // the rows of the tile (past its end its last: multiplied, never stored): lane r looks row r % 16 up.  (By way of LDS, like all the
    // others: the wait for an ordinary load would be one for the weights behind it as well.)
    const int my_row = c < rows ? c : rows - 1;
    const uint32_t at_rows = kAtF + (uint32_t)wave * 1024u;
    if (GATE_UP) load_to_lds4(lds0 + at_rows, (const uint8_t *)(p.sorted + p0), (uint32_t)my_row * 4u);

    // weights: a wave's 64 rows of a super-block in nine loads, 144 neighbouring bytes a row (the fifth load ends the first 32
    // rows and begins the others, which for gate/up lie in the other matrix)
    const uint8_t *w_base[2];
    uint32_t w_off[kLoadsW];
    {
        const uint8_t *m0 = p.w0 + (size_t)e * (size_t)p.out_dim * row_bytes;
        const uint8_t *m1 = (GATE_UP ? p.w1 : p.w0) + (size_t)e * (size_t)p.out_dim * row_bytes;
        const int first = GATE_UP ? slab * (kWCols / 2) + 32 * wave : slab * kWCols + 64 * wave;
        w_base[0] = uniform(m0 + (size_t)first * row_bytes);
        w_base[1] = uniform(m1 + (size_t)(first + (GATE_UP ? 0 : 32)) * row_bytes);
#pragma unroll
        for (int j = 0; j < kLoadsW; j++) {
            const int piece = 64 * j + lane;
            w_off[j] = (uint32_t)((piece / 9) & 31) * row_bytes + (uint32_t)(piece % 9) * 16u;
        }
    }
    auto load_w = [&](int sb, int j) {
        const uint32_t to = lds0 + kAtW + (uint32_t)wave * (64 * kBlock) + 1024u * j;
        const size_t at = (size_t)(sb < n_sb ? sb : n_sb - 1) * kBlock;
        if (j == 4) load_to_lds16(to, (lane < 32 ? w_base[0] : w_base[1]) + (at + w_off[4]));
        else load_to_lds16(to, w_base[j > 4] + at, w_off[j]);
    };
#pragma unroll
    for (int j = 0; j < kLoadsW; j++) load_w(0, j);
    uint32_t my_source = (uint32_t)(p0 + my_row);
    if (GATE_UP) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kLoadsW) : "memory");
        my_source = *(const uint32_t *)(s_lds + at_rows + lane * 4) / (uint32_t)p.k_slots;
    }
    auto source_row = [&](int r) { return (uint32_t)__shfl((int)my_source, r, 64); };
    // activations: a load holds two rows of a plane, a wave loads eight (hi: waves 0 and 1, lo: 2 and 3); piece q of row r lies at
    // q ^ r: sixteen lanes reading the same piece of the rows meet all banks
    const uint8_t *a_base = uniform((const uint8_t *)(wave & 2 ? p.a.lo : p.a.hi));
    const uint32_t a_to = lds0 + (uint32_t)((wave >> 1) * kPlane + (wave & 1) * 4096);
    uint32_t a_off[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int r = 8 * (wave & 1) + 2 * i + (lane >> 5);
        a_off[i] = source_row(r) * (uint32_t)p.in_dim * 2u + (uint32_t)((lane & 31) ^ r) * 16u;
    }
    const uint32_t f_off = source_row((lane >> 1) & 15) * (uint32_t)(p.in_dim / 32) * 4u + (uint32_t)(lane & 1) * 16u;
    const uint32_t c_off = my_source * (uint32_t)(p.in_dim / 128) * 4u + (ROW ? 0u : (uint32_t)(kg & 1) * 4u);
    auto load_a = [&](int sb, int i) {
        load_to_lds16(a_to + (uint32_t)(sb & 1) * kSlotA + 1024u * i, a_base + (size_t)(sb < n_sb ? sb : n_sb - 1) * 512, a_off[i]);
    };
    auto load_sums = [&](int sb) {
        load_to_lds16(lds0 + kAtF + (uint32_t)wave * 1024u, (const uint8_t *)p.a.ssum + (size_t)(sb < n_sb ? sb : n_sb - 1) * 32, f_off);
    };
    auto load_scales = [&](int sb) {
        load_to_lds4(lds0 + kAtC + (uint32_t)wave * 256u, (const uint8_t *)p.a.scale + (size_t)(sb < n_sb ? sb : n_sb - 1) * 8, c_off);
    };

    const f32x4 zero = {0, 0, 0, 0};
    f32x4 acc[4], c1[4];
#pragma unroll
    for (int j = 0; j < 4; j++) acc[j] = c1[j] = zero;
    uint2 raw[4][4];                // [step][block]: elements 8 kg .. + 7 of either sub-block
    Q4kHeader head[4];
    const uint8_t *w_rd = s_lds + kAtW + wave * (64 * kBlock) + c * kBlock;
    const uint32_t a_rd = (uint32_t)c * 512u + (uint32_t)(kg ^ c) * 16u;

#pragma unroll
    for (int i = 0; i < 4; i++) load_a(0, i);
    load_sums(0);
    load_scales(0);
    for (int sb = 0; sb < n_sb; sb++) {
        // this super-block's loads have landed, and the one before has been multiplied by everybody
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        // its weights into registers, so that the next one's can take their place
#pragma unroll
        for (int j = 0; j < 4; j++) {
            head[j].unpack(*(const u32x4 *)(w_rd + j * 16 * kBlock));
#pragma unroll
            for (int st = 0; st < 4; st++) raw[st][j] = *(const uint2 *)(w_rd + j * 16 * kBlock + 16 + 32 * st + 8 * kg);
        }
        // sums as pairs of halfs (every wave all of them, for itself), scales
        {
            const float4 v = *(const float4 *)(s_lds + kAtF + wave * 1024 + lane * 16);
            const float f[4] = {v.x, v.y, v.z, v.w};
            half4v hi, lo;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                hi[j] = (_Float16)f[j];
                lo[j] = (_Float16)__fsub_rn(f[j], (float)hi[j]);
            }
            uint8_t *to = s_lds + kAtS + ((lane >> 1) & 15) * 32 + (lane & 1) * (ROW ? 8 : 16);
            *(half4v *)to = hi;
            *(half4v *)(to + (ROW ? 16 : 8)) = lo;
        }
        float sr[2][4];
        if constexpr (!ROW) {
#pragma unroll
            for (int part = 0; part < 2; part++) {
                const float4 s4 = *(const float4 *)(s_lds + kAtC + wave * 256 + part * 64 + kg * 16);
                sr[part][0] = s4.x, sr[part][1] = s4.y, sr[part][2] = s4.z, sr[part][3] = s4.w;
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        load_sums(sb + 1);
        if (!ROW) load_scales(sb + 1);
        const uint8_t *a_at = s_lds + (uint32_t)(sb & 1) * kSlotA;
#pragma unroll
        for (int st = 0; st < 4; st++) {
            // (the next one's, a few beside each step's products)
            if (st < 3) {
#pragma unroll
                for (int j = 3 * st; j < 3 * st + 3; j++) load_w(sb + 1, j);
            }
            load_a(sb + 1, st);
            half2v ml[4], mh[4];
#pragma unroll
            for (int j = 0; j < 4; j++) head[j].muls(st, ml[j], mh[j]);
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const uint8_t *at = a_at + (a_rd ^ (uint32_t)((8 * st + 4 * h) * 16));   // piece 8 st + 4 h + kg
                const half8 ah = *(const half8 *)at, al = *(const half8 *)(at + kPlane);
                const bool first = h == 0 && (ROW ? st == 0 : (st & 1) == 0);
                half8 w[4];
#pragma unroll
                for (int j = 0; j < 4; j++)
                    w[j] = h == 0 ? q4k_operand<false>(raw[st][j].x, raw[st][j].y, ml[j]) : q4k_operand<true>(raw[st][j].x, raw[st][j].y, mh[j]);
#pragma unroll
                for (int j = 0; j < 4; j++) c1[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, w[j], first ? zero : c1[j], 0, 0, 0);
#pragma unroll
                for (int j = 0; j < 4; j++) c1[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al, w[j], c1[j], 0, 0, 0);
            }
            if (ROW ? st == 3 : (st & 1) == 1) {
                // what has been summed into c1 -> acc: the super-block, or 128 elements of it
                const int part = ROW ? 0 : st >> 1;
                uint2 s2 = *(const uint2 *)(s_lds + kAtS + c * 32 + (ROW ? 8 * kg : 16 * part + 8 * (kg & 1)));
                if (!ROW && kg >= 2) s2.x = s2.y = 0u;   // (K = 8 of the instruction's 16)
                half4v am;
                __builtin_memcpy(&am, &s2, 8);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    Q4kHeader h = head[j];
                    if (ROW) h.mn4[0] = kg & 1 ? h.mn4[1] : h.mn4[0];
                    const f32x4 c2 = __builtin_amdgcn_mfma_f32_16x16x16f16(am, h.offsets(part), zero, 0, 0, 0);
                    const float fd = h.d(), fm = h.minus_dmin();
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        if constexpr (ROW) acc[j][r] = fmaf(fm, c2[r], fmaf(fd, c1[j][r], acc[j][r]));
                        else acc[j][r] = fmaf(fmaf(fm, c2[r], __fmul_rn(fd, c1[j][r])), sr[part][r], acc[j][r]);
                    }
                }
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");   // (no load into LDS is under way any more)

    // element r of an accumulator: row 4 kg + r, column c
    if (GATE_UP) {
        // silu(g) * u as f32 over the stages, then in the form the down product reads
        float *s_c = (float *)s_lds;
        const float4 s4 = *(const float4 *)(s_lds + kAtC + kg * 16);
        const float sr[4] = {s4.x, s4.y, s4.z, s4.w};
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                s_c[(4 * kg + r) * kRowC + 32 * wave + 16 * j + c] = __fmul_rn(silu_of(__fmul_rn(sr[r], acc[j][r])), __fmul_rn(sr[r], acc[j + 2][r]));
        __syncthreads();
        if constexpr (OUT_H) {
#pragma unroll
            for (int pass = 0; pass < 2; pass++) {
                const int row = 8 * pass + (tid >> 5), c32 = tid & 31;
                const float4 v = *(const float4 *)&s_c[row * kRowC + 4 * c32];
                const bool active = row < rows;
                hact_store128(active ? v : make_float4(0.f, 0.f, 0.f, 0.f), active, p.act_h, (size_t)(p0 + row), p.out_dim, slab * 128 + 4 * c32);
            }
        } else {
#pragma unroll
            for (int pass = 0; pass < 2; pass++) {
                const int task = 16 * pass + (tid >> 4), row = task >> 1, cb = task & 1;
                const float4 v = *(const float4 *)&s_c[row * kRowC + cb * 64 + 4 * c];
                const bool active = row < rows;
                quantize_store64(active ? v : make_float4(0.f, 0.f, 0.f, 0.f), active, p.act_q, (size_t)(p0 + row), p.out_dim,
                                 slab * 128 + cb * 64 + 4 * c);
            }
        }
    } else {
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                if (4 * kg + r < rows) p.y[(size_t)(p0 + 4 * kg + r) * (size_t)p.out_dim + (size_t)(slab * kWCols + 64 * wave + 16 * j + c)] = acc[j][r];
    }
}

template <bool GATE_UP, bool OUT_H>
__global__ __launch_bounds__(64 * kWaves, 2) void q4k_few_kernel(Q4kArgs p) {
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
    q4k_few_tile<GATE_UP, OUT_H>(p, e, p0, rows, slab, s_lds);
}

template <bool GATE_UP, bool OUT_H>
hipError_t launch_q4k_few(const Q4kArgs &p, int max_tiles, hipStream_t s) {
    constexpr int kCols = GATE_UP ? kWCols / 2 : kWCols;
    const dim3 grid((unsigned)(max_tiles + 7) / 8 * 8 * (unsigned)(p.out_dim / kCols));
    launch_kernel(q4k_few_kernel<GATE_UP, OUT_H>, grid, dim3(64 * kWaves), kLdsBytes, s, p);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_q4k_few_gate_up(const ExpertBanks &b, HAct x, const int32_t *sorted, int k_slots, const int32_t *tiles, const int32_t *n_tiles,
                              int max_tiles, HAct act_h, QAct64 act_q, hipStream_t s) {
    const Q4kArgs p{b.gate, b.up, x, sorted, tiles, n_tiles, k_slots, b.hidden, b.inter, act_h, act_q, nullptr};
    return act_h.hi != nullptr ? launch_q4k_few<true, true>(p, max_tiles, s) : launch_q4k_few<true, false>(p, max_tiles, s);
}

hipError_t launch_q4k_few_down(const ExpertBanks &b, HAct act, const int32_t *tiles, const int32_t *n_tiles, int max_tiles, float *y, hipStream_t s) {
    const Q4kArgs p{b.down, nullptr, act, nullptr, tiles, n_tiles, 1, b.inter, b.hidden, HAct(), QAct64(), y};
    return launch_q4k_few<false, true>(p, max_tiles, s);
}

}  // namespace mummu
