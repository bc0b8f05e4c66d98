// Grouped down product of Q6_K banks on the f16 units: rows as pairs of halfs (HAct), a code -32..31 is a half as it is, and a sub-block's 16
// products are summed by v_mfma_f32_32x32x16_f16 into one f32 accumulator, hi and lo halfs alike; what is left for the vector ALUs is one
// multiply-add per output and sub-block, with the scale d * sc, and one per 128 elements, with the row's.  (d * sc in the operand would
// take 13 bits, a half has 11.)
//
// What bounds it: those multiply-adds, 16 to a pair of products, and the codes' way into halfs, 17 for eight: the vector ALUs are busy for
// 57 % of the cycles and the matrix units, which they share the issue with, for 28 (OLMoE shape, 32768 rows).  The int8 form needs three
// times as many to put two int32 sums together.  Codes are turned into halfs for 64 rows at a time (MT 2), or 32 where experts have few.
//
// A super-block (210 bytes) comes as aligned pieces of 16 bytes, each wave's own 32 rows, and a half's rows two halves ahead.  There is
// LDS for one super-block a wave: its first half goes into registers when it has landed, the second beside the products of the first,
// and the next one's loads are dealt over the products of the second.  All of it into registers at once, on rows of 14 pieces: eight
// waves queued for an LDS whose banks four rows shared; 1.23M cycles for 0.99M.  A workgroup fills a CU and takes several items, its loads
// running on from one into the next (see gemm_q8.hip).
//
// OLMoE shape, int8 form -> this, us: 64 tokens 68 -> 44.5, 600: 193 -> 128, 4096: 699 -> 492 (layers, Q4_K gate and up: 125 -> 101, 331 ->
// 272, 1334 -> 1127; three streams 99 -> 81 a layer, 1000 tokens 384 -> 303, 1413 -> 1099).
#include <type_traits>

#include "device_utils.h"
#include "kernels.h"
#include "q4k_half.h"
#include "qact.h"

namespace mummu {

namespace {

constexpr int kWaves = 8, kCols = 32 * kWaves;   // weight rows of an item: 32 a wave, which it loads for itself
constexpr int kBlock = 210;                      // bytes of a super-block: ql, qh, scales, d
constexpr int kPieces = 15, kRowW = 16 * kPieces;   // aligned pieces of 16 bytes: 14 hold one (it begins at an even byte), 15 spread rows over the banks
constexpr int kWLoads = 8, kWaveW = 32 * kRowW;  // (the last by half its lanes)
constexpr int kCusOfXcd = 32;                    // (a workgroup fills a CU)
// in LDS: [kWaves][32 rows] super-blocks, [3] halves of activations [hi, lo][row][16 pieces of 16 bytes], [4][64] their scales
constexpr int kAtA = kWaves * kWaveW;
constexpr int slot_bytes(int mt) { return 2 * 32 * mt * 256; }
constexpr int at_scales(int mt) { return kAtA + 3 * slot_bytes(mt); }
constexpr int lds_bytes(int mt) { return at_scales(mt) + 4 * 256; }
static_assert(64 * kWLoads - 32 * kPieces == 32 && lds_bytes(2) <= 160 * 1024, "whole rows; fits");

// a in sorted order, a scale per 128 elements; y[pos, n] = f32 sum.  Tiles of up to 32 MT rows, or (MT 1) of up to 16, which are the first eight
// elements of an accumulator: the others are not folded (64 tokens, OLMoE shape: 44.0 -> 41.6 us).
template <int MT, bool HALF = false>
__global__ __launch_bounds__(64 * kWaves, 2) void q6k_down_kernel(const uint8_t *__restrict__ w, HAct a, const int32_t *__restrict__ tiles,
                                                                  const int32_t *__restrict__ n_tiles, int in_dim, int out_dim, float *__restrict__ y) {
    extern __shared__ __attribute__((aligned(16))) uint8_t s_lds[];
    constexpr int kSlotA = slot_bytes(MT), kPlane = kSlotA / 2, kAtS = at_scales(MT), kALoads = 2 * MT, ROWS = HALF ? 8 : 16;   // (elements of an accumulator that count)
    static_assert(!HALF || MT == 1, "tiles of 16 rows");
    // as xcd_tile in gemm.hip: an XCD takes neighbouring tiles, the slab running fastest; a workgroup takes every gridDim.x / 8 -th of its
    // XCD's items, and its loads run on from one into the next
    const int n_slabs = out_dim / kCols;   // (whole: grouped_gemm_q4k_f16)
    const int total = *n_tiles, per_xcd = (total + 7) >> 3, tile0 = (int)(blockIdx.x & 7) * per_xcd;
    const int n_items = n_slabs * (total - tile0 < per_xcd ? total - tile0 : per_xcd), apart = (int)(gridDim.x >> 3);
    const int first_item = (int)(blockIdx.x >> 3);
    if (first_item >= n_items) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6), c = lane & 31, g = lane >> 5;
    const int n_sb = in_dim / 256, n_halves = 2 * n_sb;
    const uint32_t row_bytes = (uint32_t)n_sb * kBlock;
    const uint32_t lds0 = lds_offset(s_lds);
    auto tile_of = [&](int item, int i) { return uniform(tiles[3 * (tile0 + item / n_slabs) + i]); };

    // Where the loads stand: an item and its super-block, for the weights (one ahead of the products), and its half, for the rows (two
    // ahead).  Past the last item they stay at its last, never multiplied.
    int w_item = first_item, w_sb = 0, a_item = first_item, a_half = 0;
    const uint8_t *w_base = nullptr;
    uint32_t w_off[kWLoads], a_off[kALoads], s_off = 0;
    auto set_w = [&]() {
        const int first = w_item % n_slabs * kCols + 32 * wave;
        w_base = uniform(w + (size_t)tile_of(w_item, 0) * (size_t)out_dim * row_bytes);
        const int at_lane = again(lane);
#pragma unroll
        for (int j = 0; j < kWLoads; j++) {
            const int p = 64 * j + at_lane < 32 * kPieces ? 64 * j + at_lane : 0, col = first + p / kPieces;
            w_off[j] = (uint32_t)col * row_bytes + (uint32_t)(p % kPieces) * 16u;
        }
    };
    // Activation pieces: a load holds four rows of a plane, waves 0-3 load hi, 4-7 lo.  Piece q of row r lies at q ^ (r % 16): sixteen lanes
    // that read the same piece of neighbouring rows meet all banks.  (Rows past the tile's end repeat its last.)
    auto set_a = [&]() {
        const int p0 = tile_of(a_item, 1), rows = tile_of(a_item, 2), at_lane = again(lane);
#pragma unroll
        for (int i = 0; i < kALoads; i++) {
            const int r = 4 * ((wave & 3) * kALoads + i) + (at_lane >> 4);
            a_off[i] = (uint32_t)(p0 + (r < rows ? r : rows - 1)) * (uint32_t)in_dim * 2u + (uint32_t)((at_lane & 15) ^ (r & 15)) * 16u;
        }
        s_off = (uint32_t)(p0 + (at_lane < rows ? at_lane : rows - 1)) * (uint32_t)(in_dim / 128) * 4u;
    };
    auto next_w = [&]() {
        if (++w_sb < n_sb) return;
        if (w_item + apart < n_items) {
            w_item += apart, w_sb = 0;
            set_w();
        } else {
            w_sb = n_sb - 1;
        }
    };
    auto next_a = [&]() {
        if (++a_half < n_halves) return;
        if (a_item + apart < n_items) {
            a_item += apart, a_half = 0;
            set_a();
        } else {
            a_half = n_halves - 1;
        }
    };
    auto load_w = [&](int j) {
        load_to_lds16_if(~0u, j == kWLoads - 1 ? 0u : ~0u, lds0 + (uint32_t)wave * kWaveW + 1024u * j, w_base, (w_off[j] + (uint32_t)w_sb * kBlock) & ~15u);
    };
    const uint8_t *a_plane = uniform((const uint8_t *)(wave >= 4 ? a.lo : a.hi));
    auto load_a = [&](int slot, int which, int i) {
        if (i > kALoads) return;
        if (i < kALoads)
            load_to_lds16(lds0 + kAtA + (uint32_t)(slot * kSlotA + (wave >> 2) * kPlane + ((wave & 3) * kALoads + i) * 1024), a_plane + (size_t)a_half * 256, a_off[i]);
        else
            load_to_lds4(lds0 + kAtS + (uint32_t)which * 256u, (const uint8_t *)a.scale + (size_t)a_half * 4, s_off);   // (every wave the same)
    };
    set_w();
    set_a();
#pragma unroll
    for (int j = 0; j < kWLoads; j++) load_w(j);
#pragma unroll
    for (int i = 0; i <= kALoads; i++) load_a(0, 0, i);
    next_a();
#pragma unroll
    for (int i = 0; i <= kALoads; i++) load_a(1, 1, i);

    const float16v zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    // the lane's part of a super-block's half: segments of 8 bytes, ql 0-3 (32 jl + 16 i), qh 4, 5 (16 i); of both halves the scales, d
    uint32_t q[2][6][2], sc[4];
    float d = 0.0f;
    const uint32_t my_row = (uint32_t)(32 * wave + c) * row_bytes;
    auto row_of = [&](int sb, uint32_t &skip) {   // (begins at an even byte: `skip` into a dword)
        const uint32_t o = (my_row + (uint32_t)sb * kBlock) & 15u;
        skip = o & 2u;
        return s_lds + wave * kWaveW + c * kRowW + (o & ~3u);
    };
    auto read_w = [&](int sb, int h, int s) {
        uint32_t skip;
        const uint8_t *from = row_of(sb, skip) + (s < 4 ? 64 * h + 32 * (s >> 1) + 16 * (s & 1) : 128 + 32 * h + 16 * (s & 1)) + 8 * g;
        const uint32_t d0 = *(const uint32_t *)from, d1 = *(const uint32_t *)(from + 4), d2 = *(const uint32_t *)(from + 8);
        q[h][s][0] = __builtin_amdgcn_alignbyte(d1, d0, skip);
        q[h][s][1] = __builtin_amdgcn_alignbyte(d2, d1, skip);
        asm volatile("" : "+v"(q[h][s][0]), "+v"(q[h][s][1]));   // (aligned once)
    };
    auto read_scales = [&](int sb) {
        uint32_t skip;
        const uint8_t *row = row_of(sb, skip);
        auto dword = [&](int at) { return *(const uint32_t *)(row + at); };
#pragma unroll
        for (int i = 0; i < 4; i++) sc[i] = __builtin_amdgcn_alignbyte(dword(196 + 4 * i), dword(192 + 4 * i), skip);
        d = half_bits_to_float((uint16_t)(dword(208) >> (8u * skip)));
    };
    // Products go by units u = MT n + m: sub-block n of the half (elements 16 n .. + 15), rows 32 m .. + 31.  While one is multiplied, the
    // next one's rows are read and the sums of the one before are folded.
    half8 hi[2], lo[2];
    auto read_a = [&](int slot, int u) {
        const int n = u / MT, m = u % MT;
        const uint8_t *as = s_lds + kAtA + (uint32_t)slot * kSlotA + (uint32_t)(32 * m + c) * 256u + (uint32_t)(((2 * n + g) ^ (c & 15)) * 16);
        hi[u & 1] = *(const half8 *)as;
        lo[u & 1] = *(const half8 *)(as + kPlane);
    };
    float16v acc[MT], run[MT], s[2];
    float fd[2] = {0.0f, 0.0f};   // d * scale of sub-block n: [n & 1]
    s[0] = s[1] = zero;
#pragma unroll
    for (int m = 0; m < MT; m++) acc[m] = run[m] = zero;
    auto fold = [&](int u) {   // a unit's sums -> the 128 elements' -> (with the rows' scales) acc
        const int n = u / MT, m = u % MT;
#pragma unroll
        for (int r = 0; r < ROWS; r++) run[m][r] = n == 0 ? __fmul_rn(fd[0], s[u & 1][r]) : fmaf(fd[n & 1], s[u & 1][r], run[m][r]);
    };
    auto fold_run = [&](int m, int which) {
#pragma unroll
            for (int j = 0; j < ROWS / 4; j++) {
                const float4 sr = *(const float4 *)(s_lds + kAtS + which * 256 + (32 * m + 8 * j + 4 * g) * 4);
                const float f[4] = {sr.x, sr.y, sr.z, sr.w};
#pragma unroll
                for (int i = 0; i < 4; i++) acc[m][4 * j + i] = fmaf(run[m][4 * j + i], f[i], acc[m][4 * j + i]);
            }
    };

    int slot = 0, which = 0;   // of the half's rows, of their scales
    *(float *)(s_lds + kAtS + 3 * 256 + lane * 4) = 0.0f;   // (an item begins by folding nothing)
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kALoads + 1) : "memory");
    read_a(0, 0);
    for (int item = first_item; item < n_items; item += apart) {
        auto half = [&](int sb, auto odd) {
            const int slot1 = slot == 2 ? 0 : slot + 1, slot2 = slot1 == 2 ? 0 : slot1 + 1;
            if (!odd) {
                read_scales(sb);
#pragma unroll
                for (int i = 0; i < 6; i++) read_w(sb, 0, i);
            } else {
                next_w();
            }
            next_a();
#pragma unroll
            for (int n = 0; n < 8; n++) {
                const int j = n >> 1, i = n & 1;
                // beside the others: the other half's weights and, when they are out of LDS, the next super-block's in their place; the
                // rows of the half after the next
                if (!odd && n < 6) read_w(sb, 1, n);
                if (!odd && n <= kALoads) load_a(slot2, (which + 2) & 3, n);
                if (odd && n < 4) load_w(2 * n), load_w(2 * n + 1);
                if (odd && n >= 4 && n < 7) load_a(slot2, (which + 2) & 3, 2 * n - 8), load_a(slot2, (which + 2) & 3, 2 * n - 7);
                half8 op;
                {
                    half2v f[4];
#pragma unroll
                    for (int p = 0; p < 2; p++) {
                        const uint32_t low = q[odd][2 * (j & 1) + i][p] >> (4 * (j >> 1)), high = q[odd][4 + i][p];
                        const uint32_t codes = (low & 0x0F0F0F0Fu) | ((j < 2 ? high << (4 - 2 * j) : high >> (2 * j - 4)) & 0x30303030u);
                        f[2 * p] = q6k_code_pair(codes, 0x04020400u);
                        f[2 * p + 1] = q6k_code_pair(codes, 0x04030401u);
                    }
                    __builtin_memcpy(&op, f, 16);
                }
                const uint32_t word = sc[2 * odd + (n >> 2)];
                const float f = __fmul_rn(d, (float)(int8_t)(word >> (8 * (n & 3))));
#pragma unroll
                for (int m = 0; m < MT; m++) {
                    const int u = MT * n + m;
                    // In front of a half's last products: the next half's rows are there (and after the odd one the next super-block), for
                    // this wave; then for everybody, who have also read this half's.
                    if (u == 8 * MT - 1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kALoads + 1) : "memory");
                    const half8 h = hi[u & 1], l = lo[u & 1];
                    if (u < 8 * MT - 1) read_a(slot, u + 1);
                    else read_a(slot1, 0);
                    s[u & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(h, op, zero, 0, 0, 0);
                    s[u & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(l, op, s[u & 1], 0, 0, 0);
                    fold((u + 8 * MT - 1) % (8 * MT));
                    if (u < MT) fold_run(u, (which + 3) & 3);   // (of the half before)
                    if (m == 0) fd[n & 1] = f;
                    __builtin_amdgcn_sched_barrier(0);   // (nothing further ahead: registers)
                }
            }
            // (summed here, not where the next half reads them: the compiler would carry all eight sub-blocks' sums there)
#pragma unroll
            for (int m = 0; m < MT; m++) asm volatile("" : "+v"(run[m]));
            slot = slot1;
            which = (which + 1) & 3;
        };
        for (int sb = 0; sb < n_sb; sb++) {
            half(sb, std::integral_constant<int, 0>());
            half(sb, std::integral_constant<int, 1>());
        }
        fold(8 * MT - 1);
#pragma unroll
        for (int m = 0; m < MT; m++) fold_run(m, (which + 3) & 3);
        // element r of an accumulator: row 8 (r / 4) + 4 g + r % 4, column lane % 32
        const int p0 = tile_of(item, 1), rows = tile_of(item, 2), col = item % n_slabs * kCols + 32 * wave + again(c), g4 = 4 * again(g);
        float *to = y + (size_t)(p0 + g4) * (size_t)out_dim + (size_t)col;
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
            for (int j = 0; j < ROWS / 4; j++) {
#pragma unroll
                for (int r = 0; r < 4; r++, to += out_dim)
                    if (32 * m + 8 * j + g4 + r < rows) *to = acc[m][4 * j + r];
                to += 4 * (size_t)out_dim;
            }
#pragma unroll
        for (int m = 0; m < MT; m++) acc[m] = run[m] = zero;
        s[1] = zero;
        fd[1] = 0.0f;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (no load into LDS is under way when the workgroup ends)
}

template <int MT, bool HALF>
hipError_t launch_q6k(const uint8_t *w, HAct a, const int32_t *tiles, const int32_t *n_tiles, int max_tiles, int in_dim, int out_dim, float *y,
                      hipStream_t s) {
    const int per_xcd = (max_tiles + 7) / 8 * (out_dim / kCols);
    const dim3 grid(8u * (unsigned)(per_xcd < kCusOfXcd ? per_xcd : kCusOfXcd));
    launch_kernel(q6k_down_kernel<MT, HALF>, grid, dim3(64 * kWaves), lds_bytes(MT), s, w, a, tiles, n_tiles, in_dim, out_dim, y);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_q6k_down(const ExpertBanks &b, HAct act, const int32_t *tiles, const int32_t *n_tiles, int max_tiles, int tile_rows, float *y,
                           hipStream_t s) {
    if (tile_rows > 32) return launch_q6k<2, false>(b.down, act, tiles, n_tiles, max_tiles, b.inter, b.hidden, y, s);
    if (tile_rows <= 16) return launch_q6k<1, true>(b.down, act, tiles, n_tiles, max_tiles, b.inter, b.hidden, y, s);
    return launch_q6k<1, false>(b.down, act, tiles, n_tiles, max_tiles, b.inter, b.hidden, y, s);
}

}  // namespace mummu
