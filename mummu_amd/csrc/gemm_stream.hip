// Grouped GEMM of Q4_K banks, and down products of Q6_K, on the f16 units for a few rows per expert: the operands and arithmetic of gemm_q4k.hip
// and gemm_q6k.hip on tiles of up to 8 or 16 rows (v_mfma_f32_16x16x32_f16).  A wave keeps ONE super-block of K of the tile's rows in registers and takes the weights of 16 columns
// after 16 of it from memory straight into the registers that multiply them; the waves of a workgroup have the super-blocks of a row side by
// side, so that together they read whole rows front to back, and their sums meet in LDS in ascending order.  Tiles of 8 rows hold the high
// halfs in the operand's first eight rows and the low ones in the others: one product where 16 rows take two.
//
// What bounds it: the vector ALUs and the stream, neither wholly beside the other.  Every line of the weights is fetched once (128 experts of 2048 x 768, 27
// tokens: 177 MB where the 144-byte pieces of gemm_q4k_few.hip fetch 1.38 times that), 16 columns of a super-block take 108 vector
// instructions (two for a pair of codes; down 122) and nine products, and a CU's 16 to 20 waves keep 75 to 110 KB on the way.  Gate/up of that shape, here and
// in gemm_q4k_few.hip, 48 and 51 us, of 512 experts of 2560 x 640 with 64 tokens 152 and 176, with the loads alone 43 and 133, with the weights out of L2
// 45 and 139; OLMoE, 20 tokens, 37.2 + 20.9 and 38.7 + 23.5.  Layers among others, tiles of 8 rows here and of 16: 128 experts 27 tokens 69 and 73, 512 experts
// 64 tokens 263 and 286, OLMoE 54 and 57; 512 experts of 2048 x 768, 60 tokens 209 and 230, 128 of 3072 x 768, 30 tokens 110 and 123.
//
// Q6_K downs (tiles of 8 rows): a sub-block's 16 elements are an operand's K of 16 (v_mfma_f32_16x16x16_f16), four to a lane, so that its sum can
// be folded with d * sc; a lane loads 16 neighbouring bytes, in whole dwords, and changes dwords with the three others of its row.  Some 280 vector
// instructions a unit.  OLMoE, 24 tokens 42 -> 32 us (106 MB fetched, the weights' bytes; 35 with loads at odd halves of a dword), layers at 16 / 24 /
// 32 tokens 76 / 77 / 78 (tiles of 16 rows, q6k_down_kernel) and 62 / 64 / 65, 128 experts of 2048 x 768, 30 tokens 100 and 83.
#include "device_utils.h"
#include "kernels.h"
#include "q4k_half.h"
#include "qact.h"

namespace mummu {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kUnits = 4;            // 16 columns of one matrix each: between two meetings of the sums
constexpr int kRowC = 128 + 4;       // f32 row of the gate/up epilogue

// a / b for 0 <= a < 2^31, 1 <= b < 2^15 by the f32 quotient, one off at most up to 2^23 (else the integer one)
__device__ inline int div_small(int a, int b) {
    if (a >= (1 << 23)) return a / b;
    int q = (int)__fmul_rn((float)a, __builtin_amdgcn_rcpf((float)b));
    const int r = a - q * b;
    return r < 0 ? q - 1 : r >= b ? q + 1 : q;
}

struct StreamArgs {
    Q4kArgs q;
    int cols;        // columns of a workgroup
    int n_sb;        // waves along K
    int group_bits;  // 2^group_bits such rows of waves
};

template <bool R8>
constexpr size_t stream_lds(int waves, bool gate_up) {
    const int rows = R8 ? 8 : 16;
    return (size_t)2 * kUnits * (size_t)waves * (size_t)rows * 64 + 64 + (gate_up ? (size_t)rows * kRowC * 4 : 0);
}

// Workgroup: one wave to a super-block of K, times n_groups of them side by side where a row has one or two; group g of a step has columns
// 16 (step n_groups + g) .. + 15 of the workgroup's.
template <int WT, bool GATE_UP, bool OUT_H, bool R8, int MAXW, int PER_SIMD, int DEPTH>
__global__ __launch_bounds__(64 * MAXW, PER_SIMD) void stream_kernel(StreamArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t s_lds[];
    const Q4kArgs &p = a.q;
    constexpr bool Q6 = WT == T_Q6_K;
    static_assert(WT == T_Q4_K || (Q6 && !GATE_UP), "banks this kernel reads");
    constexpr int kBlock = block_bytes(WT);
    constexpr int kRows = R8 ? 8 : 16, kTile = kRows * 16, NB = GATE_UP ? 2 : 1, kSteps = kUnits / NB;
    // As xcd_tile in gemm.hip: an XCD takes neighbouring tiles with the slab running fastest.
    const int n_slabs = p.out_dim / a.cols;
    const int total = *p.n_tiles, per_xcd = (total + 7) >> 3;
    const int item = (int)(blockIdx.x >> 3);
    const int within = item / n_slabs, slab = item - within * n_slabs;
    const int tile = (int)(blockIdx.x & 7) * per_xcd + within;
    if (within >= per_xcd || tile >= total) return;
    const int e = uniform(p.tiles[3 * tile]), p0 = uniform(p.tiles[3 * tile + 1]), rows = uniform(p.tiles[3 * tile + 2]);

    const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6), c = lane & 15, kg = lane >> 4;
    const int n_sb = a.n_sb, n_groups = 1 << a.group_bits, n_waves = n_sb << a.group_bits;
    const int group = wave / n_sb, sb = wave - group * n_sb;
    const uint32_t row_bytes = (uint32_t)n_sb * kBlock;
    float *s_sum = (float *)s_lds;                                      // [2][unit][wave][kTile]
    float *s_scale = s_sum + 2 * kUnits * n_waves * kTile;              // [16]
    float *s_c = s_scale + 16;

    // the row that this lane multiplies (rows past the last repeat it: multiplied, never stored)
    const int my = R8 ? (c & 7) : c, my_row = my < rows ? my : rows - 1;
    int source = p0 + my_row;
    if (GATE_UP) source = p.sorted[p0 + my_row];

    // weights: 64 neighbouring bytes of a super-block's codes by the four lanes of a row, twice, and its header
    const size_t matrix = (size_t)e * (size_t)p.out_dim * row_bytes;
    const int col0 = slab * a.cols + 16 * group, n_steps = a.cols / (16 * n_groups);
    typedef __attribute__((address_space(1))) const uint8_t Global;   // (an address put together from scalars would be a flat one)
    Global *base[NB];
    base[0] = (Global *)uniform(p.w0 + matrix + (size_t)col0 * row_bytes);
    if (GATE_UP) base[NB - 1] = (Global *)uniform(p.w1 + matrix + (size_t)col0 * row_bytes);
    // (a Q6_K super-block begins at an even byte: it is read by whole dwords, from `skip` bytes in front of it on - 16 bytes at an odd half of
    // a dword keep the address units busy for several times as long.  Steps are multiples of 4 bytes.)
    const uint32_t low = Q6 ? (uint32_t)(uint64_t)base[0] & 2u : 0u, begin = (uint32_t)c * row_bytes + (uint32_t)sb * kBlock + low, skip = Q6 ? begin & 2u : 0u;
    base[0] -= low;
    const uint32_t off_h = begin - skip, off_q = off_h + (Q6 ? 0u : 16u) + 16u * (uint32_t)kg;
    const uint32_t step_bytes = 16u * (uint32_t)n_groups * row_bytes;
    // (DEPTH - 1 units on their way.  Q4_K: header, codes; Q6_K: scales and d, ql, ql, qh)
    u32x4 hd[DEPTH], q0[DEPTH], q1[DEPTH], qh[Q6 ? DEPTH : 1];
    uint32_t more[Q6 ? DEPTH : 1][4];   // ... the dword behind each of the four
    auto load = [&](int step, int j, int to) {
        Global *from = base[j] + (size_t)((uint32_t)step * step_bytes);
        typedef __attribute__((address_space(1))) const u32x4 Words;
        if constexpr (Q6) {
            typedef u32x4 Loose __attribute__((aligned(4)));
            typedef __attribute__((address_space(1))) const Loose LooseWords;
            typedef __attribute__((address_space(1))) const uint32_t Word;
            q0[to] = *(LooseWords *)(from + off_q), more[to][0] = *(Word *)(from + off_q + 16);
            q1[to] = *(LooseWords *)(from + off_q + 64), more[to][1] = *(Word *)(from + off_q + 80);
            qh[to] = *(LooseWords *)(from + off_q + 128), more[to][2] = *(Word *)(from + off_q + 144);
            hd[to] = *(LooseWords *)(from + off_h + 192), more[to][3] = *(Word *)(from + off_h + 208);   // (up to two bytes behind it: kBankSlack)
        } else {
            hd[to] = *(Words *)(from + off_h);
            q0[to] = *(Words *)(from + off_q);
            q1[to] = *(Words *)(from + off_q + 64);
        }
    };
    MUMMU_CODE_FENCE();
#pragma unroll
    for (int u = 0; u < DEPTH - 1; u++) load(u / NB, u % NB, u);
    MUMMU_CODE_FENCE();
    if (GATE_UP) source = div_small(source, p.k_slots);

    // x.  Q4_K: piece i of a plane = 8 elements; load l, half h, nibble n of the codes above meet piece 4 (4 l + 2 (kg / 2) + n) + 2 (kg % 2) + h.
    // Q6_K: elements 4 kg .. + 3 of each sub-block of 16.
    constexpr int kPlanes = R8 ? 1 : 2;
    half8 x[kPlanes][Q6 ? 1 : 2][2][2];
    half4v x6[kPlanes][Q6 ? 16 : 1];
    {
        const uint32_t at = (uint32_t)(8 * (kg >> 1) + 2 * (kg & 1)) * 16u;
        const size_t row_at = ((size_t)source * (size_t)p.in_dim + (size_t)sb * 256) * 2;
#pragma unroll
        for (int pl = 0; pl < kPlanes; pl++) {
            const uint8_t *plane = (const uint8_t *)(R8 ? (c < 8 ? p.a.hi : p.a.lo) : (pl == 0 ? p.a.hi : p.a.lo)) + row_at;
            if constexpr (Q6) {
#pragma unroll
                for (int n = 0; n < 16; n++) x6[pl][n] = *(const half4v *)(plane + 32 * n + 8 * kg);
            } else {
#pragma unroll
                for (int l = 0; l < 2; l++)
#pragma unroll
                    for (int h = 0; h < 2; h++)
#pragma unroll
                        for (int n = 0; n < 2; n++) x[pl][l][h][n] = *(const half8 *)(plane + at + (uint32_t)((16 * l + 4 * n + h) * 16));
            }
        }
    }
    // sums of 32 elements as pairs of halfs: gate/up K = 16 (high of sub-blocks 0-3, 4-7, low of both), down K = 8 for either half
    half4v am[GATE_UP ? 1 : 2];
    constexpr int kOut = R8 && !Q6 ? 2 : 4;   // sums of a lane that are multiplied by the weights' scales
    float sr[GATE_UP ? 1 : 2][4];
    {
        // (of eight rows, those that the lane groups' first two sums are of once high and low halfs have met)
        const int of_row = R8 && !Q6 ? __shfl(source, 4 * ((c >> 2) & 1) + (c >> 3) + 2 * (c & 1), 64) : source;
        const float *ss = p.a.ssum + (size_t)of_row * (size_t)(p.in_dim / 32) + (size_t)sb * 8;
        const bool low = GATE_UP ? kg >= 2 : kg == 1, none = !GATE_UP && kg >= 2;
#pragma unroll
        for (int l = 0; !Q6 && l < (GATE_UP ? 1 : 2); l++) {
            const float4 v = *(const float4 *)(ss + (GATE_UP ? 4 * (kg & 1) : 4 * l));
            const float f[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const _Float16 hi = (_Float16)f[i], lo = (_Float16)__fsub_rn(f[i], (float)hi);
                am[l][i] = none ? (_Float16)0.0f : low ? lo : hi;
            }
        }
        if (GATE_UP) {
            if (wave == 0 && lane < kRows) s_scale[lane] = p.a.scale[(size_t)source * (size_t)(p.in_dim / 128)];
        } else {
            // (element r of an accumulator: row 4 kg + r; of eight rows 4 (kg % 2) + r, or with high and low halfs summed 4 (kg % 2) + (kg / 2) + 2 r)
#pragma unroll
            for (int l = 0; l < 2; l++) {
                const float s = p.a.scale[(size_t)source * (size_t)(p.in_dim / 128) + (size_t)sb * 2 + l];
#pragma unroll
                for (int r = 0; r < kOut; r++) sr[l][r] = __shfl(s, !R8 ? 4 * kg + r : Q6 ? 4 * (kg & 1) + r : 4 * (kg & 1) + (kg >> 1) + 2 * r, 64);
            }
        }
    }

    const f32x4 zero = {0, 0, 0, 0};
    const uint32_t pick = kg >= 2 ? 0x04030402u : 0x04010400u;   // this lane's two sub-blocks of four
    auto products_q6 = [&](int b) {
        // dword kg of each 16 bytes: lane group i has loaded the 16 bytes i (and 4 + i) of ql, i of qh
        auto turn = [&](u32x4 &t) {
            auto swap = [](uint32_t &u, uint32_t &w, bool far) {
                const auto o = far ? __builtin_amdgcn_permlane32_swap(u, w, false, false) : __builtin_amdgcn_permlane16_swap(u, w, false, false);
                u = o[0], w = o[1];
            };
            uint32_t r[4] = {t[0], t[1], t[2], t[3]};
            swap(r[0], r[2], true), swap(r[1], r[3], true), swap(r[0], r[1], false), swap(r[2], r[3], false);
            t = u32x4{r[0], r[1], r[2], r[3]};
        };
        const uint32_t(&behind)[4] = more[Q6 ? b : 0];
        auto align = [&](u32x4 &t, uint32_t next) {
            const uint32_t r[5] = {t[0], t[1], t[2], t[3], next};
#pragma unroll
            for (int i = 0; i < 4; i++) t[i] = __builtin_amdgcn_alignbyte(r[i + 1], r[i], skip);
        };
        align(q0[b], behind[0]), align(q1[b], behind[1]), align(qh[Q6 ? b : 0], behind[2]), align(hd[b], behind[3]);
        turn(q0[b]), turn(q1[b]), turn(qh[Q6 ? b : 0]);
        const float d = half_bits_to_float((uint16_t)(behind[3] >> (8u * skip)));
        f32x4 v = zero;
#pragma unroll
        for (int half = 0; half < 2; half++) {
            f32x4 run = zero;
#pragma unroll
            for (int n = 0; n < 8; n++) {
                const int j = n >> 1, i = n & 1;
                const u32x4 ql = half == 0 ? q0[b] : q1[b];
                const uint32_t low = ql[2 * (j & 1) + i] >> (4 * (j >> 1)), high = qh[Q6 ? b : 0][2 * half + i];
                const uint32_t codes = (low & 0x0F0F0F0Fu) | ((j < 2 ? high << (4 - 2 * j) : high >> (2 * j - 4)) & 0x30303030u);
                const half2v f[2] = {q6k_code_pair(codes, 0x04020400u), q6k_code_pair(codes, 0x04030401u)};
                half4v w;
                __builtin_memcpy(&w, f, 8);
                f32x4 s = zero;
#pragma unroll
                for (int pl = 0; pl < kPlanes; pl++) s = __builtin_amdgcn_mfma_f32_16x16x16f16(x6[pl][Q6 ? 8 * half + n : 0], w, s, 0, 0, 0);
                const float fd = __fmul_rn(d, (float)(int8_t)(hd[b][2 * half + (n >> 2)] >> (8 * (n & 3))));
#pragma unroll
                for (int r = 0; r < 4; r++) run[r] = n == 0 ? __fmul_rn(fd, s[r]) : fmaf(fd, s[r], run[r]);
                if (n & 1) asm volatile("" : "+v"(run[0]), "+v"(run[1]), "+v"(run[2]), "+v"(run[3]));   // (summed here: the compiler would carry all sixteen sub-blocks' sums to the end)
            }
#pragma unroll
            for (int r = 0; r < 4; r++) v[r] = half == 0 ? __fmul_rn(run[r], sr[0][r]) : fmaf(run[r], sr[GATE_UP ? 0 : 1][r], v[r]);
        }
        return v;
    };
    auto products_q4 = [&](int b) {
        Q4kHeader head;
        head.unpack(hd[b]);
        f32x4 v = zero, c1 = zero;
#pragma unroll
        for (int l = 0; l < 2; l++) {
            const uint32_t t = __builtin_amdgcn_perm(0x64646464u, head.sc4[l], pick);
            half2v m;
            __builtin_memcpy(&m, &t, 4);
            m = (m - half2v{(_Float16)1024.0f, (_Float16)1024.0f}) * half2v{(_Float16)1024.0f, (_Float16)64.0f};
            const half2v ml = {m[0], m[0]}, mh = {m[1], m[1]};
            const u32x4 q = l == 0 ? q0[b] : q1[b];
            if (!GATE_UP) c1 = zero;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const half8 w[2] = {q4k_operand<false>(q[2 * h], q[2 * h + 1], ml), q4k_operand<true>(q[2 * h], q[2 * h + 1], mh)};
#pragma unroll
                for (int n = 0; n < 2; n++)
#pragma unroll
                    for (int pl = 0; pl < kPlanes; pl++) c1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[pl][Q6 ? 0 : l][h][n], w[n], c1, 0, 0, 0);
            }
            if (!GATE_UP || l == 1) {
                Q4kHeader h = head;
                if (GATE_UP) h.mn4[0] = kg & 1 ? h.mn4[1] : h.mn4[0];
                const f32x4 c2 = __builtin_amdgcn_mfma_f32_16x16x16f16(am[GATE_UP ? 0 : l], h.offsets(GATE_UP ? 0 : l), zero, 0, 0, 0);
                const float fd = head.d(), fm = head.minus_dmin();
                if constexpr (R8) {
                    // high + low in front of the scales, as on 16 rows: an infinite one (a damaged block) times either would make a NaN of them
                    c1[0] = swap32_add(c1[0], c1[1]), c1[1] = swap32_add(c1[2], c1[3]);
                }
#pragma unroll
                for (int r = 0; r < kOut; r++) {
                    const float t = fmaf(fm, c2[r], __fmul_rn(fd, c1[r]));
                    v[r] = GATE_UP ? t : l == 0 ? __fmul_rn(t, sr[0][r]) : fmaf(t, sr[GATE_UP ? 0 : 1][r], v[r]);
                }
            }
        }
        return v;
    };
    auto multiply = [&](int b, float *to) {
        f32x4 v;
        if constexpr (Q6) v = products_q6(b);
        else v = products_q4(b);
        if constexpr (R8) {
            // rows 4 (kg % 2) + (kg / 2), + 2 (Q6_K: high + low here, behind the scales: an infinite one times sixteen sums of either sign is a NaN anyhow)
            ((float2 *)to)[lane] = Q6 ? make_float2(swap32_add(v[0], v[1]), swap32_add(v[2], v[3])) : make_float2(v[0], v[1]);
        } else {
            ((f32x4 *)to)[lane] = v;
        }
    };

    const int n_phases = n_steps / kSteps;
    auto phase = [&](int ph, auto last) {
        float *sums = s_sum + (ph & 1) * kUnits * n_waves * kTile;
#pragma unroll
        for (int u = 0; u < kUnits; u++) {
            const int ahead = u + DEPTH - 1;
            if (!decltype(last)::value || ahead < kUnits) load(ph * kSteps + ahead / NB, ahead % NB, ahead % DEPTH);
            MUMMU_CODE_FENCE();
            multiply(u % DEPTH, sums + (u * n_waves + wave) * kTile);
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        const int n_out = kSteps * n_groups * kTile;
        // (the waves take turns where not all have some)
        int first = tid + (ph & 1) * 32 * n_waves;
        first -= first >= 64 * n_waves ? 64 * n_waves : 0;
        for (int i = first; i < n_out; i += 64 * n_waves) {
            const int block = i / kTile, d = i % kTile, ln = R8 ? d >> 1 : d >> 2, step = block >> a.group_bits, g = block & (n_groups - 1);
            const int row = R8 ? 4 * ((ln >> 4) & 1) + 2 * (d & 1) + (ln >> 5) : 4 * (ln >> 4) + (d & 3);
            auto sum_of = [&](int u) {
                const float *from = sums + (u * n_waves + g * n_sb) * kTile + d;
                float s = 0.0f;
                auto add = [&](auto count) {
                    float v[decltype(count)::value];
#pragma unroll
                    for (int k = 0; k < decltype(count)::value; k++) v[k] = from[k * kTile];
#pragma unroll
                    for (int k = 0; k < decltype(count)::value; k++) s = __fadd_rn(s, v[k]);
                    from += decltype(count)::value * kTile;
                };
                for (int k = 8; k <= n_sb; k += 8) add(std::integral_constant<int, 8>());
                if (n_sb & 4) add(std::integral_constant<int, 4>());
                if (n_sb & 2) add(std::integral_constant<int, 2>());
                if (n_sb & 1) add(std::integral_constant<int, 1>());
                return s;
            };
            const int col = 16 * ((ph * kSteps + step) * n_groups + g) + (ln & 15);
            if constexpr (GATE_UP) {
                const float gate = __fmul_rn(s_scale[row], sum_of(2 * step)), up = __fmul_rn(s_scale[row], sum_of(2 * step + 1));
                s_c[row * kRowC + col] = __fmul_rn(silu_of(gate), up);
            } else {
                const float v = sum_of(step);
                if (row < rows) p.y[(size_t)(p0 + row) * (size_t)p.out_dim + (size_t)(slab * a.cols + col)] = v;
            }
        }
    };
    for (int ph = 0; ph < n_phases - 1; ph++) phase(ph, std::false_type());
    phase(n_phases - 1, std::true_type());

    if constexpr (GATE_UP) {
        // silu(g) * u in the form the down product reads
        __syncthreads();
        for (int i = tid; i < kRows * 32; i += 64 * n_waves) {
            if constexpr (OUT_H) {
                const int row = i >> 5, c32 = i & 31;
                const float4 v = *(const float4 *)&s_c[row * kRowC + 4 * c32];
                const bool active = row < rows;
                hact_store128(active ? v : make_float4(0.f, 0.f, 0.f, 0.f), active, p.act_h, (size_t)(p0 + row), p.out_dim, slab * 128 + 4 * c32);
            } else {
                const int row = i >> 5, cb = (i >> 4) & 1;
                const float4 v = *(const float4 *)&s_c[row * kRowC + cb * 64 + 4 * c];
                const bool active = row < rows;
                quantize_store64(active ? v : make_float4(0.f, 0.f, 0.f, 0.f), active, p.act_q, (size_t)(p0 + row), p.out_dim,
                                 slab * 128 + cb * 64 + 4 * c);
            }
        }
    }
}

template <int WT, bool GATE_UP, bool OUT_H, bool R8>
hipError_t launch_stream(const Q4kArgs &q, int max_tiles, hipStream_t s) {
    const int n_sb = q.in_dim / 256, group_bits = n_sb >= 3 ? 0 : n_sb == 2 ? 1 : 2, groups = 1 << group_bits, waves = n_sb * groups;
    StreamArgs a{q, 128, n_sb, group_bits};   // (gate/up: what a scale of its output covers; down: the more, the less often rows are read into registers)
    // (Q6_K: a unit takes twice as long, and half the columns leave four workgroups to a CU: 16 / 24 tokens 63.7 / 65.6 -> 61.9 / 64.6 us a layer)
    if (!GATE_UP) a.cols = WT != T_Q6_K && q.out_dim % (256 * groups) == 0 ? 256 * groups : q.out_dim % (128 * groups) == 0 ? 128 * groups : 64 * groups;
    if (n_sb < 1 || n_sb > kStreamBlocks || q.in_dim % 256 != 0 || q.out_dim % a.cols != 0) return hipErrorInvalidValue;
    const dim3 grid((unsigned)(max_tiles + 7) / 8 * 8 * (unsigned)(q.out_dim / a.cols)), block(64 * waves);
    const size_t lds = stream_lds<R8>(waves, GATE_UP);
    // (five waves a SIMD hold one workgroup more than four)
    const bool five = R8 && (waves <= 6 || waves == 9 || waves == 10);
    if constexpr (WT == T_Q6_K) launch_kernel(stream_kernel<WT, GATE_UP, OUT_H, R8, 16, 4, 2>, grid, block, lds, s, a);
    else if constexpr (!R8) launch_kernel(stream_kernel<WT, GATE_UP, OUT_H, R8, 16, 4, 2>, grid, block, lds, s, a);
    else if (five) launch_kernel(stream_kernel<WT, GATE_UP, OUT_H, R8, 10, 5, 2>, grid, block, lds, s, a);
    else launch_kernel(stream_kernel<WT, GATE_UP, OUT_H, R8, 16, 4, 4>, grid, block, lds, s, a);
    return hipGetLastError();
}

}  // namespace

// Tiles of 16 rows keep 64 registers of rows, four waves a SIMD.  us a layer among others, here / gemm_q4k_few.hip: OLMoE (eight and four super-blocks) 24 / 64
// tokens 57.7 / 58.8, 61.8 / 64.2, 512 experts of 2048 x 768, 40 / 128 tokens 177 / 189, 302 / 316.  Ten super-blocks (hidden 2560) 365 / 349, sixteen (4096) 283 /
// 280, with downs of 1024 elements, 24 / 60 tokens 64.1 / 63.9, 70.8 / 68.9, six 46.5 / 43.8, three alike.  One and two, whose workgroups have several rows of waves:
// behind for gate/up (hidden 512, inter 512, 32 / 100 tokens 21.6 / 18.4, 25.0 / 21.7; hidden 256, 100 tokens 34.5 / 31.6), ahead for downs behind long rows (512 experts of
// 2048 x 512, 64 tokens 155 / 166, of 2048 x 256 91 / 94), which the rule, the same for both products, leaves to gemm_q4k_few.hip.
bool gemm_stream_takes(int in_dim, int out_dim, int tile_rows) {
    const int n_sb = in_dim / 256;
    if (in_dim % 256 != 0 || out_dim % 128 != 0) return false;
    return tile_rows <= 8 ? n_sb <= kStreamBlocks : n_sb == 4 || n_sb == 8;
}

hipError_t launch_gemm_stream_gate_up(const ExpertBanks &b, HAct x, const int32_t *sorted, int k_slots, const int32_t *tiles, const int32_t *n_tiles,
                                     int max_tiles, int tile_rows, HAct act_h, QAct64 act_q, hipStream_t s) {
    const Q4kArgs p{b.gate, b.up, x, sorted, tiles, n_tiles, k_slots, b.hidden, b.inter, act_h, act_q, nullptr};
    if (tile_rows <= 8) return act_h.hi != nullptr ? launch_stream<T_Q4_K, true, true, true>(p, max_tiles, s) : launch_stream<T_Q4_K, true, false, true>(p, max_tiles, s);
    return act_h.hi != nullptr ? launch_stream<T_Q4_K, true, true, false>(p, max_tiles, s) : launch_stream<T_Q4_K, true, false, false>(p, max_tiles, s);
}

hipError_t launch_gemm_stream_down(const ExpertBanks &b, HAct act, const int32_t *tiles, const int32_t *n_tiles, int max_tiles, int tile_rows,
                                  float *y, hipStream_t s) {
    const Q4kArgs p{b.down, nullptr, act, nullptr, tiles, n_tiles, 1, b.inter, b.hidden, HAct(), QAct64(), y};
    if (b.down_type == T_Q6_K) return tile_rows <= 8 ? launch_stream<T_Q6_K, false, true, true>(p, max_tiles, s) : hipErrorInvalidValue;
    return tile_rows <= 8 ? launch_stream<T_Q4_K, false, true, true>(p, max_tiles, s) : launch_stream<T_Q4_K, false, true, false>(p, max_tiles, s);
}

}  // namespace mummu
