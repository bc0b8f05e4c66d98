// Grouped GEMM of F16 and BF16 banks with wide tiles, for many rows per expert: the operands and arithmetic of
// grouped_gemm_f16_kernel (gemm.hip) - x and the activations between the two products as halfs, v_mfma_f32_32x32x16_f16,
// f32 accumulators - on tiles of up to 320 rows by 256 weight rows (128 of gate and 128 of up, or 256 of down).
//
// What bounds it and why it looks the way it does (OLMoE shape, 4096 tokens = 512 rows per expert):
//   - LDS reads.  A 64 x 128 tile reads one operand per matrix instruction, which keeps the LDS port (128 bytes a clock)
//     busy all the time at half the matrix rate.  Eight waves of 32 MW x 64 outputs (MW up to 5) read 7 operands for 10.
//   - The way into LDS.  Both tiles go from global memory straight into LDS, 64 elements of K (whole 128-byte lines: pieces
//     of 64 bytes come out of the L2 at half the rate, 17 against 34 TB/s) at a time, without registers in between, the weights two
//     stages ahead where the LDS holds them, and never a stage at once: 72 loads behind a barrier fill the address unit's queue, with
//     all eight waves waiting in front of it.  (Asked for in one go, one stage ahead: 4096 bf16 rows x 8 gate/up / down 620 / 416 k cycles
//     against 529 / 363, 1500 f16 rows 358 / 206 against 299 / 217.)
//   - Whole rounds.  An expert's rows are split evenly, in steps of 64, over as few tiles as hold them, so that the
//     workgroups of a launch are alike (full tiles and a remainder left a fifth of the launch to stragglers), and a wave
//     multiplies only as many row blocks as the tile has.
//   - Weights of bf16 become halfs beside the last products of the group before, not between their read and the next products.
// What remains: the matrix units are busy for 52 / 38 % of the cycles at 4096 bf16 rows x 8, and the card lowers its clock as they
// are: 15 % fewer cycles were 7 % of the time (340 / 206 us -> 316 / 194).
// OLMoE shape, grouped_gemm_f16_kernel -> the loads in one go -> now, 4096 bf16 rows x 8: gate/up 503 -> 340 -> 316 us, down 262 -> 206 -> 194 (a trace of
// it on its own; by events between launches 285 / 180, f16 270 / 174).
#include "device_utils.h"
#include "kernels.h"

namespace mummu {

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr int kWK = 64;                          // K elements of a stage: a line of 128 bytes per row, eight pieces of 16
constexpr int kWCols = 256;                      // weight rows of a tile
constexpr int kWStageB = kWCols * kWK * 2;       // bytes of a stage of weights
// Stages in LDS, for tiles of 64 MW rows: of the weights, then two of the activations.
template <int MW>
struct Ring {
    static constexpr int kB = MW <= 4 ? 3 : 2, kStageA = 64 * MW * kWK * 2, kAtA = kB * kWStageB;
    static_assert(kAtA + 2 * kStageA <= 160 * 1024, "the stages fit the LDS");
};
constexpr int kWLds = Ring<4>::kAtA + 2 * Ring<4>::kStageA;
static_assert(kWideRows == 64 * 5 && Ring<5>::kAtA + 2 * Ring<5>::kStageA <= kWLds, "... all of them");

template <int WT>
__device__ inline half8 weight_operand(u32x4 v) {
    half8 h;
    if constexpr (WT == T_F16) {
        __builtin_memcpy(&h, &v, 16);
    } else {
        // a bf16 is a half from 2^-14 up (8 significant bits); smaller weights keep an absolute error below 2^-25
#pragma unroll
        for (int i = 0; i < 4; i++) {
            h[2 * i] = (_Float16)__uint_as_float(v[i] << 16);
            h[2 * i + 1] = (_Float16)__uint_as_float(v[i] & 0xFFFF0000u);
        }
    }
    return h;
}

// x / (1 + e^-x) with the hardware's 2^y and reciprocal (1 ulp each): y = -x log2 e is split into its rounded value and
// what rounding it lost, so that the exponential is good to an ulp or two for every x; about twelve instructions where
// det_silu has sixty, which were a fifth of a gate/up tile's time.  The exponent stops at +-87, where e^-x and its
// reciprocal are both normal numbers: beyond it inf - inf and inf * 0 would give NaN.  Above 87 the quotient is x as it is, below
// -87 it stays under 2e-38 |x|, which no gate of half operands makes large enough to leave the half's zero.  A gate of -inf
// (a row with an element beyond the halfs) is NaN as in det_silu and the reference: -inf * 0.
__device__ inline float fast_silu(float x) {
    const float c = __builtin_amdgcn_fmed3f(x, -87.0f, 87.0f);
    const float y = __fmul_rn(c, -1.44269504f);
    const float lost = __builtin_fmaf(c, -1.44269504f, -y);
    float t = __builtin_amdgcn_exp2f(y);
    t = __builtin_fmaf(t, __fmul_rn(lost, 0.693147181f), t);
    return x == -__builtin_inff() ? __builtin_nanf("") : __fmul_rn(x, __builtin_amdgcn_rcpf(__fadd_rn(1.0f, t)));
}

struct WideArgs {
    const uint8_t *w0, *w1;        // gate and up, or down [experts][out_dim][in_dim]
    const _Float16 *a;             // rows of in_dim halfs: tokens (gate/up, through sorted / k_slots) or sorted positions
    const int32_t *sorted, *tiles, *n_tiles;
    int k_slots, in_dim, out_dim;
    _Float16 *act;                 // gate/up: silu(g) * u, sorted positions
    float *y;                      // down
};

// What a wave moves of a stage: rows 8 mw wave .. of the activation tile (8 to a load: a lane per 16-byte piece) and
// rows 32 wave .. of the weight tile.  Row r of a tile holds its eight pieces in the order q ^ (r % 8): eight lanes that
// read the same piece of neighbouring rows then meet all 64 banks.
template <int MW>
struct Loader {
    uint32_t a_off[MW], b_off[4];
    const uint8_t *a_base, *b_base;

    __device__ void load_a(uint32_t at, int step, int wave, int i) const {
        load_to_lds16(at + (uint32_t)(8 * MW * wave + 8 * i) * (kWK * 2), a_base + (size_t)step * (kWK * 2), a_off[i]);
    }
    __device__ void load_b(uint32_t at, int step, int wave, int i) const {
        load_to_lds16(at + (uint32_t)(32 * wave + 8 * i) * (kWK * 2), b_base + (size_t)step * (kWK * 2), b_off[i]);
    }
};

// A tile of up to 64 MW rows by one slab; wave (wm, wn) multiplies rows 32 MW wm .. by its 64 weight rows.
template <bool GATE_UP, int WT, int MW>
__device__ inline void wide_tile(const WideArgs &p, int e, int p0, int rows, int slab, uint8_t *s_lds) {
    using R = Ring<MW>;
    const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
    const int wm = wave >> 2, wn = wave & 3, g = lane >> 5, lr = lane & 31;
    const uint32_t row_bytes = (uint32_t)p.in_dim * 2u;
    const uint32_t lds0 = lds_offset(s_lds);
    const int n_steps = p.in_dim / kWK;

    Loader<MW> l;
    {
        const int lrow = lane >> 3;
        const uint32_t piece = (uint32_t)((lane & 7) ^ lrow) * 16u;
        l.a_base = (const uint8_t *)p.a;
#pragma unroll
        for (int i = 0; i < MW; i++) {
            const int r = 8 * MW * wave + 8 * i + lrow;
            const int rr = r < rows ? r : rows - 1;   // (rows past the tile's end repeat its last: multiplied, never stored)
            l.a_off[i] = (uint32_t)(GATE_UP ? p.sorted[p0 + rr] / p.k_slots : p0 + rr) * row_bytes + piece;
        }
        // weight rows: gate/up: 32 rows of gate, then 32 of up for each pair of waves; down: 64 rows for each pair
        const int col0 = GATE_UP ? slab * (kWCols / 2) + 32 * (wave >> 1) : slab * kWCols + 32 * wave;
        l.b_base = uniform((GATE_UP && (wave & 1) ? p.w1 : p.w0) + (size_t)e * (size_t)p.out_dim * row_bytes);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int col = col0 + 8 * i + lrow < p.out_dim ? col0 + 8 * i + lrow : p.out_dim - 1;
            l.b_off[i] = (uint32_t)col * row_bytes + piece;
        }
    }

    float16v acc[2][MW];
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
        for (int m = 0; m < MW; m++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[b][m][r] = 0.0f;
    uint32_t q[4];
#pragma unroll
    for (int kk = 0; kk < 4; kk++) q[kk] = (uint32_t)((2 * kk + g) ^ (lr & 7)) * 16u;
    const uint8_t *a_rd = s_lds + R::kAtA + (32 * MW * wm + lr) * (kWK * 2), *b_rd = s_lds + (64 * wn + lr) * (kWK * 2);
    // operands of 16 elements of K, read while the ones before are multiplied
    half8 ra[2][MW], rb[2][2];
    u32x4 raw[2];
    auto read = [&](uint32_t at_a, uint32_t at_b, int kk) {
#pragma unroll
        for (int j = 0; j < 2; j++) raw[j] = *(const u32x4 *)(b_rd + (at_b + q[kk]) + 32 * (kWK * 2) * j);
#pragma unroll
        for (int m = 0; m < MW; m++) ra[kk & 1][m] = *(const half8 *)(a_rd + (at_a + q[kk]) + 32 * (kWK * 2) * m);
    };
    auto convert = [&](int kk) {
#pragma unroll
        for (int j = 0; j < 2; j++) rb[kk & 1][j] = weight_operand<WT>(raw[j]);
    };
    // row block m's two products of group kk
    auto multiply = [&](int kk, int m) {
#pragma unroll
        for (int j = 0; j < 2; j++) acc[j][m] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ra[kk & 1][m], rb[kk & 1][j], acc[j][m], 0, 0, 0);
    };
    // Behind the barrier of a step, beside its last products, the rows of the step after the next are asked for; beside the first
    // products after that the weights of one step more (tiles of more than 256 rows leave no room for that: of the same step).  All at once
    // they fill the address unit's queue, and every wave stands before it.  Past the end: the last again, never multiplied.
    constexpr int kAhead = R::kB == 3 ? 2 : 1;
    const uint32_t lds_a = lds0 + R::kAtA;
    auto at_most = [&](int step) { return step < n_steps ? step : n_steps - 1; };
#pragma unroll
    for (int i = 0; i < 4; i++) l.load_b(lds0, 0, wave, i);
#pragma unroll
    for (int i = 0; i < MW; i++) l.load_a(lds_a, 0, wave, i);
    if (kAhead == 2) {
#pragma unroll
        for (int i = 0; i < 4; i++) l.load_b(lds0 + kWStageB, 1, wave, i);
    }
#pragma unroll
    for (int i = 0; i < MW; i++) l.load_a(lds_a + R::kStageA, 1, wave, i);
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(MW + (kAhead == 2 ? 4 : 0)) : "memory");
    read(0, 0, 0);
    convert(0);
    uint32_t at_b = 0, free_b = kAhead * kWStageB;   // of this step's weights; of those kAhead on
    for (int step = 0; step < n_steps; step++) {
        const uint32_t at_a = (uint32_t)(step & 1) * R::kStageA, next_a = R::kStageA - at_a;
        const uint32_t next_b = at_b == (R::kB - 1) * kWStageB ? 0u : at_b + kWStageB;
#pragma unroll
        for (int kk = 0; kk < 4; kk++) {
            // the next stage has landed and this one has been read by everybody
            if (kk == 3) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kAhead == 2 ? 4 : 0) : "memory");
            read(kk == 3 ? next_a : at_a, kk == 3 ? next_b : at_b, (kk + 1) & 3);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int m = 0; m < MW; m++) {
                multiply(kk, m);
                if (kk == 3) l.load_a(lds_a + at_a, at_most(step + 2), wave, m);
                if (kk == 0) {
#pragma unroll
                    for (int i = m; i < 4; i += MW) l.load_b(lds0 + free_b, at_most(step + kAhead), wave, i);
                }
                if (m == MW - 1) convert((kk + 1) & 3);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        free_b = at_b;
        at_b = next_b;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (no load into LDS is under way when the workgroup ends)

    // element r of an accumulator: row 8 (r / 4) + 4 g + r % 4, column lane % 32
#pragma unroll
    for (int j = 0; j < (GATE_UP ? 1 : 2); j++) {
        const int n = GATE_UP ? slab * (kWCols / 2) + 32 * wn + lr : slab * kWCols + 64 * wn + 32 * j + lr;
        if (n >= p.out_dim) continue;
#pragma unroll
        for (int m = 0; m < MW; m++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int row = 32 * (MW * wm + m) + 8 * (r >> 2) + 4 * g + (r & 3);
                if (row >= rows) continue;
                const size_t o = (size_t)(p0 + row) * (size_t)p.out_dim + (size_t)n;
                if (GATE_UP) p.act[o] = (_Float16)__fmul_rn(fast_silu(acc[0][m][r]), acc[1][m][r]);
                else p.y[o] = acc[j][m][r];
            }
    }
}

template <bool GATE_UP, int WT>
__global__ __launch_bounds__(512, 2) void wide_gemm_kernel(WideArgs p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t s_lds[];   // Ring
    // As xcd_tile in gemm.hip: an XCD (workgroup ids equal modulo 8) takes neighbouring tiles with the slab running
    // fastest: the slabs of a tile share its rows in the XCD's L2, the tiles of an expert its weights.
    constexpr int kCols = GATE_UP ? kWCols / 2 : kWCols;
    const int n_slabs = (p.out_dim + kCols - 1) / kCols;
    const int total = *p.n_tiles, per_xcd = (total + 7) >> 3;
    const int item = (int)(blockIdx.x >> 3);
    const int within = item / n_slabs, slab = item - within * n_slabs;
    const int tile = (int)(blockIdx.x & 7) * per_xcd + within;
    if (within >= per_xcd || tile >= total) return;
    const int e = uniform(p.tiles[3 * tile]), p0 = uniform(p.tiles[3 * tile + 1]), rows = uniform(p.tiles[3 * tile + 2]);
    switch ((rows + kWideUnit - 1) / kWideUnit) {
    case 1: wide_tile<GATE_UP, WT, 1>(p, e, p0, rows, slab, s_lds); break;
    case 2: wide_tile<GATE_UP, WT, 2>(p, e, p0, rows, slab, s_lds); break;
    case 3: wide_tile<GATE_UP, WT, 3>(p, e, p0, rows, slab, s_lds); break;
    case 4: wide_tile<GATE_UP, WT, 4>(p, e, p0, rows, slab, s_lds); break;
    default: wide_tile<GATE_UP, WT, 5>(p, e, p0, rows, slab, s_lds); break;
    }
}

template <bool GATE_UP, int WT>
hipError_t launch_wide(const WideArgs &p, int max_tiles, hipStream_t s) {
    constexpr int kCols = GATE_UP ? kWCols / 2 : kWCols;
    const unsigned n_slabs = (unsigned)((p.out_dim + kCols - 1) / kCols);
    launch_kernel(wide_gemm_kernel<GATE_UP, WT>, dim3((unsigned)(max_tiles + 7) / 8 * 8 * n_slabs), dim3(512), (size_t)kWLds, s, p);
    return hipGetLastError();
}

}  // namespace

bool wide_gemm_takes(const ExpertBanks &b, int n_tokens, int n_assign) {
    // (rows are addressed with 32-bit byte offsets; two stages of K are loaded ahead)
    auto fits = [](int in_dim, int out_dim) {
        return in_dim % kWK == 0 && in_dim >= 2 * kWK && (size_t)in_dim * (size_t)out_dim * 2 < (1ull << 32);
    };
    if (!((b.gate_type == T_F16 || b.gate_type == T_BF16) && b.up_type == b.gate_type && b.down_type == b.gate_type &&
          fits(b.hidden, b.inter) && fits(b.inter, b.hidden) && (size_t)n_tokens * (size_t)b.hidden * 2 < (1ull << 32) &&
          (size_t)n_assign * (size_t)b.inter * 2 < (1ull << 32)))
        return false;
    // Up to 64 rows per expert either kernel streams the weights once, and the smaller workgroups of grouped_gemm_f16_kernel,
    // several to a CU, do it better (this kernel with its loads still in one go; OLMoE layers, 64 rows: 207 us there, 237 us here; 72: 256 / 245, 80: 260 / 249, 128: 325 / 276; 512
    // experts of 2560 x 640, 64: 1852 / 1907, 72: 2195 / 2018; 128 of 2048 x 768, 64: 366 / 354, 72: 427 / 381; 16 of 4096 x 1792, 64: 411 /
    // 402, 72: 428 / 417, 128: 568 / 490).
    // One workgroup fills a CU here, so the line also asks for about as many of them as there are CUs.  The one smaller launch that
    // was measured on both sides is ahead all the same (8 experts of 4096 x 1536, 96 workgroups, 72 rows 311 / 275, 256: 491 / 484).
    const size_t tiles = (size_t)n_assign / kWideRows > (size_t)b.n_experts ? (size_t)n_assign / kWideRows : (size_t)b.n_experts;
    const size_t out_dim = (size_t)(b.inter * 2 < b.hidden ? b.inter * 2 : b.hidden);
    return (size_t)n_assign >= 72 * (size_t)b.n_experts && tiles * (out_dim / kWCols) >= 224;
}

hipError_t launch_wide_gate_up(const ExpertBanks &b, const _Float16 *x16, const int32_t *sorted, int k_slots, const int32_t *tiles,
                               const int32_t *n_tiles, int max_tiles, _Float16 *act16, hipStream_t s) {
    const WideArgs p{b.gate, b.up, x16, sorted, tiles, n_tiles, k_slots, b.hidden, b.inter, act16, nullptr};
    return b.gate_type == T_F16 ? launch_wide<true, T_F16>(p, max_tiles, s) : launch_wide<true, T_BF16>(p, max_tiles, s);
}

hipError_t launch_wide_down(const ExpertBanks &b, const _Float16 *act16, const int32_t *tiles, const int32_t *n_tiles, int max_tiles,
                            float *y, hipStream_t s) {
    const WideArgs p{b.down, nullptr, act16, nullptr, tiles, n_tiles, 1, b.inter, b.hidden, nullptr, y};
    return b.down_type == T_F16 ? launch_wide<false, T_F16>(p, max_tiles, s) : launch_wide<false, T_BF16>(p, max_tiles, s);
}

}  // namespace mummu
