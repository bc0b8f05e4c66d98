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
//   - One workgroup fills a CU, so that nothing hides what it does outside its loop over K.  It stays and takes items - from a counter
//     of its XCD, since tiles are of unlike heights - and asks for the first stages of the next before it stores the results of the last.
//     A workgroup an item, 4096 / 3000 bf16 tokens a layer 554 -> 519, 443 -> 416 us, 4096 / 2000 of f16 537 -> 514, 309 -> 304; where the
//     stream of the weights bounds it the same (1000 tokens 235, 600: 203; with the next item looked up behind the last step, and both
//     stages waited for, 600 tokens were 3 % slower).
// What remains: the matrix units were busy for 52 / 38 % of the cycles at 4096 bf16 rows x 8 with a workgroup an item, and the card lowers its
// clock as they are: 15 % fewer cycles were 7 % of the time (340 / 206 us -> 316 / 194, a trace of it on its own).
#include <type_traits>

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
    const int32_t *sorted, *tiles;
    int32_t *n_tiles;              // the number of tiles, then the counters of items (WORK_GATE_UP, WORK_DOWN)
    int k_slots, in_dim, out_dim;
    _Float16 *act;                 // gate/up: silu(g) * u, sorted positions
    float *y;                      // down
};

// (What follows from it is formed again for every item: kept over the items, for each height of a tile, it would not fit the registers.)
__device__ inline int thread_id() {
    int t = (int)threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
}

// A tile and its slab; no rows: there is none.
struct Item {
    int e, p0, rows, slab;
};

// Item i of the workgroup's XCD.  As xcd_tile in gemm.hip: an XCD (workgroup ids equal modulo 8) takes neighbouring tiles with the
// slab running fastest: the slabs of a tile share its rows in the XCD's L2, the tiles of an expert its weights.
template <bool GATE_UP>
__device__ inline Item item_of(const WideArgs &p, int i) {
    constexpr int kCols = GATE_UP ? kWCols / 2 : kWCols;
    const int n_slabs = (p.out_dim + kCols - 1) / kCols;
    const int total = p.n_tiles[0], per_xcd = (total + 7) >> 3;
    const int within = i / n_slabs, tile = (int)(blockIdx.x & 7) * per_xcd + within;
    if (within >= per_xcd || tile >= total) return Item{0, 0, 0, 0};
    return Item{uniform(p.tiles[3 * tile]), uniform(p.tiles[3 * tile + 1]), uniform(p.tiles[3 * tile + 2]), i - within * n_slabs};
}

// What a wave moves of a stage: rows 8 mw wave .. of the activation tile (8 to a load: a lane per 16-byte piece) and
// rows 32 wave .. of the weight tile.  Row r of a tile holds its eight pieces in the order q ^ (r / 2 % 8): sixteen lanes that
// read the same piece of neighbouring rows then meet all 64 banks.
struct Loader {
    uint32_t a_off[5], b_off[4];
    const uint8_t *a_base, *b_base;

    __device__ void load_a(uint32_t at, int step, int mw, int wave, int i) const {
        load_to_lds16(at + (uint32_t)(8 * mw * wave + 8 * i) * (kWK * 2), a_base + (size_t)step * (kWK * 2), a_off[i]);
    }
    __device__ void load_b(uint32_t at, int step, int wave, int i) const {
        load_to_lds16(at + (uint32_t)(32 * wave + 8 * i) * (kWK * 2), b_base + (size_t)step * (kWK * 2), b_off[i]);
    }

    // The rows of an item of 64 mw rows.
    template <bool GATE_UP>
    __device__ void rows_of(const WideArgs &p, const Item &t, int mw) {
        const int tid = thread_id(), lane = tid & 63, wave = uniform(tid >> 6), lrow = lane >> 3;
        const uint32_t row_bytes = (uint32_t)p.in_dim * 2u, piece = (uint32_t)((lane & 7) ^ (lrow >> 1)) * 16u;   // (of an even eight of rows)
        a_base = (const uint8_t *)p.a;
#pragma unroll
        for (int i = 0; i < 5; i++) {
            const int r = 8 * mw * wave + 8 * i + lrow;
            const int rr = r < t.rows ? r : t.rows - 1;   // (rows past the tile's end repeat its last: multiplied, never stored)
            a_off[i] = (uint32_t)(GATE_UP ? p.sorted[t.p0 + rr] / p.k_slots : t.p0 + rr) * row_bytes + (piece ^ (uint32_t)(((mw * wave + i) & 1) * 64));
        }
        // weight rows: gate/up: 32 rows of gate, then 32 of up for each pair of waves; down: 64 rows for each pair
        const int col0 = GATE_UP ? t.slab * (kWCols / 2) + 32 * (wave >> 1) : t.slab * kWCols + 32 * wave;
        b_base = uniform((GATE_UP && (wave & 1) ? p.w1 : p.w0) + (size_t)t.e * (size_t)p.out_dim * row_bytes);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int col = col0 + 8 * i + lrow < p.out_dim ? col0 + 8 * i + lrow : p.out_dim - 1;
            b_off[i] = (uint32_t)col * row_bytes + (piece ^ (uint32_t)((i & 1) * 64));
        }
    }
    // Its first two stages: for each of them four loads of weights and mw of rows.
    __device__ void begin(int mw, uint32_t lds0, int wave) {
        const uint32_t lds_a = lds0 + (mw <= 4 ? Ring<4>::kAtA : Ring<5>::kAtA);
#pragma unroll
        for (int step = 0; step < 2; step++) {
#pragma unroll
            for (int i = 0; i < 4; i++) load_b(lds0 + step * kWStageB, step, wave, i);
#pragma unroll
            for (int i = 0; i < 5; i++)
                if (i < mw) load_a(lds_a + (uint32_t)(step * 64 * mw * (kWK * 2)), step, mw, wave, i);
        }
    }
};

// What is behind an item's first two stages when it begins: nothing, stores that may be left out of the wait for its second one, or so many
// that this has landed too.
enum Behind { NOTHING, SOME_STORES, MANY_STORES };

// One item, of up to 64 MW rows; wave (wm, wn) multiplies rows 32 MW wm .. by its 64 weight rows.  Its first stage has landed as far as
// this wave asked for it, the second is on its way.  Returns the workgroup's next item, of which the same is true then.
template <bool GATE_UP, int WT, int MW>
__device__ inline Item wide_tile(const WideArgs &p, const Item t, Loader &l, Behind &behind, uint8_t *s_lds) {
    using R = Ring<MW>;
    const int tid = thread_id(), lane = tid & 63, wave = uniform(tid >> 6);
    const int wm = wave >> 2, wn = wave & 3, g = lane >> 5, lr = lane & 31;
    const uint32_t lds0 = lds_offset(s_lds);
    const int n_steps = p.in_dim / kWK;

    float16v acc[2][MW];
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
        for (int m = 0; m < MW; m++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[b][m][r] = 0.0f;
    // piece 2 kk + g of the wave's rows: where group 0's is, and 2 kk more of a row's order
    const uint32_t q = (uint32_t)(g ^ (lr >> 1 & 7)) * 16u;
    uint32_t a_rd = R::kAtA + (uint32_t)(32 * MW * wm + lr) * (kWK * 2) + q, b_rd = (uint32_t)(64 * wn + lr) * (kWK * 2) + q;
    // operands of 16 elements of K, read while the ones before are multiplied
    half8 ra[2][MW], rb[2][2];
    u32x4 raw[2];
    auto read = [&](uint32_t at_a, uint32_t at_b, int kk) {
#pragma unroll
        for (int j = 0; j < 2; j++) raw[j] = *(const u32x4 *)(s_lds + ((b_rd ^ (32u * kk)) + at_b) + 32 * (kWK * 2) * j);
#pragma unroll
        for (int m = 0; m < MW; m++) ra[kk & 1][m] = *(const half8 *)(s_lds + ((a_rd ^ (32u * kk)) + at_a) + 32 * (kWK * 2) * m);
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
    // they fill the address unit's queue, and every wave stands before it.
    constexpr int kAhead = R::kB == 3 ? 2 : 1, kJ = GATE_UP ? 1 : 2;
    const uint32_t lds_a = lds0 + R::kAtA;
    asm volatile("s_barrier" ::: "memory");
    read(0, 0, 0);
    convert(0);
    uint32_t at_b = 0, free_b = kAhead * kWStageB;   // of this step's weights; of those kAhead on
    int taken = 0;
    // The word that tells the other waves the next item, where no load is under way to: the weights' third stage, or behind the last
    int *const told = (int *)(s_lds + (R::kB == 3 ? n_steps % 3 * kWStageB : R::kAtA + 2 * R::kStageA));
    Item next{0, 0, 0, 0};
    // LEFT: steps behind this one (2: or more)
    auto multiply_step = [&](int step, auto left) {
        constexpr int LEFT = decltype(left)::value;
        asm volatile("" : "+v"(a_rd), "+v"(b_rd));   // (no registers for their eight sums and differences over the steps)
        const uint32_t at_a = (uint32_t)(step & 1) * R::kStageA, next_a = R::kStageA - at_a;
        const uint32_t next_b = at_b == (R::kB - 1) * kWStageB ? 0u : at_b + kWStageB;
        // The next item is taken late, so that a workgroup with much to do takes fewer, and looked up in the last step.
        if (LEFT == 1 && tid == 0) taken = (int)(gridDim.x >> 3) + atomicAdd(p.n_tiles + (GATE_UP ? WORK_GATE_UP : WORK_DOWN) + (blockIdx.x & 7), 1);
        if (LEFT == 0) taken = *told;
#pragma unroll
        for (int kk = 0; kk < 4; kk++) {
            if (LEFT == 0 && kk == 1) next = item_of<GATE_UP>(p, uniform(taken));
            if (LEFT == 0 && kk == 2 && next.rows > 0) l.rows_of<GATE_UP>(p, next, (next.rows + kWideUnit - 1) / kWideUnit);
            if (LEFT == 1 && kk == 3 && tid == 0) *told = taken;
            // The next stage has landed and this one has been read by everybody.  (In the first step the stores of the item before stand between the
            // second stage and the third's weights.)
            if (kk == 3) {
                if ((LEFT == 0 && kAhead == 2) || (LEFT > 0 && step == 0 && behind == MANY_STORES)) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
                else if (step == 0 && behind == SOME_STORES) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(16 * kJ) : "memory");
                else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kAhead == 2 && LEFT == 2 ? 4 : 0) : "memory");
            }
            if (LEFT > 0 || kk < 3) read(kk == 3 ? next_a : at_a, kk == 3 ? next_b : at_b, (kk + 1) & 3);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int m = 0; m < MW; m++) {
                multiply(kk, m);
                if (kk == 3 && LEFT == 2) l.load_a(lds_a + at_a, step + 2, MW, wave, m);
                if (kk == 0 && LEFT >= kAhead) {
#pragma unroll
                    for (int i = m; i < 4; i += MW) l.load_b(lds0 + free_b, step + kAhead, wave, i);
                }
                if (m == MW - 1 && (LEFT > 0 || kk < 3)) convert((kk + 1) & 3);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        free_b = at_b;
        at_b = next_b;
    };
    for (int step = 0; step < n_steps - 2; step++) multiply_step(step, std::integral_constant<int, 2>());
    multiply_step(n_steps - 2, std::integral_constant<int, 1>());
    multiply_step(n_steps - 1, std::integral_constant<int, 0>());

    // The next item's first stages are on their way while this one's results leave, and those have the next one's first step for it.
    if (next.rows > 0) l.begin((next.rows + kWideUnit - 1) / kWideUnit, lds0, wave);
    // Element r of an accumulator: row 8 (r / 4) + 4 g + r % 4, column lane % 32.  Stores by a resource that ends behind the tile's last
    // row: what lies beyond is dropped, so that every tile makes the same number of them.
    const uint32_t ld = (uint32_t)p.out_dim * (GATE_UP ? 2u : 4u);
    uint8_t *const base = (GATE_UP ? (uint8_t *)p.act : (uint8_t *)p.y) + (size_t)t.p0 * ld;
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, (int)((uint32_t)t.rows * ld), 0x20000);
#pragma unroll
    for (int j = 0; j < kJ; j++) {
        const int n = GATE_UP ? t.slab * (kWCols / 2) + 32 * wn + lr : t.slab * kWCols + 64 * wn + 32 * j + lr;
        const uint32_t at = n < p.out_dim ? (uint32_t)(32 * MW * wm + 4 * g) * ld + (uint32_t)n * (GATE_UP ? 2u : 4u) : 1u << 31;
#pragma unroll
        for (int m = 0; m < MW; m++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const uint32_t o = at + (uint32_t)(32 * m + 8 * (r >> 2) + (r & 3)) * ld;
                if constexpr (GATE_UP) {
                    const _Float16 h = (_Float16)__fmul_rn(fast_silu(acc[0][m][r]), acc[1][m][r]);
                    short v;
                    __builtin_memcpy(&v, &h, 2);
                    __builtin_amdgcn_raw_buffer_store_b16(v, rsrc, (int)o, 0, 0);
                } else {
                    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[j][m][r]), rsrc, (int)o, 0, 0);
                }
            }
    }
    // The first stage, in front of the second's five loads or more and the stores.
    constexpr int kStores = 16 * MW * kJ;
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kStores + 5 < 63 ? kStores + 5 : 63) : "memory");
    behind = kStores >= 63 ? MANY_STORES : SOME_STORES;
    return next;
}

// A workgroup fills a CU, so what it does outside the loop over K is hidden by no other: it takes items until its XCD's are gone.
template <bool GATE_UP, int WT>
__global__ __launch_bounds__(512, 2) void wide_gemm_kernel(WideArgs p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t s_lds[];   // Ring
    Item t = item_of<GATE_UP>(p, (int)(blockIdx.x >> 3));
    if (t.rows == 0) return;
    Loader l;
    Behind behind = NOTHING;
    const int mw0 = (t.rows + kWideUnit - 1) / kWideUnit;
    l.rows_of<GATE_UP>(p, t, mw0);
    l.begin(mw0, lds_offset(s_lds), uniform((int)threadIdx.x >> 6));
    asm volatile("s_waitcnt vmcnt(5) lgkmcnt(0)" ::: "memory");
    while (t.rows > 0) {
        switch ((t.rows + kWideUnit - 1) / kWideUnit) {
        case 1: t = wide_tile<GATE_UP, WT, 1>(p, t, l, behind, s_lds); break;
        case 2: t = wide_tile<GATE_UP, WT, 2>(p, t, l, behind, s_lds); break;
        case 3: t = wide_tile<GATE_UP, WT, 3>(p, t, l, behind, s_lds); break;
        case 4: t = wide_tile<GATE_UP, WT, 4>(p, t, l, behind, s_lds); break;
        default: t = wide_tile<GATE_UP, WT, 5>(p, t, l, behind, s_lds); break;
        }
    }
}

template <bool GATE_UP, int WT>
hipError_t launch_wide(const WideArgs &p, int max_tiles, hipStream_t s) {
    constexpr int kCols = GATE_UP ? kWCols / 2 : kWCols, kCusOfXcd = 32;
    const int per_xcd = (max_tiles + 7) / 8 * ((p.out_dim + kCols - 1) / kCols);
    launch_kernel(wide_gemm_kernel<GATE_UP, WT>, dim3(8u * (unsigned)(per_xcd < kCusOfXcd ? per_xcd : kCusOfXcd)), dim3(512), (size_t)kWLds, s, p);
    return hipGetLastError();
}

}  // namespace

bool wide_gemm_takes(const ExpertBanks &b, int n_tokens, int n_assign) {
    // (rows are addressed with 32-bit byte offsets, a tile's results with 31 bits; two stages of K are loaded ahead)
    auto fits = [](int in_dim, int out_dim) {
        return in_dim % kWK == 0 && in_dim >= 2 * kWK && (size_t)in_dim * (size_t)out_dim * 2 < (1ull << 32) &&
               (size_t)kWideRows * (size_t)out_dim * 4 < (1ull << 31);
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
                               int32_t *n_tiles, int max_tiles, _Float16 *act16, hipStream_t s) {
    const WideArgs p{b.gate, b.up, x16, sorted, tiles, n_tiles, k_slots, b.hidden, b.inter, act16, nullptr};
    return b.gate_type == T_F16 ? launch_wide<true, T_F16>(p, max_tiles, s) : launch_wide<true, T_BF16>(p, max_tiles, s);
}

hipError_t launch_wide_down(const ExpertBanks &b, const _Float16 *act16, const int32_t *tiles, int32_t *n_tiles, int max_tiles,
                            float *y, hipStream_t s) {
    const WideArgs p{b.down, nullptr, act16, nullptr, tiles, n_tiles, 1, b.inter, b.hidden, nullptr, y};
    return b.down_type == T_F16 ? launch_wide<false, T_F16>(p, max_tiles, s) : launch_wide<false, T_BF16>(p, max_tiles, s);
}

}  // namespace mummu
