// Grouped GEMM of F16 and BF16 banks with wide tiles, for many rows per expert: x and the activations between the two products as halfs and
// f32 accumulators as in grouped_gemm_f16_kernel (gemm.hip), v_mfma_f32_16x16x32_f16, on tiles of up to 320 rows by 256 weight rows (128 of
// gate and 128 of up, or 256 of down).
//
// What bounds it and why it looks the way it does (OLMoE shape, 4096 tokens = 512 rows per expert):
//   - Power.  The card lowers its clock as the matrix units are busy: with weights of zeros the same layer took 421 us instead of 540.  A product of 16 by
//     16 and 32 of K passes through the accumulators half as often as one of 32 by 32 and 16 (on registers alone, normal data, 1950 against
//     1697 TFLOP/s; 1726 / 1544 with four vector instructions to every 32 k operations): 1.79 -> 2.05 GHz, gate/up 277 -> 250 us; layers, us:
//     4096 / 3000 bf16 tokens 517 -> 492, 413 -> 387, 4096 of f16 506 -> 483.  The same bits.
//   - LDS reads.  A 64 x 128 tile reads one operand per 32 k operations, which keeps the LDS port (128 bytes a clock)
//     busy all the time at half the matrix rate.  Eight waves of 32 MW x 64 outputs (MW up to 5) read 7 for 10.
//   - The way into LDS.  Both tiles go from global memory straight into LDS, 64 elements of K (whole 128-byte lines: pieces
//     of 64 bytes come out of the L2 at half the rate, 17 against 34 TB/s) at a time, without registers in between, the weights two
//     stages ahead where the LDS holds them, and never a stage at once: 72 loads behind a barrier fill the address unit's queue, with
//     all eight waves waiting in front of it.  (Asked for in one go, one stage ahead: 4096 bf16 rows x 8 gate/up / down 620 / 416 k cycles
//     against 529 / 363, 1500 f16 rows 358 / 206 against 299 / 217.)
//   - Whole rounds.  An expert's rows are split evenly, in steps of 64, over as few tiles as hold them, so that the
//     workgroups of a launch are alike (full tiles and a remainder left a fifth of the launch to stragglers), and a wave
//     multiplies only as many row blocks as the tile has.
//   - Weights of bf16 become halfs beside the last products of the half stage before, not between their read and the next products.
//   - One workgroup fills a CU, so that nothing hides what it does outside its loop over K.  With many rows (items_in_turn) it stays and takes
//     items - from a counter of its XCD, since tiles are of unlike heights - and asks for the first stages of the next before it stores
//     the results of the last.
//   - What a lane keeps from item to item - offsets of rows - has to stay in registers: reloaded ones are waited for in the loop, behind every load
//     that is under way (bf16, 4096 tokens 492 -> 558).
// What remains: the matrix units are busy for 54 / 37 % of the cycles at 4096 bf16 rows x 8, and an XCD's L2 fetches more than
// the operands hold, 830 / 406 MB of 554 and 336 (the form on 32 x 32 x 16 products, with items of its own to each workgroup, 755 / 354; an item to a workgroup here 817 /
// 412, so that it is not the order of the items; the cause is not known).
#include <type_traits>

#include "device_utils.h"
#include "gemm_wide_ring.h"
#include "kernels.h"

namespace mummu {

namespace {

using namespace wide;

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

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
    const _Float16 *a;             // rows of in_dim halfs: tokens (gate/up, through sorted / slots) or sorted positions
    const int32_t *sorted, *tiles;
    int32_t *n_tiles;              // the number of tiles, then the counters of items (WORK_GATE_UP, WORK_DOWN)
    uint32_t per_slot;             // 2^32 / k_slots, rounded up: an assignment's token is the upper half of their product (0: one slot)
    int in_dim, out_dim;
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
    uint32_t a_off[5], b_off;
    const uint8_t *a_base, *b_base;

    __device__ void load_a(uint32_t at, int step, int mw, int wave, int i) const {
        load_to_lds16(at + (uint32_t)(8 * mw * wave + 8 * i) * (kWK * 2), a_base + (size_t)step * (kWK * 2), a_off[i]);
    }
    // (eight rows of LDS: every second or fourth of the matrix from the (i % 2) * 16-th or * 32-nd, i / 2 on)
    template <bool GATE_UP>
    __device__ void load_b(uint32_t at, int step, uint32_t row_bytes, int wave, int i) const {
        load_to_lds16(at + (uint32_t)(32 * wave + 8 * i) * (kWK * 2),
                      b_base + (size_t)step * (kWK * 2) + (size_t)((i & 1) * (GATE_UP ? 16 : 32) + (i >> 1)) * row_bytes, b_off ^ (uint32_t)((i & 1) * 64));
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
            uint32_t row = (uint32_t)(t.p0 + rr);
            if (GATE_UP) {
                row = (uint32_t)p.sorted[row];
                row = p.per_slot != 0 ? __umulhi(row, p.per_slot) : row;
            }
            a_off[i] = row * row_bytes + (piece ^ (uint32_t)(((mw * wave + i) & 1) * 64));
        }
        // weight rows: gate/up: 32 rows of gate, then 32 of up for each pair of waves; down: 64 rows for each pair (out_dim % 64 == 0: all of them there, or
        // none, and the last ones instead).  Sixteen rows of LDS are an operand: those of operand j hold rows j, j + n, j + 2 n .. of the wave's 64
        // (n: 4) or of the 32 of gate or up (2), so that a lane's results lie side by side.
        constexpr int kRun = GATE_UP ? 32 : 64;
        const int run0 = GATE_UP ? t.slab * (kWCols / 2) + 32 * (wave >> 1) : t.slab * kWCols + 64 * (wave >> 1);
        const int first = (run0 < p.out_dim ? run0 : p.out_dim - kRun) + (GATE_UP ? 0 : 2 * (wave & 1));
        b_base = uniform((GATE_UP && (wave & 1) ? p.w1 : p.w0) + ((size_t)t.e * (size_t)p.out_dim + (size_t)first) * row_bytes);
        b_off = (uint32_t)((GATE_UP ? 2 : 4) * lrow) * row_bytes + piece;
    }
    // Its first two stages: for each of them four loads of weights and mw of rows.
    template <bool GATE_UP>
    __device__ void begin(int mw, uint32_t lds0, uint32_t row_bytes, int wave) {
        const uint32_t lds_a = lds0 + (mw <= 4 ? Ring<4>::kAtA : Ring<5>::kAtA);
#pragma unroll
        for (int step = 0; step < kBegun; step++) {
#pragma unroll
            for (int i = 0; i < 4; i++) load_b<GATE_UP>(lds0 + step * kWStageB, step, row_bytes, wave, i);
#pragma unroll
            for (int i = 0; i < 5; i++)
                if (i < mw) load_a(lds_a + (uint32_t)(step * 64 * mw * (kWK * 2)), step, mw, wave, i);
        }
    }
};

// A step's wait: its loads but for so many have landed, and everybody has read what the next ones overwrite.
template <int LOADS>
__device__ inline void wait_and_meet() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(LOADS) : "memory");
}

// One item, of up to 64 MW rows; wave (wm, wn) multiplies rows 32 MW wm .. by its 64 weight rows.  Its first stage has landed as far as
// this wave asked for it, the second is on its way.  Returns the workgroup's next item, of which the same is true then.
template <bool GATE_UP, int WT, int MW>
__device__ inline Item wide_tile(const WideArgs &p, const Item t, Loader &l, int &behind, uint8_t *s_lds) {
    using R = Ring<MW>;
    const int tid = thread_id(), lane = tid & 63, wave = uniform(tid >> 6);
    const int wm = wave >> 2, wn = wave & 3;
    const uint32_t lds0 = lds_offset(s_lds);
    const int n_steps = p.in_dim / kWK;
    const uint32_t row_bytes = (uint32_t)p.in_dim * 2u;

    // Products of 16 rows by 16 columns and 32 of K: two row blocks for a product of 32 by 32 and 16, as many clocks, but half the
    // passes through the accumulators, and the card's power is what its clock goes by.  A unit: row block m of a half stage, by the wave's four operands
    // of weights.  Lane (row or column lane % 16, K group lane / 16).
    constexpr int kBlocks = 2 * MW, kUnits = 2 * kBlocks;
    constexpr int kEnd = MW == 1 ? 2 : 3;   // units behind a step's barrier, and how far ahead the rows are read
    const int kg = lane >> 4, lr = lane & 15;
    f32x4 acc[kBlocks][4];
#pragma unroll
    for (int m = 0; m < kBlocks; m++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[m][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    // (piece 4 half + kg of a row)
    const uint32_t q = (uint32_t)(kg ^ (lr >> 1 & 7)) * 16u;
    uint32_t a_rd = R::kAtA + (uint32_t)(32 * MW * wm + lr) * (kWK * 2) + q, b_rd = (uint32_t)(64 * wn + lr) * (kWK * 2) + q;
    half8 a_first[kEnd], b_now[4];   // of the step's first units
    auto read_a = [&](uint32_t at, int u) {
        return *(const half8 *)(s_lds + ((a_rd ^ (uint32_t)(u / kBlocks * 64)) + at) + 16 * (kWK * 2) * (u % kBlocks));
    };
    auto read_b = [&](uint32_t at, int half, int j) { return *(const u32x4 *)(s_lds + ((b_rd ^ (uint32_t)(half * 64)) + at) + 16 * (kWK * 2) * j); };
    // Behind the barrier of a step, beside its last products, the rows of the step after the next are asked for; beside the first
    // products after that the weights of one step more (tiles of more than 256 rows leave no room for that: of the same step).  All at once
    // they fill the address unit's queue, and every wave stands before it.
    constexpr int kAhead = R::kAhead;
    const uint32_t lds_a = lds0 + R::kAtA;
    asm volatile("s_barrier" ::: "memory");
#pragma unroll
    for (int u = 0; u < kEnd; u++) a_first[u] = read_a(0, u);
#pragma unroll
    for (int j = 0; j < 4; j++) b_now[j] = weight_operand<WT>(read_b(0, 0, j));
    uint32_t at_b = 0, free_b = kAhead * kWStageB;   // of this step's weights; of those kAhead on
    int taken = 0;
    // The word that tells the other waves the next item, where no load is under way to: the weights' third stage, or behind the last
    int *const told = (int *)(s_lds + (R::kB == 3 ? n_steps % 3 * kWStageB : R::kAtA + 2 * R::kStageA));
    Item next{0, 0, 0, 0};
    // LEFT: steps behind this one (2: or more); FIRST: the first of three or more
    auto multiply_step = [&](int step, auto left, auto first) {
        constexpr int LEFT = decltype(left)::value;
        constexpr bool FIRST = decltype(first)::value;
        asm volatile("" : "+v"(a_rd), "+v"(b_rd));   // (no registers for their sums and differences over the steps)
        const uint32_t at_a = (uint32_t)(step & 1) * R::kStageA, next_a = R::kStageA - at_a;
        const uint32_t next_b = at_b == (R::kB - 1) * kWStageB ? 0u : at_b + kWStageB;
        // The next item is taken late, so that a workgroup with much to do takes fewer, and looked up in the last step.
        if (LEFT == 1 && tid == 0) taken = (int)(gridDim.x >> 3) + atomicAdd(p.n_tiles + (GATE_UP ? WORK_GATE_UP : WORK_DOWN) + (blockIdx.x & 7), 1);
        if (LEFT == 0) taken = *told;
        half8 a[kUnits + kEnd], b[3][4];
        u32x4 raw[4];
#pragma unroll
        for (int u = 0; u < kEnd; u++) a[u] = a_first[u];
#pragma unroll
        for (int j = 0; j < 4; j++) b[0][j] = b_now[j];
#pragma unroll
        for (int u = 0; u < kUnits; u++) {
            const int half = u / kBlocks, m = u % kBlocks, behind_barrier = u - (kUnits - kEnd), to_half_end = m - (kBlocks - kEnd);
            if (LEFT == 0 && u == kUnits / 2) next = item_of<GATE_UP>(p, uniform(taken));
            if (LEFT == 0 && u == kUnits - 2 && next.rows > 0) l.template rows_of<GATE_UP>(p, next, (next.rows + kWideUnit - 1) / kWideUnit);
            if (behind_barrier == 0) {
                if (LEFT == 1 && tid == 0) *told = taken;
                // (In an item's first step the stores of the one before, eight to 64 of its rows, stand behind the stage that is waited for.)
                if (FIRST && behind == 1) wait_and_meet<step_wait(kAhead, LEFT, 1)>();
                else if (FIRST && behind == 2) wait_and_meet<step_wait(kAhead, LEFT, 2)>();
                else if (FIRST && behind == 3) wait_and_meet<step_wait(kAhead, LEFT, 3)>();
                else if (FIRST && behind == 4) wait_and_meet<step_wait(kAhead, LEFT, 4)>();
                else if (FIRST && behind == 5) wait_and_meet<step_wait(kAhead, LEFT, 5)>();
                else wait_and_meet<step_wait(kAhead, LEFT, 0)>();
            }
            // Rows kEnd units ahead; the stage's last two together, so that the barrier's wait for them is short
            if (u < kUnits - kEnd - 1) a[u + kEnd] = read_a(at_a, u + kEnd);
            if (u == kUnits - kEnd - 2) a[u + kEnd + 1] = read_a(at_a, u + kEnd + 1);
            if (behind_barrier >= 0 && LEFT > 0) a[kUnits + behind_barrier] = read_a(next_a, behind_barrier);
            // the next half stage's weights
            if (half == 0 || LEFT > 0) {
                const uint32_t from = half == 0 ? at_b : next_b;
#pragma unroll
                for (int j = 0; j < 4; j++)
                    if (to_half_end == (kEnd == 2 ? 0 : j / 2)) raw[j] = read_b(from, half ^ 1, j);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < 4; j++) acc[m][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[u], b[half][j], acc[m][j], 0, 0, 0);
            if (behind_barrier >= 0 && LEFT == 2) {
#pragma unroll
                for (int i = behind_barrier; i < MW; i += kEnd) l.load_a(lds_a + at_a, step + 2, MW, wave, i);
            }
            if (half == 0 && asks_weights(kAhead, LEFT, FIRST)) {
#pragma unroll
                for (int i = m; i < 4; i += kBlocks) l.template load_b<GATE_UP>(lds0 + free_b, step + kAhead, row_bytes, wave, i);
            }
            if ((half == 0 || LEFT > 0) && to_half_end >= 1) {
                // (two of them in each of the last two units; one unit: all)
#pragma unroll
                for (int j = 0; j < 4; j++)
                    if (kEnd == 2 || j / 2 == to_half_end - 1) b[half + 1][j] = weight_operand<WT>(raw[j]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (LEFT > 0) {
#pragma unroll
            for (int u = 0; u < kEnd; u++) a_first[u] = a[kUnits + u];
#pragma unroll
            for (int j = 0; j < 4; j++) b_now[j] = b[2][j];
        }
        free_b = at_b;
        at_b = next_b;
    };
    if (n_steps > 2) multiply_step(0, std::integral_constant<int, 2>(), std::true_type());
    for (int step = 1; step < n_steps - 2; step++) multiply_step(step, std::integral_constant<int, 2>(), std::false_type());
    multiply_step(n_steps - 2, std::integral_constant<int, 1>(), std::false_type());
    multiply_step(n_steps - 1, std::integral_constant<int, 0>(), std::false_type());

    // The next item's first stages are on their way while this one's results leave, and those have the next one's first step for it.
    if (next.rows > 0) l.template begin<GATE_UP>((next.rows + kWideUnit - 1) / kWideUnit, lds0, row_bytes, wave);
    // Element r of an accumulator: row 4 kg + r, column lane % 16, which is every second or fourth of the matrix's.  Stores by a resource that
    // ends behind the tile's last row: what lies beyond is dropped, so that every tile makes the same number of them.
    const uint32_t ld = (uint32_t)p.out_dim * (GATE_UP ? 2u : 4u);
    uint8_t *const base = (GATE_UP ? (uint8_t *)p.act : (uint8_t *)p.y) + (size_t)t.p0 * ld;
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, (int)((uint32_t)t.rows * ld), 0x20000);
    const int n = GATE_UP ? t.slab * (kWCols / 2) + 32 * wn + 2 * lr : t.slab * kWCols + 64 * wn + 4 * lr;   // (whole: out_dim % 64 == 0)
    const uint32_t at = n < p.out_dim ? (uint32_t)(32 * MW * wm + 4 * kg) * ld + (uint32_t)n * (GATE_UP ? 2u : 4u) : 1u << 31;
#pragma unroll
    for (int m = 0; m < kBlocks; m++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const uint32_t o = at + (uint32_t)(16 * m + r) * ld;
            if constexpr (GATE_UP) {
                _Float16 h[2];
#pragma unroll
                for (int j = 0; j < 2; j++) h[j] = (_Float16)__fmul_rn(fast_silu(acc[m][j][r]), acc[m][2 + j][r]);
                uint32_t v;
                __builtin_memcpy(&v, h, 4);
                __builtin_amdgcn_raw_buffer_store_b32(v, rsrc, (int)o, 0, 0);
            } else {
                u32x4 v;
#pragma unroll
                for (int j = 0; j < 4; j++) v[j] = __float_as_uint(acc[m][j][r]);
                __builtin_amdgcn_raw_buffer_store_b128(v, rsrc, (int)o, 0, 0);
            }
        }
    // The first stage, in front of the second's five loads or more and the stores.
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(begin_wait(MW)) : "memory");
    behind = MW;
    return next;
}

// A workgroup fills a CU, so what it does outside the loop over K is hidden by no other: it takes items until its XCD's are gone.
template <bool GATE_UP, int WT>
__global__ __launch_bounds__(512, 2) void wide_gemm_kernel(WideArgs p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t s_lds[];   // Ring
    Item t = item_of<GATE_UP>(p, (int)(blockIdx.x >> 3));
    if (t.rows == 0) return;
    Loader l;
    int behind = 0;   // (the height of the item before)
    const int mw0 = (t.rows + kWideUnit - 1) / kWideUnit;
    l.rows_of<GATE_UP>(p, t, mw0);
    l.begin<GATE_UP>(mw0, lds_offset(s_lds), (uint32_t)p.in_dim * 2u, uniform((int)threadIdx.x >> 6));
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(begin_wait(0)) : "memory");
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
hipError_t launch_wide(const WideArgs &p, int max_tiles, bool in_turn, hipStream_t s) {
    constexpr int kCols = GATE_UP ? kWCols / 2 : kWCols, kCusOfXcd = 32;
    const int per_xcd = (max_tiles + 7) / 8 * ((p.out_dim + kCols - 1) / kCols);
    launch_kernel(wide_gemm_kernel<GATE_UP, WT>, dim3(8u * (unsigned)(per_xcd < kCusOfXcd || !in_turn ? per_xcd : kCusOfXcd)), dim3(512), (size_t)kWLds, s, p);
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
          (size_t)n_assign * (size_t)b.inter * 2 < (1ull << 32) &&
          // (a - n_assign and less - over the slots of a token by way of 2^32 / slots: exact while a * slots < 2^32)
          (size_t)n_assign * (size_t)(n_assign / n_tokens) < (1ull << 32)))
        return false;
    // Up to one tile per expert either kernel streams the weights once, and the smaller workgroups of grouped_gemm_f16_kernel, several to a CU, do it
    // better, on tiles of 96 rows, until too many experts need a second one: at 79 rows one in 35, of evenly drawn ones (layers among others, us, there / here: OLMoE 64 rows 163 / 188, 69: 165 / 188, 74: 167 / 193, 80: 182 / 189, 83: 180 / 189, 86: 193 /
    // 194, 95: 217 / 199; 128 experts of 2048 x 768, 78 rows 273 / 288, 88: 302 / 298; 16 of 4096 x 1792, 81: 331 / 329, 88: 368 / 343; 64 of 1024 x 512, 72 / 82:
    // 56 / 62, 59 / 64; 128 of 512 x 512, 72 / 82: 64 / 71, 66 / 74).  Rows of a few steps of K are no stream: 224 experts of 256 x 128, 72 / 80 rows 73 / 71, 81 / 79.
    const size_t from = b.hidden >= 512 && b.inter >= 512 ? 79 : 72;
    // One workgroup fills a CU here, so the line also asks for about as many of them as there are CUs.  The one smaller launch that
    // was measured on both sides is ahead all the same (8 experts of 4096 x 1536, 96 workgroups, 72 rows 311 / 275, 256: 491 / 484).
    const size_t tiles = (size_t)n_assign / kWideRows > (size_t)b.n_experts ? (size_t)n_assign / kWideRows : (size_t)b.n_experts;
    const size_t out_dim = (size_t)(b.inter * 2 < b.hidden ? b.inter * 2 : b.hidden);
    return (size_t)n_assign >= from * (size_t)b.n_experts && tiles * (out_dim / kWCols) >= 224;
}

// Whether the workgroups of a launch are a CU's each and take items in turn, or an item's: where the stream of the weights bounds it, other streams'
// workgroups come in between as one ends, which is worth more.  Layers among others (three streams), us, an item / in turn: 600 tokens of f16 194 /
// 204, 800 bf16 201 / 214, 1000: 209 / 213-220, 1200 f16 224 / 232, 1500 bf16 240 / 240-250, 2000: 294 / 290-293, 2800: 390 / 385, 4096: 518 / 503.
static bool items_in_turn(const ExpertBanks &b, int n_assign) { return n_assign / 256 >= b.n_experts; }

hipError_t launch_wide_gate_up(const ExpertBanks &b, const _Float16 *x16, const int32_t *sorted, int k_slots, const int32_t *tiles,
                               int32_t *n_tiles, int max_tiles, int n_assign, _Float16 *act16, hipStream_t s) {
    const uint32_t per_slot = k_slots == 1 ? 0u : (uint32_t)(((1ull << 32) + (unsigned)k_slots - 1) / (unsigned)k_slots);
    const WideArgs p{b.gate, b.up, x16, sorted, tiles, n_tiles, per_slot, b.hidden, b.inter, act16, nullptr};
    return b.gate_type == T_F16 ? launch_wide<true, T_F16>(p, max_tiles, items_in_turn(b, n_assign), s) : launch_wide<true, T_BF16>(p, max_tiles, items_in_turn(b, n_assign), s);
}

hipError_t launch_wide_down(const ExpertBanks &b, const _Float16 *act16, const int32_t *tiles, int32_t *n_tiles, int max_tiles,
                            int n_assign, float *y, hipStream_t s) {
    const WideArgs p{b.down, nullptr, act16, nullptr, tiles, n_tiles, 0, b.inter, b.hidden, nullptr, y};
    return b.down_type == T_F16 ? launch_wide<false, T_F16>(p, max_tiles, items_in_turn(b, n_assign), s) : launch_wide<false, T_BF16>(p, max_tiles, items_in_turn(b, n_assign), s);
}

}  // namespace mummu
