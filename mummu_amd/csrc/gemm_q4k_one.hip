// One expert of Q4_K banks on its own, for few rows: the operands and arithmetic of gemm_q4k.hip, from f32 rows to f32 rows.
//
// What bounds it: nothing but latency.  The expert's 3.5 MB (OLMoE shape) are there in a microsecond, and a grouped GEMM of 48 rows is
// two dozen workgroups that walk eight super-blocks one after the other.  Here a wave has one super-block of K (or every eighth) and 16 weight
// rows of each matrix, so that a launch is one round trip to memory: weights and rows come straight into the registers that multiply
// them, the rows become pairs of halfs there (a scale per row and super-block), and the waves' sums meet in LDS in ascending order.
//
// A row's scale covers a super-block, the per-row kernels' one 16 elements: those keep more of what stands beside sub-blocks that are more than
// 2^23 above it and meet weights of 0 (off the 64-bit result, such a sub-block 2^20 / 2^23 / 2^26 above: 3.6e-6 / 1.9e-5 / 2.2e-4, those 1.8e-5 each
// time; none above: 1.1e-7).  The largest element lies below 2^15 for that (below 2^10, with room for the sums of 32 as halfs: 1.1e-4 / 5.6e-4 /
// 5.7e-3); the sums are of elements over 2^5 again.
//
// OLMoE shape, 48 rows: quantizing, gate/up and down by the per-row kernels 3.5 + 17.8 + 10.0 us -> 9.8 + 9.0, half of it the launch and the way
// to memory and back, half the instructions of a wave, two to a SIMD; the host call 77 -> 66 us.
#include "device_utils.h"
#include "kernels.h"
#include "q4k_half.h"
#include "qact.h"

namespace mummu {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kWaves = 8, kRows = 16, kBlock = 144;

struct OneArgs {
    const uint8_t *w0, *w1;   // the expert's gate and up, or down [out_dim][in_dim]
    const float *x;           // [rows][in_dim]
    float *out;               // [rows][out_dim]: silu(g) * u, or the down product
    int rows, in_dim, out_dim;
};

// Wave w: columns 16 (w / SLICES) .. + 15 of the workgroup's, super-blocks w % SLICES, + SLICES, ...  (gate/up: of gate and of up).
template <bool GATE_UP, int SLICES>
__global__ __launch_bounds__(64 * kWaves, 4) void q4k_one_kernel(OneArgs p) {
    constexpr int NB = GATE_UP ? 2 : 1, kGroups = kWaves / SLICES;
    __shared__ __attribute__((aligned(16))) f32x4 s_sum[kWaves][NB][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6), c = lane & 15, kg = lane >> 4;
    const int n_sb = p.in_dim / 256, group = wave / SLICES, row0 = (int)blockIdx.y * kRows;
    const int rows = p.rows - row0 < kRows ? p.rows - row0 : kRows;
    const size_t row_bytes = (size_t)n_sb * kBlock;
    const int col = ((int)blockIdx.x * kGroups + group) * 16 + c;
    const uint8_t *w_row[2] = {p.w0 + (size_t)col * row_bytes, (GATE_UP ? p.w1 : p.w0) + (size_t)col * row_bytes};
    const float *x_row = p.x + (size_t)(row0 + (c < rows ? c : rows - 1)) * (size_t)p.in_dim + 8 * kg;   // (rows past the last repeat it)

    const f32x4 zero = {0, 0, 0, 0};
    f32x4 acc[NB];
#pragma unroll
    for (int j = 0; j < NB; j++) acc[j] = zero;
    for (int sb = wave % SLICES; sb < n_sb; sb += SLICES) {
        // everything the super-block takes is asked for at once
        float4 xv[8][2];
        u32x4 h[NB];
        uint2 raw[NB][4];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float4 *from = (const float4 *)(x_row + 256 * sb + 32 * i);
            xv[i][0] = from[0], xv[i][1] = from[1];
        }
#pragma unroll
        for (int j = 0; j < NB; j++) {
            const uint8_t *from = w_row[j] + (size_t)sb * kBlock;
            h[j] = *(const u32x4 *)from;
#pragma unroll
            for (int st = 0; st < 4; st++) raw[j][st] = *(const uint2 *)(from + 16 + 32 * st + 8 * kg);
        }
        // the row's scale: of the largest of its 256 elements, which lanes c + 16 i hold
        float m = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; i++)
#pragma unroll
            for (int q = 0; q < 2; q++) m = fmaxf(fmaxf(fmaxf(m, fabsf(xv[i][q].x)), fmaxf(fabsf(xv[i][q].y), fabsf(xv[i][q].z))), fabsf(xv[i][q].w));
        m = fmaxf(m, __shfl_xor(m, 16, 64));
        m = fmaxf(m, __shfl_xor(m, 32, 64));
        float inv, scale;
        hact_scale_of(m, inv, scale, kHActLift);
        scale = __fmul_rn(scale, (float)(1 << kHActLift));   // (of the sums; d takes the elements' lift)
        // (element order of HAct; sums of 32 elements, over 2^kHActLift again to be halfs, hi and lo halfs of the first four in lanes c, of c + 32, of the others beside them)
        half8 hi[8], lo[8];
        half4v am;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float f[8] = {__fmul_rn(xv[i][0].x, inv), __fmul_rn(xv[i][0].z, inv), __fmul_rn(xv[i][0].y, inv), __fmul_rn(xv[i][0].w, inv),
                                __fmul_rn(xv[i][1].x, inv), __fmul_rn(xv[i][1].z, inv), __fmul_rn(xv[i][1].y, inv), __fmul_rn(xv[i][1].w, inv)};
            float sum = 0.0f;
#pragma unroll
            for (int q = 0; q < 8; q++) {
                hi[i][q] = (_Float16)f[q];
                lo[i][q] = (_Float16)__fsub_rn(f[q], (float)hi[i][q]);
                sum = fmaf(f[q], 1.0f / (1 << kHActLift), sum);
            }
            sum = __fadd_rn(sum, __shfl_xor(sum, 16, 64));
            sum = __fadd_rn(sum, __shfl_xor(sum, 32, 64));
            const _Float16 sh = (_Float16)sum, sl = (_Float16)__fsub_rn(sum, (float)sh);
            if (i / 4 == (kg & 1)) am[i & 3] = kg < 2 ? sh : sl;
        }
        float sr[4];
#pragma unroll
        for (int r = 0; r < 4; r++) sr[r] = __shfl(scale, 4 * kg + r, 64);
#pragma unroll
        for (int j = 0; j < NB; j++) {
            Q4kHeader head;
            head.unpack(h[j]);
            f32x4 c1 = zero;
#pragma unroll
            for (int st = 0; st < 4; st++) {
                half2v ml, mh;
                head.muls(st, ml, mh);
                const half8 w[2] = {q4k_operand<false>(raw[j][st].x, raw[j][st].y, ml), q4k_operand<true>(raw[j][st].x, raw[j][st].y, mh)};
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    c1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi[2 * st + q], w[q], c1, 0, 0, 0);
                    c1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo[2 * st + q], w[q], c1, 0, 0, 0);
                }
            }
            head.mn4[0] = kg & 1 ? head.mn4[1] : head.mn4[0];
            const f32x4 c2 = __builtin_amdgcn_mfma_f32_16x16x16f16(am, head.offsets(0), zero, 0, 0, 0);
            const float fd = head.d(kHActLift), fm = head.minus_dmin();
#pragma unroll
            for (int r = 0; r < 4; r++) acc[j][r] = fmaf(fmaf(fm, c2[r], __fmul_rn(fd, c1[r])), sr[r], acc[j][r]);
        }
    }
    // element r of lane (c, kg): row 4 kg + r, column c
#pragma unroll
    for (int j = 0; j < NB; j++) s_sum[wave][j][lane] = acc[j];
    __syncthreads();
    for (int i = tid; i < kGroups * 256; i += 64 * kWaves) {
        const int row = (i / 16) % 16, g = i / 256;
        auto sum_of = [&](int j) {
            float s = 0.0f;
#pragma unroll
            for (int k = 0; k < SLICES; k++) s = __fadd_rn(s, s_sum[g * SLICES + k][j][(row >> 2) * 16 + (i & 15)][row & 3]);
            return s;
        };
        if (row >= rows) continue;
        float v = sum_of(0);
        if (GATE_UP) v = __fmul_rn(silu_of(v), sum_of(NB - 1));
        p.out[(size_t)(row0 + row) * (size_t)p.out_dim + (size_t)(((int)blockIdx.x * kGroups + g) * 16 + (i & 15))] = v;
    }
}

template <bool GATE_UP, int SLICES>
hipError_t launch_one(const OneArgs &p, hipStream_t s) {
    constexpr int kCols = 16 * kWaves / SLICES;
    launch_kernel(q4k_one_kernel<GATE_UP, SLICES>, dim3((unsigned)(p.out_dim / kCols), (unsigned)((p.rows + kRows - 1) / kRows)), dim3(64 * kWaves), 0, s, p);
    return hipGetLastError();
}
// (as many waves along K as there are super-blocks, up to all of them)
template <bool GATE_UP>
hipError_t launch_one(const OneArgs &p, hipStream_t s) {
    const int n_sb = p.in_dim / 256;
    return n_sb >= 8 ? launch_one<GATE_UP, 8>(p, s) : n_sb >= 3 ? launch_one<GATE_UP, 4>(p, s) : launch_one<GATE_UP, 2>(p, s);
}

}  // namespace

hipError_t launch_q4k_one_gate_up(const ExpertBanks &b, int expert, const float *x, int rows, float *act, hipStream_t s) {
    const size_t at = (size_t)expert * (size_t)b.inter * (size_t)(b.hidden / 256) * kBlock;
    return launch_one<true>(OneArgs{b.gate + at, b.up + at, x, act, rows, b.hidden, b.inter}, s);
}

hipError_t launch_q4k_one_down(const ExpertBanks &b, int expert, const float *act, int rows, float *out, hipStream_t s) {
    const size_t at = (size_t)expert * (size_t)b.hidden * (size_t)(b.inter / 256) * kBlock;
    return launch_one<false>(OneArgs{b.down + at, nullptr, act, out, rows, b.inter, b.hidden}, s);
}

}  // namespace mummu
