// Token -> expert dispatch for batched (prefill) calls: a stable counting sort of the
// (token, slot) assignments by expert id, with the per-expert histograms, ranks and scans held
// in LDS.
//
// Reference: SparseMoePerExpert::route builds, per expert, the token rows it serves in
// token-major, slot-minor order (nn/moe.rs:275-285); RoutedExperts::apply_routing buckets
// (token, weight) the same way (models/qwen4exp/experts.rs:1108-1120).  The sort is stable, so
// every expert's segment lists its assignments in ascending a = token*k + slot, which is that
// order.
//
// Two small launches over chunks of 1024 assignments (one fused launch of one workgroup for up to three
// chunks, where the launches themselves are most of the time):
//   count   per chunk: every assignment's rank among the chunk's assignments to the same expert
//           (wave ballots, then a prefix over the workgroup's 16 waves in LDS) and the chunk's
//           per-expert counts
//   scan + place   per chunk: per expert the count over the chunks before this one and the total, the
//           exclusive scan of the totals over experts (offsets), then
//           position = offsets[e] + rows of e in earlier chunks + rank.  Workgroup 0 also adds the totals to
//           the layer's hit counters when asked (8 atomics per token from the router would all land on the same
//           few cache lines) and writes the grouped GEMM's work list of (expert, first sorted position,
//           rows <= tile_rows) triples - every expert writes its own tiles at the position an exclusive scan of
//           the tile counts gives it
//
// Outputs (device):
//   offsets[E+1]      expert e owns sorted positions [offsets[e], offsets[e+1])
//   sorted[A]         sorted position -> assignment index a
//   inv[A]            assignment index a -> sorted position
//   tiles, n_tiles    the work list, its length and the zeroed counters behind that
#include "device_utils.h"
#include "kernels.h"
#include "qact.h"

namespace mummu {

constexpr int kDispatchThreads = 1024;
constexpr int kDispatchWaves = kDispatchThreads / 64;
constexpr int kDispatchMaxExperts = 512;

// Workgroup b of n_b of a launch makes its share of the rows that the products read.  Nothing of the sort waits for it, and the launch of its own that
// it had took as long as the sort's first one: 2 to 6 us of a layer alone; among others, which fill the launch's gaps, up to 4 (a launch of its own / here, among others and
// (alone), us: 320 tokens of Q8_0 180 / 176 (196 / 193), 512 of f16 163 / 163 (174 / 171), 300 of 512 experts with int8 downs 393 / 394 (438 / 432), 300 of Q4_K 104.6 / 103.7
// (125.6 / 122.5), 1000: 260 / 261 (298 / 297), 4096 of bf16 500 / 499 (532 / 530)).
__device__ inline void rows_part(const RowsJob &job, int b, int n_b) {
    __shared__ float s_max[kDispatchWaves];
    const int tid = threadIdx.x;
    if (job.h.hi != nullptr && job.h.lo == nullptr) {
        const size_t n4 = (size_t)job.n * (size_t)job.d / 4;
        for (size_t i = (size_t)b * kDispatchThreads + tid; i < n4; i += (size_t)n_b * kDispatchThreads) {
            const float4 v = ((const float4 *)job.x)[i];
            ((uint2 *)job.h.hi)[i] = make_uint2(pack_half2(v.x, v.y), pack_half2(v.z, v.w));
        }
        return;
    }
    // a row to four waves
    constexpr int NT = 256, kAtOnce = kDispatchThreads / NT;
    const int part = tid / NT, t = tid % NT;
    for (int row0 = b * kAtOnce; row0 < job.n; row0 += n_b * kAtOnce) {
        const int row = row0 + part;
        if (job.h.lo != nullptr) {
            hact_quantize_row<NT>(job.x, job.d, job.h, row, s_max + part * (NT / 64), t, row < job.n);
            __syncthreads();   // (s_max is free again)
        } else {
            for (int e0 = t * 4; e0 - t * 4 < job.d; e0 += NT * 4) {   // (whole groups of 16 lanes run together)
                const bool active = e0 < job.d && row < job.n;
                const float4 v = active ? *(const float4 *)(job.x + (size_t)row * (size_t)job.d + e0) : make_float4(0.f, 0.f, 0.f, 0.f);
                quantize_store64(v, active, job.q, (size_t)row, job.d, e0);
            }
        }
    }
}
unsigned rows_workgroups(const RowsJob &job) {
    if (job.x == nullptr) return 0;
    const size_t all = job.h.hi != nullptr && job.h.lo == nullptr ? ((size_t)job.n * (size_t)job.d / 4 + kDispatchThreads - 1) / kDispatchThreads
                                                                  : ((size_t)job.n + 3) / 4;
    return (unsigned)(all < 2048 ? all : 2048);
}

// Expert e's n tiles over its `rows` sorted rows from `begin`: whole units of rows dealt evenly, the first tiles one more.
__device__ inline void write_tiles(int32_t *__restrict__ tiles, int at, int n, int e, int begin, int rows, int unit) {
    if (n == 0) return;
    const int units = (rows + unit - 1) / unit, each = units / n, more = units - each * n;
    for (int i = 0, r = 0; i < n; i++) {
        const int take = (each + (i < more ? 1 : 0)) * unit;
        tiles[3 * (at + i)] = e;
        tiles[3 * (at + i) + 1] = begin + r;
        tiles[3 * (at + i) + 2] = rows - r < take ? rows - r : take;
        r += take;
    }
}

// Rank of this lane among the lanes of its wave with the same expert, whose number the first of them leaves in counts[e] (e < 0: no
// expert).  The lanes of an expert by a ballot per bit of its number: six to nine steps, where one per distinct expert of 64
// assignments, some forty, kept the four waves of a SIMD busy for two thirds of the launch (count, 1200 assignments to 64 experts 9.0 -> 5.0 us; the fused form, 216
// to 128 10.4 -> 4.7, 640 to 512 13.1 -> 5.2).
__device__ inline int rank_in_wave(int e, int n_experts, int lane, int *counts) {
    unsigned long long same = __ballot(e >= 0);
    for (int bit = 1; bit < n_experts; bit <<= 1) {
        const unsigned long long set = __ballot((e & bit) != 0);
        same &= e & bit ? set : ~set;
    }
    const int rank = __builtin_popcountll(same & ((1ull << lane) - 1ull));
    if (e >= 0 && rank == 0) counts[e] = __builtin_popcountll(same);
    return rank;
}

__global__ __launch_bounds__(kDispatchThreads) void dispatch_count_kernel(const int32_t *__restrict__ ids, int n_assign,
                                                                          int n_experts, int32_t *__restrict__ rank_out,
                                                                          int32_t *__restrict__ counts,
                                                                          int32_t *__restrict__ flags, int n_chunks, RowsJob job) {
    __shared__ __attribute__((aligned(16))) int s_wave[kDispatchWaves][kDispatchMaxExperts];  // per-wave counts of this chunk
    if ((int)blockIdx.x >= n_chunks) {
        rows_part(job, (int)blockIdx.x - n_chunks, (int)gridDim.x - n_chunks);
        return;
    }
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int chunk = blockIdx.x;
    for (int i = tid; i < kDispatchWaves * kDispatchMaxExperts / 4; i += kDispatchThreads) ((int4 *)s_wave)[i] = make_int4(0, 0, 0, 0);
    __syncthreads();
    const int a = chunk * kDispatchThreads + tid;
    int e = a < n_assign ? ids[a] : -1;
    if (a < n_assign && (unsigned)e >= (unsigned)n_experts) {
        atomicAdd(&flags[FLAG_BAD_ID], 1);
        e = -1;
    }
    const int rank = rank_in_wave(e, n_experts, lane, s_wave[wave]);
    __syncthreads();
    if (e >= 0) {
        int before = 0;
        for (int w = 0; w < wave; w++) before += s_wave[w][e];
        rank_out[a] = before + rank;
    }
    for (int x = tid; x < n_experts; x += kDispatchThreads) {
        int total = 0;
#pragma unroll
        for (int w = 0; w < kDispatchWaves; w++) total += s_wave[w][x];
        counts[(size_t)chunk * n_experts + x] = total;
    }
}

// scan + place: every chunk's workgroup scans the (chunks x experts) counts for itself - a few thousand integers out
// of L2 - instead of waiting for a launch of one workgroup to do it once (a third launch costs 4-5 us, the repeated
// scan a fraction of that even at 64k tokens); workgroup 0 also writes offsets, the tile list and the hit counters.
__global__ __launch_bounds__(kDispatchThreads) void dispatch_scan_place_kernel(
    const int32_t *__restrict__ ids, int n_assign, int n_experts, int n_chunks, int tile_rows, int unit,
    const int32_t *__restrict__ rank_in, const int32_t *__restrict__ counts, int32_t *__restrict__ offsets,
    int32_t *__restrict__ sorted, int32_t *__restrict__ inv, int32_t *__restrict__ tiles, int32_t *__restrict__ n_tiles,
    unsigned long long *__restrict__ hits) {
    __shared__ int s_carry[kDispatchMaxExperts / 64][2];
    __shared__ int s_pos[kDispatchMaxExperts];   // offsets[e] + rows of e in the chunks before this one
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int chunk = blockIdx.x;
    const int e = tid;
    int total = 0, before = 0;
    if (e < n_experts) {
#pragma unroll 8
        for (int c = 0; c < n_chunks; c++) {
            const int v = counts[(size_t)c * n_experts + e];
            before += c < chunk ? v : 0;
            total += v;
        }
    }
    const int my_tiles = (total + tile_rows - 1) / tile_rows;
    int incl = total, incl_t = my_tiles;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int up = __shfl_up(incl, off, 64), up_t = __shfl_up(incl_t, off, 64);
        if (lane >= off) {
            incl += up;
            incl_t += up_t;
        }
    }
    if (lane == 63 && wave < kDispatchMaxExperts / 64) {
        s_carry[wave][0] = incl;
        s_carry[wave][1] = incl_t;
    }
    __syncthreads();
    if (e < n_experts) {
        int base = 0, base_t = 0;
        for (int w = 0; w < wave; w++) {
            base += s_carry[w][0];
            base_t += s_carry[w][1];
        }
        const int begin = base + incl - total;
        s_pos[e] = begin + before;
        if (chunk == 0) {
            if (hits) hits[e] += (unsigned long long)total;  // rows served per expert (nn/moe.rs:1562-1564)
            offsets[e] = begin;
            if (e == n_experts - 1) offsets[n_experts] = begin + total;
            if (tiles != nullptr) {
                write_tiles(tiles, base_t + incl_t - my_tiles, my_tiles, e, begin, total, unit);
                if (e == n_experts - 1) {
                    *n_tiles = base_t + incl_t;
                    for (int i = 1; i < WORK_INTS; i++) n_tiles[i] = 0;
                }
            }
        }
    }
    __syncthreads();
    const int a = chunk * kDispatchThreads + tid;
    if (a >= n_assign) return;
    const int ea = ids[a];
    if ((unsigned)ea >= (unsigned)n_experts) return;
    const int pos = s_pos[ea] + rank_in[a];
    sorted[pos] = a;
    inv[a] = pos;
}

// The three steps above in one launch of one workgroup, for batches of at most kFusedChunks
// chunks: the per-chunk counts never leave LDS and every thread keeps its assignments' experts and
// ranks in registers between the steps.  Same outputs, element for element.  One workgroup takes
// 4.7 us for one chunk, 7.3 for two, 8.5 for three and 21.7 for eight, the two launches 10 us and the gap between them
// whatever the size.
constexpr int kFusedChunks = 3;

__global__ __launch_bounds__(kDispatchThreads) void dispatch_fused_kernel(
    const int32_t *__restrict__ ids, int n_assign, int n_experts, int tile_rows, int unit, int32_t *__restrict__ offsets,
    int32_t *__restrict__ sorted, int32_t *__restrict__ inv, int32_t *__restrict__ tiles, int32_t *__restrict__ n_tiles,
    unsigned long long *__restrict__ hits, int32_t *__restrict__ flags, RowsJob job) {
    if (blockIdx.x > 0) {
        rows_part(job, (int)blockIdx.x - 1, (int)gridDim.x - 1);
        return;
    }
    __shared__ __attribute__((aligned(16))) int s_wave[kDispatchWaves][kDispatchMaxExperts];   // per-wave counts of the current chunk
    __shared__ int s_chunk[kFusedChunks][kDispatchMaxExperts];    // per-chunk counts, then exclusive running counts
    __shared__ int s_off[kDispatchMaxExperts];
    __shared__ int s_carry[kDispatchMaxExperts / 64][2];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int chunks = (n_assign + kDispatchThreads - 1) / kDispatchThreads;
    int my_e[kFusedChunks], my_rank[kFusedChunks];
#pragma unroll
    for (int c = 0; c < kFusedChunks; c++) {
        my_e[c] = -1;
        my_rank[c] = 0;
        if (c >= chunks) continue;  // uniform over the workgroup
        for (int i = tid; i < kDispatchWaves * kDispatchMaxExperts / 4; i += kDispatchThreads) ((int4 *)s_wave)[i] = make_int4(0, 0, 0, 0);
        __syncthreads();
        const int a = c * kDispatchThreads + tid;
        int e = a < n_assign ? ids[a] : -1;
        if (a < n_assign && (unsigned)e >= (unsigned)n_experts) {
            atomicAdd(&flags[FLAG_BAD_ID], 1);
            e = -1;
        }
        const int rank = rank_in_wave(e, n_experts, lane, s_wave[wave]);
        __syncthreads();
        if (e >= 0) {
            int before = 0;
            for (int w = 0; w < wave; w++) before += s_wave[w][e];
            my_rank[c] = before + rank;
        }
        my_e[c] = e;
        for (int x = tid; x < n_experts; x += kDispatchThreads) {
            int total = 0;
#pragma unroll
            for (int w = 0; w < kDispatchWaves; w++) total += s_wave[w][x];
            s_chunk[c][x] = total;
        }
        __syncthreads();  // s_wave is cleared again for the next chunk
    }
    // running counts over chunks, offsets over experts, the work list (threads = experts)
    const int e = tid;
    int total = 0;
    if (e < n_experts) {
        for (int c = 0; c < chunks; c++) {
            const int v = s_chunk[c][e];
            s_chunk[c][e] = total;
            total += v;
        }
    }
    const int my_tiles = (total + tile_rows - 1) / tile_rows;
    int incl = total, incl_t = my_tiles;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int up = __shfl_up(incl, off, 64), up_t = __shfl_up(incl_t, off, 64);
        if (lane >= off) {
            incl += up;
            incl_t += up_t;
        }
    }
    if (lane == 63 && wave < kDispatchMaxExperts / 64) {
        s_carry[wave][0] = incl;
        s_carry[wave][1] = incl_t;
    }
    __syncthreads();
    if (e < n_experts) {
        int base = 0, base_t = 0;
        for (int w = 0; w < wave; w++) {
            base += s_carry[w][0];
            base_t += s_carry[w][1];
        }
        const int begin = base + incl - total;
        if (hits) hits[e] += (unsigned long long)total;
        offsets[e] = begin;
        s_off[e] = begin;
        if (e == n_experts - 1) offsets[n_experts] = begin + total;
        if (tiles != nullptr) {
            write_tiles(tiles, base_t + incl_t - my_tiles, my_tiles, e, begin, total, unit);
            if (e == n_experts - 1) {
                *n_tiles = base_t + incl_t;
                for (int i = 1; i < WORK_INTS; i++) n_tiles[i] = 0;
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < kFusedChunks; c++) {
        if (c >= chunks || my_e[c] < 0) continue;
        const int a = c * kDispatchThreads + tid;
        const int pos = s_off[my_e[c]] + s_chunk[c][my_e[c]] + my_rank[c];
        sorted[pos] = a;
        inv[a] = pos;
    }
}

// The work list of ONE expert that serves every row in order (the shared expert of a Qwen-style
// block on the batched path; a single expert on its own): sorted[i] = i, tiles of tile_rows rows.
__global__ __launch_bounds__(256) void identity_tiles_kernel(int n, int tile_rows, int expert, int32_t *__restrict__ sorted,
                                                             int32_t *__restrict__ tiles, int32_t *__restrict__ n_tiles) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) sorted[i] = i;
    const int nt = (n + tile_rows - 1) / tile_rows;
    if (i < nt) {
        tiles[3 * i] = expert;
        tiles[3 * i + 1] = i * tile_rows;
        tiles[3 * i + 2] = (n - i * tile_rows) < tile_rows ? (n - i * tile_rows) : tile_rows;
    }
    if (i == 0) *n_tiles = nt;
}

hipError_t launch_identity_tiles(int n, int tile_rows, int expert, int32_t *sorted, int32_t *tiles, int32_t *n_tiles, hipStream_t s) {
    if (n <= 0 || tile_rows < 1) return hipErrorInvalidValue;
    launch_kernel(identity_tiles_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, tile_rows, expert, sorted, tiles, n_tiles);
    return hipGetLastError();
}

size_t dispatch_scratch_ints(int n_assign, int n_experts) {
    const size_t chunks = ((size_t)n_assign + kDispatchThreads - 1) / kDispatchThreads;
    return (size_t)n_assign + chunks * (size_t)n_experts;
}

hipError_t launch_dispatch(const int32_t *ids, int n_assign, int n_experts, int tile_rows, int unit, int32_t *offsets,
                           int32_t *sorted, int32_t *inv, int32_t *tiles, int32_t *n_tiles, int32_t *scratch,
                           unsigned long long *hits, int32_t *flags, const RowsJob &rows, hipStream_t s) {
    if (n_assign <= 0) return hipSuccess;
    if (rows.x != nullptr && rows.d % (rows.h.lo != nullptr ? 128 : (rows.h.hi != nullptr ? 4 : 64)) != 0) return hipErrorInvalidValue;
    const unsigned beside = rows_workgroups(rows);
    if (n_experts > kDispatchMaxExperts || tile_rows < 1 || unit < 1 || tile_rows % unit != 0) return hipErrorInvalidValue;
    const int chunks = (n_assign + kDispatchThreads - 1) / kDispatchThreads;
    if (chunks <= kFusedChunks) {
        launch_kernel(dispatch_fused_kernel, dim3(1 + beside), dim3(kDispatchThreads), 0, s, ids, n_assign, n_experts, tile_rows, unit, offsets,
                      sorted, inv, tiles, n_tiles, hits, flags, rows);
        return hipGetLastError();
    }
    int32_t *rank = scratch, *counts = scratch + n_assign;
    // per-kernel timing brackets the two launches as one: start from the first, stop from the last
    const LaunchTiming timing = g_launch_timing;
    g_launch_timing.stop = nullptr;
    launch_kernel(dispatch_count_kernel, dim3((unsigned)chunks + beside), dim3(kDispatchThreads), 0, s, ids, n_assign, n_experts, rank, counts,
                  flags, chunks, rows);
    g_launch_timing.start = nullptr;
    g_launch_timing.stop = timing.stop;
    launch_kernel(dispatch_scan_place_kernel, dim3(chunks), dim3(kDispatchThreads), 0, s, ids, n_assign, n_experts, chunks,
                  tile_rows, unit, (const int32_t *)rank, (const int32_t *)counts, offsets, sorted, inv, tiles, n_tiles, hits);
    g_launch_timing = timing;
    return hipGetLastError();
}

}  // namespace mummu
