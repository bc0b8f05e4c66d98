// Pinned staging of host rows (see host_staging.h).
#include "host_staging.h"

#include <cstring>

#include "device_utils.h"

namespace mummu {

namespace {

// Workgroups that share a range, and the words that they mark it with.
constexpr int kStageWgs = 64;

// Byte ranges copied by one launch, 16 bytes per lane and step; either side may be pinned host memory.  Both pointers of
// a range are 16-byte aligned.  blockIdx.y takes every gridDim.y-th range.  done (nullable, pinned): each workgroup that has
// written its share of range i writes mark to its word of row[i], so that the host sees a range that is there while the next
// is on its way, and the last one without the launch's own end.
struct StageRanges {
    static constexpr int kMax = HostStaging::kSlots + 1;
    int n;
    uint32_t mark;
    uint32_t *done;
    const uint8_t *src[kMax];
    uint8_t *dst[kMax];
    size_t bytes[kMax];
    int row[kMax];
};

__global__ __launch_bounds__(256) void stage_copy_kernel(StageRanges r) {
    for (int i = (int)blockIdx.y; i < r.n; i += (int)gridDim.y) {
        const uint8_t *src = r.src[i];
        uint8_t *dst = r.dst[i];
        const size_t n16 = r.bytes[i] >> 4, stride = (size_t)gridDim.x * 256;
        for (size_t j = (size_t)blockIdx.x * 256 + threadIdx.x; j < n16; j += stride) ((uint4 *)dst)[j] = ((const uint4 *)src)[j];
        const size_t tail = r.bytes[i] & 15;
        if (blockIdx.x == 0 && threadIdx.x < tail) dst[(n16 << 4) + threadIdx.x] = src[(n16 << 4) + threadIdx.x];
        if (r.done) {
            // (each wave's own stores have arrived before the workgroup meets: a barrier alone, and the release of the one thread
            // behind it, wait for no other wave's)
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            if (threadIdx.x == 0)
                __hip_atomic_store(r.done + r.row[i] * kStageWgs + (int)blockIdx.x, r.mark, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
}

// Workgroups for ranges that are copied side by side: 4 KB each (one 16-byte load per lane: a load over PCIe takes about 2 us,
// so what counts is how many are in flight), at most 64 - from there on the link is full (393 KB: 41 us with 4 workgroups, 20 with
// 16 or 64).
int stage_wgs(const StageRanges &r) {
    size_t most = 1;
    for (int i = 0; i < r.n; i++) most = r.bytes[i] > most ? r.bytes[i] : most;
    const size_t want = (most + 4095) / 4096;
    return (int)(want < kStageWgs ? want : kStageWgs);
}
hipError_t launch_stage_copy(const StageRanges &r, int wgs, int side_by_side, hipStream_t s) {
    launch_kernel(stage_copy_kernel, dim3((unsigned)wgs, (unsigned)side_by_side), dim3(256), 0, s, r);
    return hipGetLastError();
}
// ... that are handed on one after the other: half the workgroups each for two of them, so that one is on its way while the
// other waits for its last bytes to be there.
constexpr int kChunkWgs = kStageWgs / 2;

size_t round16(size_t n) { return (n + 15) & ~(size_t)15; }

}  // namespace

struct HostStaging::Slab {
    uint8_t *base = nullptr;   // [in slots | out slots | early | done words]
    uint32_t mark = 0;         // of the last launch: no row's words hold the next one
    struct Row {
        uint32_t mark = 0;     // what the row's words will hold, and how many of them
        int wgs = 0;
    } rows[StageRanges::kMax];
    uint8_t *in(int i) const { return base + (size_t)i * kSlot; }
    uint8_t *out(int i) const { return base + (size_t)(kSlots + i) * kSlot; }
    uint8_t *early() const { return base + 2 * kSlots * kSlot; }
    uint32_t *done() const { return (uint32_t *)(early() + kEarlyMax); }

    static Slab *make() {
        Slab *s = new Slab();
        const size_t words = sizeof(uint32_t) * StageRanges::kMax * kStageWgs;
        // (coherent: the words are read while the launch that writes them runs)
        if (hipHostMalloc((void **)&s->base, 2 * kSlots * kSlot + kEarlyMax + words, hipHostMallocCoherent) == hipSuccess) {
            memset(s->done(), 0, words);
            return s;
        }
        (void)hipGetLastError();
        delete s;
        return nullptr;
    }
    void free() {
        (void)hipHostFree(base);
        delete this;
    }
};

SlabPool<HostStaging::Slab> &HostStaging::pool() {
    static auto *p = new SlabPool<Slab>();  // (never destroyed: handles may outlive static objects)
    return *p;
}

void HostStaging::retain() { pool().retain(); }
void HostStaging::release() { pool().release(); }

HostStaging::HostStaging() { slab_ = pool().take(); }

HostStaging::~HostStaging() {
    if (!slab_) return;
    if (in_flight_) (void)hipStreamSynchronize(pending_);  // (a call that failed half way)
    pool().give(slab_);
}

hipError_t HostStaging::upload(void *dev, const void *host, size_t bytes, hipStream_t s) {
    pending_ = s;
    for (size_t at = 0; at < bytes; at += kSlot) {
        if (used_in_ == kSlots) {  // every slot is on its way: wait for them all (once per 4 MB)
            const hipError_t e = finish(s);
            if (e != hipSuccess) return e;
        }
        const size_t n = bytes - at < kSlot ? bytes - at : kSlot;
        uint8_t *slot = slab_->in(used_in_++);
        memcpy(slot, (const uint8_t *)host + at, n);
        StageRanges r{};
        r.n = 1;
        r.src[0] = slot;
        r.dst[0] = (uint8_t *)dev + at;
        r.bytes[0] = n;
        in_flight_ = true;
        const hipError_t e = launch_stage_copy(r, stage_wgs(r), 1, s);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t HostStaging::finish(hipStream_t s) {
    const hipError_t e = hipStreamSynchronize(s);
    in_flight_ = false;
    used_in_ = 0;
    return e;
}

void *HostStaging::out_direct(size_t bytes) const { return slab_ && bytes <= kSlot ? slab_->out(0) : nullptr; }

const void *HostStaging::early_host() const { return slab_->early(); }

HostStaging::Chunk HostStaging::chunk_at(int i) const {
    for (int p = 0; p < n_pieces_; p++) {
        const int here = (int)((piece_[p].bytes + kSlot - 1) / kSlot);
        if (i < here) {
            const size_t at = (size_t)i * kSlot, left = piece_[p].bytes - at;
            return {(uint8_t *)piece_[p].host + at, (const uint8_t *)piece_[p].dev + at, left < kSlot ? left : kSlot};
        }
        i -= here;
    }
    return {nullptr, nullptr, 0};
}

// Waits for the words of a row.  They are written within microseconds of the work ahead of them; after a while the stream
// is asked (a launch that failed writes none), then waited for.
hipError_t HostStaging::wait_row(int row, hipStream_t s) {
    const Slab::Row &want = slab_->rows[row];
    const uint32_t *words = slab_->done() + row * kStageWgs;
    auto there = [&] {
        for (int i = 0; i < want.wgs; i++)
            if (__atomic_load_n(words + i, __ATOMIC_ACQUIRE) != want.mark) return false;
        return true;
    };
    for (int look = 0; look < (1 << 14); look++) {
        if (there()) return hipSuccess;
        __builtin_ia32_pause();
        if ((look & 0xFFF) == 0xFFF) {
            const hipError_t e = hipStreamQuery(s);
            if (e == hipSuccess) break;
            (void)hipGetLastError();
            if (e != hipErrorNotReady) return e;
        }
    }
    const hipError_t e = hipStreamSynchronize(s);
    return e != hipSuccess ? e : (there() ? hipSuccess : hipErrorUnknown);
}

hipError_t HostStaging::launch_out(const void *ranges, int wgs, int side_by_side, hipStream_t s) {
    StageRanges r = *(const StageRanges *)ranges;
    r.done = slab_->done();
    r.mark = ++slab_->mark;
    for (int i = 0; i < r.n; i++) {
        slab_->rows[r.row[i]].mark = r.mark;
        slab_->rows[r.row[i]].wgs = wgs;
    }
    return launch_stage_copy(r, wgs, side_by_side, s);
}

// Rows of done words: 0 for the early bytes, 1 + slot for what lies in an output slot (a small read-back: 1 + piece).
hipError_t HostStaging::enqueue_out(int from, int to, const void *early, size_t early_bytes, hipStream_t s) {
    StageRanges r{};
    if (early) {
        r.src[0] = (const uint8_t *)early;
        r.dst[0] = slab_->early();
        r.bytes[0] = early_bytes;
        r.row[r.n++] = 0;
    }
    for (int c = from; c < to && c < n_chunks_; c++) {
        const Chunk ch = chunk_at(c);
        r.src[r.n] = ch.dev;
        r.dst[r.n] = slab_->out(c % kSlots);
        r.bytes[r.n] = ch.bytes;
        r.row[r.n++] = 1 + c % kSlots;
    }
    return r.n == 0 ? hipSuccess : launch_out(&r, kChunkWgs, 2, s);
}

hipError_t HostStaging::begin_download(const Piece *pieces, int n, const void *early, size_t early_bytes, hipStream_t s) {
    pending_ = s;
    in_flight_ = true;
    n_pieces_ = n;
    n_chunks_ = 0;
    size_t total = 0;
    for (int i = 0; i < n; i++) {
        piece_[i] = pieces[i];
        total += round16(pieces[i].bytes);
        n_chunks_ += (int)((pieces[i].bytes + kSlot - 1) / kSlot);
    }
    small_ = total <= kSlot;
    hipError_t e;
    if (small_) {
        StageRanges r{};
        if (early) {
            r.src[0] = (const uint8_t *)early;
            r.dst[0] = slab_->early();
            r.bytes[0] = early_bytes;
            r.row[r.n++] = 0;
        }
        size_t at = 0;
        for (int i = 0; i < n; i++) {
            r.src[r.n] = (const uint8_t *)pieces[i].dev;
            r.dst[r.n] = slab_->out(0) + at;
            r.bytes[r.n] = pieces[i].dev == slab_->out(0) ? 0 : pieces[i].bytes;   // (out_direct: the one piece)
            r.row[r.n++] = 1 + i;
            at += round16(pieces[i].bytes);
        }
        e = launch_out(&r, stage_wgs(r), r.n, s);
    } else {
        e = enqueue_out(0, kSlots, early, early_bytes, s);
    }
    // While the GPU is at work: pages of the caller's memory that were never written to are given to it now (a fresh array of
    // 2.4 MB has 600: the first forward of 300 tokens 520 -> 485 us).  What is there stays as it is.
    for (int i = 0; i < n && e == hipSuccess; i++)
        for (size_t at = 0; at < pieces[i].bytes; at += 4096) (void)__atomic_fetch_or((uint8_t *)pieces[i].host + at, 0, __ATOMIC_RELAXED);
    return e != hipSuccess || !early ? e : wait_row(0, s);
}

hipError_t HostStaging::finish_download(hipStream_t s) {
    hipError_t e = hipSuccess;
    if (small_) {
        size_t at = 0;
        for (int i = 0; i < n_pieces_; i++) {
            if ((e = wait_row(1 + i, s)) != hipSuccess) return e;
            memcpy(piece_[i].host, slab_->out(0) + at, piece_[i].bytes);
            at += round16(piece_[i].bytes);
        }
    } else {
        constexpr int kHalf = kSlots / 2;
        for (int c = 0; c < n_chunks_; c++) {
            if ((e = wait_row(1 + c % kSlots, s)) != hipSuccess) return e;
            const Chunk ch = chunk_at(c);
            memcpy(ch.host, slab_->out(c % kSlots), ch.bytes);
            // (half the slots are empty: the chunks after the ones under way)
            if (c % kHalf == kHalf - 1 && (e = enqueue_out(c + 1 + kHalf, c + 1 + kSlots, nullptr, 0, s)) != hipSuccess) return e;
        }
    }
    // All bytes are here, and with them everything ahead of them on the stream is done: the slab is free without a wait for
    // the launch's own end.
    in_flight_ = false;
    used_in_ = 0;
    return hipSuccess;
}

}  // namespace mummu
