// Pinned staging of host rows (see host_staging.h).
#include "host_staging.h"

#include <cstring>
#include <mutex>
#include <vector>

#include "device_utils.h"

namespace mummu {

namespace {

// Up to four byte ranges copied by one launch (blockIdx.y picks the range), 16 bytes per lane and step; either side may
// be pinned host memory.  Both pointers of a range are 16-byte aligned.
struct StageRanges {
    const uint8_t *src[4];
    uint8_t *dst[4];
    size_t bytes[4];
};

__global__ __launch_bounds__(256) void stage_copy_kernel(StageRanges r) {
    const int i = blockIdx.y;
    const uint8_t *src = r.src[i];
    uint8_t *dst = r.dst[i];
    const size_t n16 = r.bytes[i] >> 4, stride = (size_t)gridDim.x * 256;
    for (size_t j = (size_t)blockIdx.x * 256 + threadIdx.x; j < n16; j += stride) ((uint4 *)dst)[j] = ((const uint4 *)src)[j];
    const size_t tail = r.bytes[i] & 15;
    if (blockIdx.x == 0 && threadIdx.x < tail) dst[(n16 << 4) + threadIdx.x] = src[(n16 << 4) + threadIdx.x];
}

// Workgroups per range: 4 KB each (one 16-byte load per lane: a load over PCIe takes about 2 us, so what counts is how
// many are in flight), at most 64 - from there on the link is full (393 KB: 41 us with 4 workgroups, 20 with 16 or 64).
hipError_t launch_stage_copy(const StageRanges &r, int n, hipStream_t s) {
    size_t most = 1;
    for (int i = 0; i < n; i++) most = r.bytes[i] > most ? r.bytes[i] : most;
    const size_t want = (most + 4095) / 4096;
    launch_kernel(stage_copy_kernel, dim3((unsigned)(want < 64 ? want : 64), (unsigned)n), dim3(256), 0, s, r);
    return hipGetLastError();
}

size_t round16(size_t n) { return (n + 15) & ~(size_t)15; }

}  // namespace

struct HostStaging::Slab {
    uint8_t *base = nullptr;   // [in slots | out slots | early]
    hipEvent_t done[kSlots] = {};
    uint8_t *in(int i) const { return base + (size_t)i * kSlot; }
    uint8_t *out(int i) const { return base + (size_t)(kSlots + i) * kSlot; }
    uint8_t *early() const { return base + 2 * kSlots * kSlot; }

    static Slab *make() {
        Slab *s = new Slab();
        bool ok = hipHostMalloc((void **)&s->base, 2 * kSlots * kSlot + kEarlyMax, hipHostMallocDefault) == hipSuccess;
        for (int i = 0; i < kSlots && ok; i++) ok = hipEventCreateWithFlags(&s->done[i], hipEventDisableTiming) == hipSuccess;
        if (ok) return s;
        (void)hipGetLastError();
        s->free();
        return nullptr;
    }
    void free() {
        for (hipEvent_t e : done)
            if (e) (void)hipEventDestroy(e);
        if (base) (void)hipHostFree(base);
        delete this;
    }
};

struct HostStaging::Pool {
    std::mutex mu;
    std::vector<Slab *> idle;
    int handles = 0;
};

HostStaging::Pool &HostStaging::pool() {
    static Pool *p = new Pool();  // (never destroyed: handles may outlive static objects)
    return *p;
}

void HostStaging::retain() {
    {
        Pool &p = pool();
        std::lock_guard<std::mutex> lock(p.mu);
        if (p.handles++ > 0 || !p.idle.empty()) return;
    }
    HostStaging first;  // the first handle's creation pays for the slab, not its first call
}

void HostStaging::release() {
    std::vector<Slab *> gone;
    {
        Pool &p = pool();
        std::lock_guard<std::mutex> lock(p.mu);
        if (--p.handles == 0) gone.swap(p.idle);
    }
    for (Slab *s : gone) s->free();
}

HostStaging::HostStaging() {
    {
        Pool &p = pool();
        std::lock_guard<std::mutex> lock(p.mu);
        if (!p.idle.empty()) {
            slab_ = p.idle.back();
            p.idle.pop_back();
        }
    }
    if (!slab_) slab_ = Slab::make();
}

HostStaging::~HostStaging() {
    if (!slab_) return;
    if (in_flight_) (void)hipStreamSynchronize(pending_);  // (a call that failed half way)
    {
        Pool &p = pool();
        std::lock_guard<std::mutex> lock(p.mu);
        if (p.handles > 0 && (int)p.idle.size() < kMaxIdle) {
            p.idle.push_back(slab_);
            slab_ = nullptr;
        }
    }
    if (slab_) slab_->free();
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
        r.src[0] = slot;
        r.dst[0] = (uint8_t *)dev + at;
        r.bytes[0] = n;
        in_flight_ = true;
        const hipError_t e = launch_stage_copy(r, 1, s);
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

hipError_t HostStaging::enqueue_out(int chunk, hipStream_t s) {
    const Chunk c = chunk_at(chunk);
    StageRanges r{};
    r.src[0] = c.dev;
    r.dst[0] = slab_->out(chunk % kSlots);
    r.bytes[0] = c.bytes;
    const hipError_t e = launch_stage_copy(r, 1, s);
    return e != hipSuccess ? e : hipEventRecord(slab_->done[chunk % kSlots], s);
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
    StageRanges r{};
    int nr = 0;
    if (early) {
        r.src[nr] = (const uint8_t *)early;
        r.dst[nr] = slab_->early();
        r.bytes[nr++] = early_bytes;
    }
    if (small_) {
        size_t at = 0;
        for (int i = 0; i < n; i++) {
            r.src[nr] = (const uint8_t *)pieces[i].dev;
            r.dst[nr] = slab_->out(0) + at;
            r.bytes[nr++] = pieces[i].bytes;
            at += round16(pieces[i].bytes);
        }
        const hipError_t e = launch_stage_copy(r, nr, s);
        return e != hipSuccess ? e : finish(s);
    }
    hipError_t e = nr ? launch_stage_copy(r, nr, s) : hipSuccess;
    for (int c = 0; c < n_chunks_ && c < kSlots && e == hipSuccess; c++) e = enqueue_out(c, s);
    return e != hipSuccess ? e : hipEventSynchronize(slab_->done[0]);  // (the early bytes came before chunk 0)
}

hipError_t HostStaging::finish_download(hipStream_t s) {
    if (small_) {
        size_t at = 0;
        for (int i = 0; i < n_pieces_; i++) {
            memcpy(piece_[i].host, slab_->out(0) + at, piece_[i].bytes);
            at += round16(piece_[i].bytes);
        }
        return hipSuccess;
    }
    for (int c = 0; c < n_chunks_; c++) {
        hipError_t e = hipEventSynchronize(slab_->done[c % kSlots]);
        if (e != hipSuccess) return e;
        const Chunk ch = chunk_at(c);
        memcpy(ch.host, slab_->out(c % kSlots), ch.bytes);
        if (c + kSlots < n_chunks_ && (e = enqueue_out(c + kSlots, s)) != hipSuccess) return e;
    }
    return finish(s);
}

}  // namespace mummu
