// Host rows to the GPU and back for the entry points that take host pointers.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "slab_pool.h"

namespace mummu {

// One call's way between the caller's pageable memory and the GPU: a slab of pinned memory cut into slots, filled (or
// emptied) by memcpy on the calling thread while a small kernel moves the slots before (or after) it over PCIe.
//
// What bounds it: PCIe, 55 GB/s each way.  memcpy into pinned memory runs at 80 GB/s on the caller's core, so with slots
// of 512 KB it hides behind the transfer: 2.4 MB take 55 us each way, where hipMemcpy from / to pageable memory takes
// 97 us in and 154 us out (393 KB: 20 against 28 us).  Kernels move the bytes, not the copy engines: a transfer by a
// copy engine is handed to and from the compute queue by signals, which costs a call of one token 6 us each way.
//
// What has arrived is marked by the kernel in words that the calling thread watches: an event per slot cost 25 us a slot, the wait
// for the stream's end 4 (expert_run of 96 / 192 / 512 / 1024 Q4_K rows: 135 / 175 / 317 / 596 -> 106 / 155 / 310 / 549 us).
//
// A slab (8.4 MB) belongs to one call at a time.  Slabs come from a pool of the process, which keeps as many as calls have run
// side by side, at most one per handle (slab_pool.h).
class HostStaging {
public:
    static constexpr size_t kSlot = 512 * 1024;
    static constexpr int kSlots = 8;       // each way

    HostStaging();                         // takes a slab; valid() is false if pinned memory cannot be had
    ~HostStaging();                        // hands it back (every transfer has to have been waited for, or is waited for here)
    HostStaging(const HostStaging &) = delete;
    HostStaging &operator=(const HostStaging &) = delete;
    bool valid() const { return slab_ != nullptr; }

    // Enqueues the copy of `bytes` bytes to dev; `host` may be reused when the call returns.
    hipError_t upload(void *dev, const void *host, size_t bytes, hipStream_t s);

    // Where a last kernel can leave `bytes` bytes for the host by itself: given to download() as a piece's `dev`, they are not copied, only
    // marked as there behind everything enqueued before.  Null where they take more than a slot (several are copied and read in
    // turns).  The kernel writes every byte once and reads none of them.
    void *out_direct(size_t bytes) const;

    // Up to kPieces device arrays read back together behind everything enqueued on s.  `early` (nullable) is read back
    // ahead of them: check(early copy) runs before anything is written to the caller's memory, and its non-zero status
    // ends the call (returned through *status).
    struct Piece {
        void *host;
        const void *dev;
        size_t bytes;
    };
    static constexpr int kPieces = 3;
    static constexpr size_t kEarlyMax = 64;
    template <typename F>
    hipError_t download(const Piece *pieces, int n, const void *early, size_t early_bytes, hipStream_t s, F &&check, int *status) {
        *status = 0;
        hipError_t e = begin_download(pieces, n, early, early_bytes, s);
        if (e != hipSuccess) return e;
        if (early && (*status = check(early_host())) != 0) return finish(s);
        return finish_download(s);
    }

    static void retain();    // a handle was made / is gone: the pool holds a slab per handle at most
    static void release();

private:
    struct Slab;
    static SlabPool<Slab> &pool();
    const void *early_host() const;
    hipError_t begin_download(const Piece *pieces, int n, const void *early, size_t early_bytes, hipStream_t s);
    hipError_t finish_download(hipStream_t s);
    hipError_t enqueue_out(int from, int to, const void *early, size_t early_bytes, hipStream_t s);
    hipError_t launch_out(const void *ranges, int wgs, int side_by_side, hipStream_t s);
    hipError_t wait_row(int row, hipStream_t s);
    hipError_t finish(hipStream_t s);

    Slab *slab_ = nullptr;
    int used_in_ = 0;          // input slots whose transfer has been enqueued and not waited for
    hipStream_t pending_ = nullptr;
    bool in_flight_ = false;
    // the read-back under way: chunks of at most kSlot bytes over the pieces, in order
    struct Chunk {
        uint8_t *host;
        const uint8_t *dev;
        size_t bytes;
    };
    Piece piece_[kPieces];
    int n_pieces_ = 0, n_chunks_ = 0;
    bool small_ = false;       // everything fits one slot: all pieces side by side
    Chunk chunk_at(int i) const;
};

}  // namespace mummu
