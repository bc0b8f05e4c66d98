// Objects that calls borrow one at a time, kept between the calls.
#pragma once

#include <mutex>
#include <vector>

namespace mummu {

// Slab::make() allocates one (null if it cannot), free() gives it back.  A handle serves one call at a time, so calls under way
// never hold more slabs than there are handles, and the pool keeps that many: a call allocates only where more calls run side by
// side than ever before, and none frees.  (With a bound of four, every call beyond it allocated 8.4 MB of pinned memory and
// freed it behind a wait for the device.)  A slab too many is freed when a handle goes, the last with the last handle.
template <typename Slab>
class SlabPool {
public:
    void retain() {
        {
            std::lock_guard<std::mutex> lock(mu_);
            if (handles_++ > 0 || !idle_.empty()) return;
        }
        if (Slab *first = take()) give(first);  // the first handle's creation pays for the slab, not its first call
    }
    void release() {
        std::vector<Slab *> gone;
        {
            std::lock_guard<std::mutex> lock(mu_);
            handles_--;
            while ((int)idle_.size() > handles_) {
                gone.push_back(idle_.back());
                idle_.pop_back();
            }
        }
        for (Slab *s : gone) s->free();
    }
    Slab *take() {
        {
            std::lock_guard<std::mutex> lock(mu_);
            if (!idle_.empty()) {
                Slab *s = idle_.back();
                idle_.pop_back();
                return s;
            }
        }
        return Slab::make();
    }
    void give(Slab *s) {
        {
            std::lock_guard<std::mutex> lock(mu_);
            if ((int)idle_.size() < handles_) {
                idle_.push_back(s);
                return;
            }
        }
        s->free();
    }

private:
    std::mutex mu_;
    std::vector<Slab *> idle_;
    int handles_ = 0;
};

}  // namespace mummu
