// The pool that host calls borrow their pinned slabs from (mummu_amd/csrc/slab_pool.h): rounds of calls side by side, one per
// handle, allocate a slab each in the first round and none afterwards, free none while the handles live, and leave none
// behind.
#include <atomic>
#include <cstdio>
#include <thread>
#include <vector>

#include "slab_pool.h"

static std::atomic<int> made{0}, freed{0};
static bool refuse = false;

struct Slab {
    static Slab *make() {
        if (refuse) return nullptr;
        made++;
        return new Slab();
    }
    void free() {
        freed++;
        delete this;
    }
};

static int failures = 0;
static void expect(const char *what, int got, int want) {
    if (got == want) return;
    failures++;
    printf("%s: %d, expected %d\n", what, got, want);
}

int main() {
    mummu::SlabPool<Slab> pool;
    for (int handles : {1, 4, 5, 12}) {
        made = freed = 0;
        for (int i = 0; i < handles; i++) pool.retain();
        expect("slabs before the first call", made, 1);
        for (int round = 0; round < 20; round++) {
            std::vector<Slab *> held;
            for (int i = 0; i < handles; i++) held.push_back(pool.take());
            for (Slab *s : held) pool.give(s);
        }
        expect("slabs made by calls side by side", made, handles);
        expect("slabs freed by calls", freed, 0);
        // the same from threads of their own
        std::vector<std::thread> threads;
        for (int i = 0; i < handles; i++)
            threads.emplace_back([&] {
                for (int round = 0; round < 1000; round++) pool.give(pool.take());
            });
        for (std::thread &t : threads) t.join();
        expect("slabs made, threads", made, handles);
        expect("slabs freed, threads", freed, 0);
        // handles that go take what is idle beyond the rest with them; a slab on its way comes back to fewer
        if (handles > 1) {
            Slab *out = pool.take();
            for (int i = 1; i < handles; i++) pool.release();
            expect("slabs freed with all handles but one", freed, handles - 2);
            pool.give(out);
            expect("... and the one that came back too late", freed, handles - 1);
        }
        pool.release();
        expect("slabs freed in the end", freed, made);
    }
    // no memory to be had: no slab, and nothing to give back
    refuse = true;
    pool.retain();
    expect("a slab without memory", pool.take() != nullptr, 0);
    pool.release();
    if (!failures) printf("slab pool: ok\n");
    return failures != 0;
}
