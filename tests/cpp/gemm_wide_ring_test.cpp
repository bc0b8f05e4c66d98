// The wide GEMM's stages in LDS (gemm_wide_ring.h), walked as one of its waves does, over items of every height behind every other: each stage is asked for
// once (of two steps with the weights a step ahead the second: twice), has landed when the barrier in front of its products opens, and nothing is on its way into a place that may be read.
#include <cstdio>
#include <deque>
#include <map>

#include "gemm_wide_ring.h"

using namespace mummu::wide;

static int bad = 0;
static void wrong(const char *what, int mw, int steps, int step) {
    if (bad++ < 10) std::printf("%s: %d rows, %d steps, step %d\n", what, 64 * mw, steps, step);
}

// A load of a stage (rows or weights) or a store (stage -1).
struct Op {
    bool weights;
    int stage;
};

static std::deque<Op> queue;   // what is under way, the oldest first
static void wait(int left) {
    while ((int)queue.size() > left) queue.pop_front();
}
static bool under_way(bool weights, int stage) {
    for (const Op &o : queue)
        if (o.weights == weights && o.stage == stage) return true;
    return false;
}

static void begin(int mw, std::map<int, int> &asked) {
    for (int s = 0; s < kBegun; s++) {
        for (int i = 0; i < kLoadsB; i++) queue.push_back({true, s});
        asked[s]++;
        for (int i = 0; i < mw; i++) queue.push_back({false, s});
    }
}

// One item; `behind` as in the kernel, `next`: the height of the one after it (0: none).
template <int MW>
static void item(int steps, int behind, int next, std::map<int, int> &asked_b) {
    using R = Ring<MW>;
    for (int step = 0; step < steps; step++) {
        const int left = steps - 1 - step < 2 ? steps - 1 - step : 2;
        const bool first = step == 0 && steps > 2;
        // beside the first products, which read the weights of this stage's second half and its rows
        if (asks_weights(R::kAhead, left, first)) {
            const int s = step + R::kAhead;
            if (s >= steps) wrong("a stage past the last", MW, steps, step);
            if (s % R::kB == step % R::kB) wrong("weights into the place that is read", MW, steps, step);
            for (int i = 0; i < kLoadsB; i++) queue.push_back({true, s});
            asked_b[s]++;
        }
        // the barrier, behind which the next stage is read, and this one's place of rows is free
        wait(step_wait(R::kAhead, left, first ? behind : 0));
        if (left > 0) {
            if (under_way(true, step + 1) || under_way(false, step + 1)) wrong("a stage that has not landed", MW, steps, step);
            if (asked_b[step + 1] != (R::kAhead == 1 && steps == 2 ? 2 : 1)) wrong("a stage asked for not once", MW, steps, step);
        }
        for (const Op &o : queue)   // (weights two stages on lie in the third place, rows in the place of this step's)
            if (o.weights && o.stage >= 0 && left > 0 && o.stage % R::kB == (step + 1) % R::kB) wrong("under way into the next stage's place", MW, steps, step);
        if (left == 2)
            for (int i = 0; i < MW; i++) queue.push_back({false, step + 2});
    }
    for (const Op &o : queue)
        if (o.stage >= 0) wrong("a load left behind an item", MW, steps, steps - 1);
    asked_b.clear();
    if (next > 0) begin(next, asked_b);
    for (int i = 0; i < kStoresOfUnit * MW; i++) queue.push_back({false, -1});
    wait(begin_wait(MW));
    if (next > 0 && (under_way(true, 0) || under_way(false, 0))) wrong("an item's first stage has not landed", next, steps, 0);
}

static void any_item(int mw, int steps, int behind, int next, std::map<int, int> &asked) {
    switch (mw) {
    case 1: item<1>(steps, behind, next, asked); break;
    case 2: item<2>(steps, behind, next, asked); break;
    case 3: item<3>(steps, behind, next, asked); break;
    case 4: item<4>(steps, behind, next, asked); break;
    default: item<5>(steps, behind, next, asked); break;
    }
}

int main() {
    for (int steps = 2; steps <= 9; steps++)
        for (int a = 1; a <= 5; a++)
            for (int b = 0; b <= 5; b++)
                for (int c = 0; c <= (b ? 5 : 0); c++) {
                    queue.clear();
                    std::map<int, int> asked;
                    begin(a, asked);
                    wait(begin_wait(0));
                    if (under_way(true, 0) || under_way(false, 0)) wrong("the first stage has not landed", a, steps, 0);
                    any_item(a, steps, 0, b, asked);
                    if (b) any_item(b, steps, a, c, asked);
                    if (c) any_item(c, steps, b, 0, asked);
                }
    static_assert(Ring<5>::kAtA + 2 * Ring<5>::kStageA + 4 <= kWLds, "a word behind the stages of the highest tiles");
    if (bad) std::printf("wide ring: %d wrong\n", bad);
    else std::printf("wide ring: ok\n");
    return bad != 0;
}
