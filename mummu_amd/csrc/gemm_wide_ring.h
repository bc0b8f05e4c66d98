// The stages of the wide GEMM (gemm_wide.hip) in LDS, what its waves ask for when, and how many of their loads and stores may be under way when a step's barrier
// lets the next stage be read: plain C++, so that a test on the host can walk it.
#pragma once

namespace mummu {
namespace wide {

constexpr int kWK = 64;                          // K elements of a stage: a line of 128 bytes per row, eight pieces of 16
constexpr int kWCols = 256;                      // weight rows of a tile
constexpr int kWStageB = kWCols * kWK * 2;       // bytes of a stage of weights
// Stages in LDS, for tiles of 64 MW rows: of the weights, then two of the activations.
template <int MW>
struct Ring {
    static constexpr int kB = MW <= 4 ? 3 : 2, kStageA = 64 * MW * kWK * 2, kAtA = kB * kWStageB;
    static constexpr int kAhead = kB - 1;   // a step asks for the weights of so many steps on
    static_assert(kAtA + 2 * kStageA <= 160 * 1024, "the stages fit the LDS");
};
constexpr int kWLds = Ring<4>::kAtA + 2 * Ring<4>::kStageA;

// An item's start asks for its first two stages, rows (MW loads of a wave each) and weights (four each).
constexpr int kBegun = 2, kLoadsB = 4, kStoresOfUnit = 8;   // (and its end makes 8 MW stores)

// Whether a step, `left` steps (2: or more) in front of the item's last, asks for the weights of `ahead` steps on.  first: the first of three steps or more, where the
// item's start has asked for the next one's: a second copy would not have landed behind the barrier that counts the first (step_wait), under the reads of it.  (The
// first of two, a step ahead, asks for them again; its barrier waits for everything.  Left out there by a condition in the item's start, the loop lost a register
// that it then waited for: 4096 rows of bf16 503 -> 513 us.)
constexpr bool asks_weights(int ahead, int left, bool first) { return left >= ahead && !(ahead == 1 && first); }

// The loads and stores of a wave that may be under way at a step's barrier, behind which the next step's stage is read.  behind: in an item's first step of three
// or more, the height (in 64 rows) of the item before, whose stores stand behind the stage that is waited for; else 0.
constexpr int step_wait(int ahead, int left, int behind) {
    if (left == 0) return ahead == 2 ? 63 : 0;
    if (behind > 0) return kStoresOfUnit * behind;
    return ahead == 2 && left == 2 ? kLoadsB : 0;
}
// ... in front of an item, whose first stage has landed then: the second one's loads (five or more) and the stores of the item before.
constexpr int begin_wait(int behind) { return kStoresOfUnit * behind + kLoadsB + 1; }

}  // namespace wide
}  // namespace mummu
