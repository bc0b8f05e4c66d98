// Where the workgroups of gemm_q8.hip keep things in LDS, and where their lanes read rows.  Plain C++: a test on the CPU goes through
// every address.
#pragma once

#include <stdint.h>

namespace mummu {
namespace q8 {

constexpr int kRows = 32;                    // rows of a tile
constexpr int kWaves = 8, kWCols = 32 * kWaves;
constexpr int kStep = 128, kBlocks = 4;      // K elements and blocks of a stage
constexpr int kRowW = 136;                   // bytes of a weight row's stage
constexpr int kWLoads = 5;                   // loads of a wave's weights: 64 pieces of 16 bytes each
constexpr int kWaveW = kWLoads * 1024, kStageW = kWaves * kWaveW, kRing = 3;
constexpr int kPlane = kRows * kStep * 2, kStageA = 2 * kPlane;   // hi, lo: [row][16 pieces of 16 bytes]
constexpr int kLdsBytes = kRing * kStageW + 2 * kStageA;          // [kRing][kStageW], then [2][kStageA]

// Stage `which` of the rows.
constexpr uint32_t rows_at(int which) { return (uint32_t)(kRing * kStageW + which * kStageA); }

// Where lane column c reads within a stage: its high halfs at row_read, its low ones row_low behind them.  An item of up to 16 rows has its low
// halfs' rows behind its high halfs' in one operand, which the former is: there is no other, and a read of it stays in the same place (the
// item's end reads ahead whatever kind the next item is; a plane further would be past the second stage, the last thing in LDS).
constexpr uint32_t row_read(int c, bool few) {
    return few ? (uint32_t)((c & 15) * (kStep * 2) + (c >> 4) * kPlane) : (uint32_t)(c * (kStep * 2));
}
constexpr uint32_t row_low(bool few) { return few ? 0u : (uint32_t)kPlane; }

// The piece of a row for product kk of block blk, K group g: piece q of row r lies at q ^ (r % 16), so that sixteen lanes that read the
// same piece of neighbouring rows meet all banks.
constexpr uint32_t row_piece(int c, int g, int blk, int kk) { return (uint32_t)((4 * blk + 2 * g + kk) ^ (c & 15)) * 16u; }

}  // namespace q8
}  // namespace mummu
