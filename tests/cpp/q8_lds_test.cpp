// Every address at which gemm_q8.hip reads rows from LDS: inside the stage it is meant for, hence inside the workgroup's LDS, and on
// the element it is meant for.
#include <cstdio>
#include <initializer_list>

#include "gemm_q8_lds.h"

using namespace mummu::q8;

int main() {
    int bad = 0;
    for (int which = 0; which < 2; which++)
        for (int few = 0; few < 2; few++)
            for (int lane = 0; lane < 64; lane++)
                for (int blk = 0; blk < kBlocks; blk++)
                    for (int kk = 0; kk < 2; kk++) {
                        const int c = lane & 31, g = lane >> 5, row = few ? c & 15 : c, q = 4 * blk + 2 * g + kk;
                        const uint32_t stage = rows_at(which), hi = row_read(c, few != 0) + row_piece(c, g, blk, kk), lo = hi + row_low(few != 0);
                        for (uint32_t at : {stage + hi, stage + lo})   // (both are read ahead, whatever the item's kind)
                            if (at % 16 != 0 || at < stage || at + 16 > stage + kStageA || at + 16 > (uint32_t)kLdsBytes) bad++;
                        // (piece q of row r lies at q ^ (r % 16) of the row, the low halfs' plane behind the high ones')
                        const uint32_t place = (uint32_t)(row * kStep * 2 + (q ^ (row & 15)) * 16);
                        if (hi != place + (few && c >= 16 ? kPlane : 0)) bad++;
                        if (!few && lo != place + kPlane) bad++;
                    }
    if (kLdsBytes > 160 * 1024 - 2 * 2 * 64 * 4) bad++;   // (beside it: two scales and two entries of `sorted` a lane)
    if (bad) std::printf("q8 lds: %d reads out of place\n", bad);
    else std::printf("q8 lds: ok\n");
    return bad != 0;
}
