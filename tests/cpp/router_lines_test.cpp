// Which calls of the router's logits take the matrix units: many workgroups of 16 tokens by 64 experts, and experts in two thirds of their columns.  Which of the logits with the
// routing behind: 33 to 64 experts, fewer than 57 of them only where the streaming form has two tokens to a wave or does not take the rows.
#include <cstdio>

#include "router_lines.h"

int main() {
    const struct {
        int n, experts;
        bool matrix;
    } cases[] = {
        // as many workgroups as the line asks for, on either side of it
        {1024, 128, false}, {1025, 128, true}, {2048, 64, false}, {2049, 64, true}, {256, 512, false}, {257, 512, true}, {4096, 512, true}, {9, 512, false},
        // columns that are mostly empty: the tiles of four by four cost what their experts are
        {2049, 8, false}, {4096, 8, false}, {4096, 16, false}, {4096, 32, false}, {1 << 20, 32, false}, {1041, 65, false}, {2049, 72, false}, {4096, 80, false},
        // ... and in two thirds of them
        {4096, 42, false}, {4096, 43, true}, {4096, 85, false}, {4096, 86, true}, {4096, 96, true}, {4096, 129, true}, {1 << 30, 512, true},
    };
    int bad = 0;
    for (const auto &c : cases)
        if (mummu::router_matrix_should(c.n, c.experts) != c.matrix) {
            std::printf("%d tokens, %d experts\n", c.n, c.experts);
            bad++;
        }
    const struct {
        int n, experts, hidden;
        bool matrix;
    } routes[] = {
        {1024, 64, 2048, false}, {1025, 64, 2048, true}, {1025, 57, 512, true}, {1025, 56, 2048, false}, {1025, 33, 2048, false}, {2048, 33, 512, false}, {2048, 48, 2048, false},
        {2048, 56, 1536, false}, {2049, 56, 2048, true}, {2049, 33, 2048, true}, {4096, 32, 2048, false}, {4096, 65, 2048, false}, {1024, 33, 2560, false}, {1025, 33, 2560, true},
        {1025, 64, 4096, true}, {4096, 32, 4096, false},
    };
    for (const auto &c : routes)
        if (mummu::router_matrix_routes(c.n, c.experts, c.hidden) != c.matrix) {
            std::printf("routes: %d tokens, %d experts, %d elements\n", c.n, c.experts, c.hidden);
            bad++;
        }
    if (bad) std::printf("router lines: %d wrong\n", bad);
    else std::printf("router lines: ok\n");
    return bad != 0;
}
