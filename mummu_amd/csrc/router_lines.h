// Which calls take the router's matrix form (router_matrix.hip): plain C++, so that a test on the host can ask.
#pragma once

namespace mummu {

// The logits of n tokens: from 128 workgroups of 16 tokens by 64 experts on, whose one round takes 21 to 24 us whatever their number (2048 elements, more in
// proportion), which is what router_tile_kernel takes for as many: us of that / of the matrix units, a launch among those of its layer, 128 experts of 2048, 600 tokens
// 14 / 21 (76 workgroups), 1025: 23 / 21, 2000: 38 / 24, 4096: 61 / 44; 512 experts of 2560, 150 tokens 14 / 23 (80), 300: 26 / 25 (152), 1024: 65 / 48.
// ... while experts fill two thirds of the tiles' columns: a round takes the same for a tile with one expert in it, router_tile_kernel what its experts are.
// Calls of the routing alone, 2048 elements (between two copies, a tenth more than in a layer): 8 experts 2049 / 4096 tokens 10 / 26, 16 / 28; 16: 11 / 26, 17 / 28; 32: 16 / 26, 27 / 30; 48: 22 / 25,
// 36 / 31; 65 at 1025 / 2049 / 4096 tokens 17 / 25, 29 / 46, 44 / 51; 80: 18 / 25, 30 / 46, 48 / 52; 96: 21 / 25, 35 / 46, 54 / 51.  Layers of 2048 x 768, among others and (alone),
// where the matrix units leave other streams some of the chip: 72 experts, 2049 tokens 408 / 403 (438 / 451), 3000: 581 / 578 (609 / 617), 4096: 766 / 769 (790 / 796); 96
// experts 2049: 422 / 410 (453 / 463), 3000: 594 / 588 (621 / 622), 4096: 781 / 783 (804 / 799).
inline bool router_matrix_should(int n, int n_experts) {
    const long long columns = (n_experts + 63) / 64;
    return (long long)((n + 15) / 16) * columns > 128 && 3LL * n_experts >= 2 * 64 * columns;
}

// The logits and the routing of n tokens in one launch, of up to 64 experts (a tile's columns want more than 32).  Rows of up to 2048 elements, which router_stream_kernel
// takes: 16 tokens to a workgroup, one round of which takes 25 to 29 us up to 4096 tokens (2048 elements; 13, 17, 21 us for 512, 1024, 1536), the streaming form what its experts are,
// and half of that again where it goes over to two tokens a wave, above 2048.  us of that / of the matrix units, a launch among those of its layer, 1025 / 2048 / 2100 / 4096 tokens: 33
// experts 13 / 25, 17 / 25, 25 / 25, 28 / 28; 48: 17 / 25, 22 / 26, 33 / 26, 36 / 29; 56: 19 / 26, 24 / 26, 37 / 26, 39 / 28; 64: 21 / 25, 27 / 26, 41 / 26, 45 / 29.  Layers of 2048 x 512 f16 banks
// on their own and (among others, which have the CUs that a round leaves): 33 experts, 1025 tokens 164 / 176 (121 / 123), 2048: 258 / 264 (227 / 228); 48: 176 / 185 (135 / 132), 264 / 270
// (242 / 240); 56: 164 / 173 (123 / 117), 231 / 233 (209 / 198); 57, 60 and 64 experts are 2, 7 and 0 us slower on their own at 1025, within 3 from 1536 on, and 5 to 12 faster among others.
// Longer rows have launch_router_block instead: 2560 elements, 1025 / 4096 tokens 196 / 28, 711 / 33; 4096: 291 / 40, 1066 / 49, 33 experts or 64.
inline bool router_matrix_routes(int n, int n_experts, int hidden) {
    return n_experts > 32 && n_experts <= 64 && n > (hidden <= 2048 && n_experts <= 56 ? 2048 : 1024);
}

}  // namespace mummu
