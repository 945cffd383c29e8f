// Which of two tilings the brick kernels take on a grid of one z plane; usable
// on the host.
#pragma once
#include <cstdint>

namespace p3d {

// A brick is 4 x 8 x 8 tokens, so a one-plane grid fills one of its four planes.
// In strips the four planes hold four strips of 8 rows instead: up to four times
// fewer workgroups, each of which costs `cost` bricks (one with fewer strips, less
// in proportion).  What counts is how many rounds of 256 compute units either
// takes: `paired` kernels run two workgroups on a unit, and an odd last round,
// one to a unit, costs 1.25.  Fewer than `least` strips are not taken.
constexpr double cu_rounds(int64_t workgroups, bool paired) {
    const int64_t rounds = (workgroups + 255) / 256;
    return (double)rounds + (paired && rounds % 2 ? 0.25 : 0.0);
}

constexpr bool take_strips(int64_t bricks_y, int64_t bricks_x, int64_t planes, double cost, bool paired,
                           int64_t least = 0) {
    const int64_t groups = (bricks_y + 3) / 4, strips = groups * bricks_x * planes;
    const double each = 1.0 + (cost - 1.0) * (double)bricks_y / (double)(4 * groups);
    return strips >= least && cu_rounds(bricks_y * bricks_x * planes, paired) > each * cu_rounds(strips, paired);
}

// Forward attention (64 summaries): a workgroup of four strips costs 2.3 to 2.9
// bricks, 3.4 in bf16 at head_dim 64, whose strips spill 58 registers; more
// summaries, which strips sweep once for four bricks, cost less (1.7 to 2.9 with
// 256).  Bricks / strips in us at 16 x 16 bricks of 16 heads: bf16 83 / 56 (head_dim
// 16), 157 / 106 (48), 159 / 146 (64), 671 / 472 (128); fp32 150 / 91, 364 / 206,
// 642 / 378, 1,636 / 1,085.  At 8 x 8 bricks of 16 heads 29 / 26, 44 / 45, 45 / 60,
// 165 / 100; fp32 44 / 37, 83 / 70, 145 / 86, 390 / 267: bf16 at 64 keeps the bricks
// there.  Head_dim 16, whose workgroups are short, loses as soon as strips leave
// compute units idle (21 / 26 for 672 bricks or 224 workgroups of strips).
constexpr bool strips_forward(int head_dim, bool bf16, int64_t bricks_y, int64_t bricks_x, int64_t planes) {
    return take_strips(bricks_y, bricks_x, planes, bf16 && head_dim == 64 ? 3.4 : 2.75, true, head_dim == 16 ? 256 : 0);
}

// Local backward (dQ and dK/dV together; planes: batch * kv heads): 2.3 to 2.8
// bricks in a 16-bit type, up to 3.2 at head_dim 32 and in fp32, 1.3 at 16-bit
// head_dim 128.  16 x 16 bricks, 16 heads of 4 kv heads: bf16 119 / 88 us (head_dim
// 16), 179 / 124 (48), 195 / 140 (64), 1,101 / 469 (128); fp32 213 / 168, 525 / 402,
// 686 / 502.  8 x 8 bricks, 16 of 8: 40 / 45, 56 / 55, 62 / 62, 294 / 142; fp32
// 66 / 83, 148 / 162, 191 / 203: bricks there, but for head_dim 128.
constexpr bool strips_backward(int head_dim, bool fp32, int64_t bricks_y, int64_t bricks_x, int64_t planes) {
    return take_strips(bricks_y, bricks_x, planes,
                       fp32 || head_dim == 32 ? 3.0 : head_dim >= 128 ? 1.3 : 2.6, false);
}

}  // namespace p3d
