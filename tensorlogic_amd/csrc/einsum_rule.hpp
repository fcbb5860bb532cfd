// einsum_rule.hpp -- which kernel the attention einsums take (plain C++).
#pragma once

#include <cstdint>

namespace tlhip {

// Scores on the matrix cores from 2^16 outputs on.  Up to there the 8-lane
// kernel takes about the launch floor (3.2 - 4.0 us); the other, whose waves
// each load 96 whole rows first, takes 3.4 at head dim 64 and up to 5.0 at 128.
// Beyond, 8-lane / matrix cores: 8 heads of 128, 16 x 129 4.5 / 3.4 us; 33 x
// 1000 keys of 2 heads of 128 4.5 / 4.6, 64 x 1000 6.5 / 5.0; 400 x 400, 32 heads
// of 64 137 / 10.
constexpr bool scores_mfma_wins(int64_t I, int64_t H, int64_t J) { return I >= 16 && J >= 16 && I * H * J >= 1 << 16; }

// Context: the 8-lane kernel has a workgroup per row (i, h) and the matrix-core
// one a workgroup per 32 rows of a head, whose 4 waves walk the keys 128 a
// step.  So the one is bound by its rows (past 512 of them, two workgroups per
// CU, by rounds) and the other, up to 256 workgroups, by the key walk alone:
// 2 heads of 128 over 8000 keys, 16 rows each, take 55 / 117 us, 32 heads of 64
// over 400 keys 4.7 / 5.6 us at 16 rows, 6.3 / 5.9 at 32, 40 / 8.5 at 400.  The
// estimates (us) are fitted to both kernels on 629 shapes (I 16 - 400, J 16 -
// 8000, 1 - 32 heads); picking the smaller one is 0.4 % slower than the better
// kernel on average, 19 % (0.7 us) at worst.
constexpr bool context_mfma_wins(int64_t I, int64_t H, int64_t J, int D) {
    if (I < 16 || J < 16) return false;
    const double c64[2][5] = {{3.07, 3.52, 1.78, 0.77, 5.42}, {3.20, 0.55, 5.58, 3.83, 0.0}};
    const double c80[2][5] = {{3.27, 7.53, 1.93, 1.18, 11.49}, {3.13, 1.01, 3.52, 4.73, 0.0}};
    const double c128[2][5] = {{3.63, 6.32, 3.76, 1.94, 9.30}, {3.83, 1.89, 8.13, 11.83, 0.0}};
    const double(&c)[2][5] = D == 64 ? c64 : (D == 80 ? c80 : c128);
    const double keys = J / 1000.0, rows = I * H > 512 ? (I * H - 512) / 1000.0 : 0.0;
    const double lanes8 = c[0][0] + c[0][1] * keys + (I * H > 512 ? c[0][2] * keys : 0.0) + rows * (c[0][3] + c[0][4] * keys);
    const double steps = (double)((J + 127) / 128), wgs = (double)((I + 31) / 32 * H);
    const double over = wgs > 256 ? (wgs - 256) / 1000.0 : 0.0;
    return c[1][0] + c[1][1] * steps + over * (c[1][2] + c[1][3] * steps) < lanes8;
}

}  // namespace tlhip
