// Zero-coding contexts as a table, for the tests' sequential coder and decoder: the kernels form
// them from masks (t1_cm_masks.h). Test infrastructure.
#pragma once
#include <algorithm>
#include <cstdint>

namespace gail_amd {

// Table D.1 for the four orientations (0 LL, 1 HL, 2 LH, 3 HH), indexed [orient * 128 +
// code] by a 7-bit neighbourhood code h | v << 2 | d << 4: h, v the significant horizontal
// and vertical neighbours (0..2), d the diagonal ones (0..4), each as a binary count.
// Codes no neighbourhood produces clamp to the largest counts.
inline void build_zc_table(uint8_t z[4 * 128]) {
    uint8_t t[4 * 45];
    for (int o = 0; o < 4; ++o)
        for (int h = 0; h < 3; ++h)
            for (int v = 0; v < 3; ++v)
                for (int d = 0; d < 5; ++d) {
                    int hh = h, vv = v, c;
                    if (o == 1) {  // HL: horizontal and vertical trade places
                        hh = v;
                        vv = h;
                    }
                    if (o == 3) {
                        const int hv = hh + vv;
                        c = d >= 3 ? 8 : d == 2 ? (hv ? 7 : 6) : d == 1 ? (hv >= 2 ? 5 : hv ? 4 : 3) : (hv >= 2 ? 2 : hv);
                    } else {
                        c = hh == 2 ? 8 : hh == 1 ? (vv ? 7 : d ? 6 : 5) : vv ? (vv == 2 ? 4 : 3) : (d >= 2 ? 2 : d);
                    }
                    t[o * 45 + h * 15 + v * 5 + d] = (uint8_t)c;
                }
    for (int o = 0; o < 4; ++o)
        for (int i = 0; i < 128; ++i) {
            const int h = std::min(2, i & 3), v = std::min(2, (i >> 2) & 3), d = std::min(4, (i >> 4) & 7);
            z[o * 128 + i] = t[o * 45 + h * 15 + v * 5 + d];
        }
}

}  // namespace gail_amd
