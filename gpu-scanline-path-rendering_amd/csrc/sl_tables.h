// sl_tables.h -- host-built lookup tables of the renderer.
#pragma once

#include <stdint.h>
#include <vector>

namespace sl {

// Sample positions of one pixel for n = 8, 16 or 32 samples, x/y pairs in [0,1)^2.
void sample_positions(int n, float *xy);

// 256x256 line -> sample-mask table, words per texel: 1 (8 spp), 2 (16 spp), 4 (32 spp).
void build_pixel_table(int n, std::vector<uint32_t> &out);

struct ColorTables {
    float dec[256];    // 8-bit code -> value (sRGB decoded, or k/255)
    float thr[256];    // smallest value encoding to k (thr[0] = -inf)
    // sRGB: intervals of [0, 1] on which the code takes at most two values, k and k + 1 from thr on:
    // value v lies in interval (bits(v + kQuantShift) >> 16) - kQuantBase.  The sum's exponent
    // makes the intervals grow with v as the sRGB thresholds' distances do.
    struct Step { float thr, dec, dec_next; uint32_t code; } step[645];
};
constexpr float kQuantShift = 0.03125f;          // 2^-5
constexpr uint32_t kQuantBase = 0x3D000000u >> 16;  // interval of v = 0
constexpr int kQuantSteps = 645;                 // up to v = 1
bool build_color_tables(int srgb, ColorTables &t);

}  // namespace sl
