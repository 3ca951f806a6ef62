// How many output rows a wave of the depthwise matrix kernel walks down (conv_dw_mfma.hip). Plain C++: chosen on the host for every
// launch, and gone over by a test without a GPU.
#pragma once

#include <algorithm>
#include <cmath>

namespace ohip {

// Its wave takes `row` microseconds per row whatever else runs, and as much as `extra` rows more where the strip is longer than the
// ring of input rows holds; a SIMD with several waves takes their instructions one after the other, and up to six of them the fullest
// SIMD (ceil) counts. columns: waves side by side at one strip per image. Fitted to 260 drawn layers of 16 .. 960 channels, 7x7 to
// 208x208, 1 .. 64 images: the chosen height is 0.5 % slower than the best on average, 9 % at worst. With the rule and kernel before
// (the tallest strips that leave 2048 waves, 8 / stride rows at least; seven divisions per wave) 128 channels 5x5 LeakyReLU @13x13 x16
// took 4.4 us (now 3.1), 384 @14x14 x1 3.6 (2.8), 88 @52x52 x16 6.0 (5.1).
struct DwStrips {
    int rows, stride, kernel;  // output rows of the image
    float row, columns;

    // vector instructions of a row, relative: result kind 0 int8, 1 int8 never negative, 2 fp32
    DwStrips(int rows_, int stride_, int kernel_, int result, float columns_)
        : rows(rows_), stride(stride_), kernel(kernel_),
          row(0.139f * (stride_ == 2 ? 0.624f : 1.f) * (kernel_ == 5 ? 0.763f : 1.f) * (result == 1 ? 0.89f : result == 0 ? 1.f : 0.596f)),
          columns(columns_) {}

    int ring() const { return (8 - kernel) / stride + 1; }  // output rows that the first input rows make

    float time(int r, int strips) const {
        const int step = 8 / stride;  // output rows of a step
        const float extra = r <= ring() ? 0.f : r % step ? 4.258f : kExtra, walk = row * ((float)r + extra);
        const float m = columns * (float)strips / 1024.f, full = m <= 6.f ? std::ceil(m) : m + 0.311f;
        return 0.788f * walk + (0.88f * std::max(m, 1.f) + 0.443f * full) * (0.306f + 0.55f * walk);
    }

    // The height with the least time, the tallest of equals. Only heights that some number of strips has are looked at, and of those:
    //  * while all waves have a SIMD of their own a shorter strip is a faster one, but for one row (`extra`, where it is whole steps):
    //    the first height is the shortest of these, or the next;
    //  * all strips together are all rows, and every wave costs its SIMD a part beside its rows: where that alone takes longer than the
    //    best height so far, more strips do too, first those longer than the ring, then all.
    // (looked: how many heights that were. All of them are about 2 sqrt(rows), 0.07 us a launch at 14 rows, 0.23 at 112 and 1.4 at 4096;
    // these take 0.03, 0.05 to 0.1 and 0.5 to 1.1.)
    int choose(int* looked = nullptr) const {
        const int alone = (int)std::min(std::max(1024.f / columns, 1.f), (float)rows);
        const int shortest = (rows + alone - 1) / alone;
        int strips = (rows + shortest) / (shortest + 1), r = (rows + strips - 1) / strips, best_rows = r, count = 0;
        // no more than the sums that time() makes (0.9999: their rounding)
        const float waves = 0.9999f * 1.323f * columns / 1024.f;
        const float in_ring = waves * 0.55f * row * (float)rows, beyond = in_ring + 0.788f * row * ((float)ring() + kExtra);
        float best = INFINITY;
        for (;; ++count) {
            strips = (rows + r - 1) / r;
            if (best <= in_ring + waves * 0.306f * (float)strips) break;
            if (r > ring() && best <= beyond + waves * (0.306f + 0.55f * row * kExtra) * (float)strips) {
                strips = (rows + ring() - 1) / ring(), r = (rows + strips - 1) / strips;
                if (best <= in_ring + waves * 0.306f * (float)strips) break;
            }
            const float t = time(r, strips);
            if (t < best) best = t, best_rows = r;
            if (r == 1) break;
            r = std::min(r - 1, (rows + strips) / (strips + 1));  // the height of the next number of strips
        }
        if (looked) *looked = count;
        return best_rows;
    }

private:
    static constexpr float kExtra = 2.865f;  // the least of `extra` beyond the ring
};

}  // namespace ohip
