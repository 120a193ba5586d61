// box_overlap.h -- how much a scene's instance boxes overlap (host code; runtime.cpp).
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>

namespace lchip {

// Boxes that a point of the scene lies in, on average: the boxes' volumes over that of the box around
// them. Where the boxes that meet the largest one hold nine tenths of all the volume, the scene is those:
// what lies apart from them, however far, is too little to matter and does not enlarge it. `boxes` holds
// 8 floats per box (low corner and a pad, high corner and a pad).
inline double box_overlap(const float *boxes, uint32_t n) {
    struct Sum {
        double volume = 0.0;
        float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
        void add(const float *b, double v) {
            volume += v;
            for (int k = 0; k < 3; k++) {
                lo[k] = std::min(lo[k], b[k]);
                hi[k] = std::max(hi[k], b[4 + k]);
            }
        }
        double overlap() const {
            const double around = ((double)hi[0] - lo[0]) * ((double)hi[1] - lo[1]) * ((double)hi[2] - lo[2]);
            return around > 0.0 && std::isfinite(around) ? volume / around : 0.0;
        }
    };
    // 0 for boxes without geometry (degenerate) or a finite size, which take no part
    const auto volume = [](const float *b) {
        const double v = ((double)b[4] - b[0]) * ((double)b[5] - b[1]) * ((double)b[6] - b[2]);
        return v > 0.0 && std::isfinite(v) ? v : 0.0;
    };
    Sum all, group;
    const float *largest = nullptr;
    double most = 0.0;
    for (uint32_t i = 0; i < n; i++) {
        const float *b = boxes + 8 * (uint64_t)i;
        const double v = volume(b);
        if (v == 0.0) continue;
        all.add(b, v);
        if (v > most) {
            most = v;
            largest = b;
        }
    }
    if (!largest) return 0.0;
    for (uint32_t i = 0; i < n; i++) {
        const float *b = boxes + 8 * (uint64_t)i;
        const double v = volume(b);
        bool meets = v != 0.0;
        for (int k = 0; k < 3; k++) meets = meets && b[k] <= largest[4 + k] && b[4 + k] >= largest[k];
        if (meets) group.add(b, v);
    }
    return group.volume >= 0.9 * all.volume ? std::max(group.overlap(), all.overlap()) : all.overlap();
}

} // namespace lchip
