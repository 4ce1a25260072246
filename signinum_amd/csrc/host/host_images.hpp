// Host arrays that a decode writes.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <vector>

namespace sgn {

// An image in a call's device block (rows without gaps) and its host array.
struct HostImage {
    uint8_t *dst;
    size_t stride, off, row, rows;
};

// Whether two images write a common byte, or may: pairs of different strides
// whose ranges meet count as such, and so does a list with more meeting ranges
// than are looked at.  Tiles of one canvas meet in range without sharing bytes.
inline bool images_overlap(const std::vector<HostImage> &images) {
    std::vector<const HostImage *> v;
    for (const HostImage &im : images)
        if (im.row && im.rows) v.push_back(&im);
    std::sort(v.begin(), v.end(),
              [](const HostImage *a, const HostImage *b) { return a->dst < b->dst; });
    size_t looked = 256 * v.size();
    for (size_t i = 0; i < v.size(); ++i) {
        const HostImage &a = *v[i];
        const uintptr_t a0 = reinterpret_cast<uintptr_t>(a.dst);
        const size_t span = a.stride * (a.rows - 1) + a.row;
        for (size_t k = i + 1; k < v.size(); ++k) {
            const HostImage &b = *v[k];
            const size_t d = reinterpret_cast<uintptr_t>(b.dst) - a0;
            if (d >= span) break;
            if (!looked-- || (b.rows > 1 && a.rows > 1 && b.stride != a.stride)) return true;
            // b's first row starts in a's line y at column x; it may run into line y + 1
            if (a.rows == 1) return true;
            const size_t y = d / a.stride, x = d % a.stride;
            if (x < a.row || (x + b.row > a.stride && y + 1 < a.rows)) return true;
        }
    }
    return false;
}

}  // namespace sgn
