// images_overlap against a map of written bytes: random rectangles of one or two
// canvases.  Where no two share a byte it may still say so only for pairs of
// different strides.
#include <cstdio>
#include <random>

#include "../signinum_amd/csrc/host/host_images.hpp"

int main() {
    using sgn::HostImage;
    std::mt19937 rng(7);
    auto pick = [&](size_t lo, size_t hi) { return lo + rng() % (hi - lo + 1); };
    int seen[2] = {0, 0};
    for (int it = 0; it < 200000; ++it) {
        std::vector<uint8_t> mem(600);
        std::vector<HostImage> v;
        const size_t strides[2] = {pick(1, 20), pick(1, 20)};
        const bool mixed = it % 8 == 0;
        bool same = true;
        for (size_t n = pick(0, 4); n; --n) {
            const size_t stride = strides[mixed ? rng() % 2 : 0];
            const size_t row = pick(0, stride), rows = pick(0, 5);
            v.push_back({mem.data() + pick(0, it % 2 ? 60 : 400), stride, 0, row, rows});
            same &= stride == v[0].stride;
        }
        std::vector<int> count(mem.size() + 400, 0);
        bool shared = false;
        for (const HostImage &im : v)
            for (size_t y = 0; y < im.rows; ++y)
                for (size_t x = 0; x < im.row; ++x)
                    shared |= ++count[size_t(im.dst - mem.data()) + y * im.stride + x] > 1;
        const bool got = sgn::images_overlap(v);
        if (shared ? !got : got && same) {
            std::printf("iteration %d: %d images, shared %d, said %d\n", it, int(v.size()), shared,
                        got);
            return 1;
        }
        ++seen[shared];
    }
    // a canvas of 64 x 64 tiles, then one tile a byte too wide
    std::vector<uint8_t> mem(64 * 64 * 4 * 4);
    std::vector<HostImage> v;
    for (size_t k = 0; k < 64 * 64; ++k)
        v.push_back({mem.data() + (k / 64) * 4 * 256 + (k % 64) * 4, 256, 0, 4, 4});
    if (sgn::images_overlap(v)) return std::printf("canvas\n"), 1;
    v[1234].row = 5;
    if (!sgn::images_overlap(v)) return std::printf("wide tile\n"), 1;
    std::printf(seen[0] && seen[1] ? "ok\n" : "one outcome only\n");
    return 0;
}
