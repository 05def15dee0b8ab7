// Checks rf::outcode (rf_math.hpp) against the sign of each plane's distance,
// rf::plane_dist, over every quadruple of special values and random ones.
// Built as host code by tests/test_outcode.py; prints "cases mismatches".
#include <cmath>
#include <cstdio>
#include <cstring>
#include <limits>
#include <random>

#include "../../retrofire_amd/csrc/rf_math.hpp"

int main() {
    const float inf = std::numeric_limits<float>::infinity(), nan = std::numeric_limits<float>::quiet_NaN();
    const float big = std::numeric_limits<float>::max(), tiny = std::numeric_limits<float>::denorm_min();
    const float v[] = {0.0f, -0.0f, 1.0f, -1.0f, std::nextafter(1.0f, 2.0f), -std::nextafter(1.0f, 0.0f), tiny, -tiny,
                       big,  -big,  inf,  -inf,  nan,                       0.1f};
    long total = 0, bad = 0;
    auto check = [&](float x, float y, float z, float w) {
        uint32_t want = 0;
        for (int p = 0; p < 6; ++p) want |= rf::plane_dist(p, x, y, z, w) > 0.0f ? 1u << p : 0u;
        ++total;
        bad += rf::outcode(x, y, z, w) != want;
    };
    for (float x : v)
        for (float y : v)
            for (float z : v)
                for (float w : v) check(x, y, z, w);
    std::mt19937_64 rng(7);
    for (int i = 0; i < 2000000; ++i) {
        float f[4];
        for (float& c : f) {
            const uint32_t b = (uint32_t)rng();
            std::memcpy(&c, &b, 4);
        }
        check(f[0], f[1], f[2], f[3]);                     // any bits
        check(f[0], f[1], f[2], (i & 1) ? f[0] : -f[2]);  // on a plane
    }
    std::printf("%ld %ld\n", total, bad);
    return bad != 0;
}
