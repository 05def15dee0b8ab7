// rf::CopyPool (rf_copy.cpp): copies of many shapes, from several callers at
// once, arrive whole and write nothing between their rows. Built as host code by
// tests/test_copy_pool.py; prints "copies mismatches".
#include <cstdio>
#include <cstring>
#include <random>
#include <thread>
#include <vector>

#include "../../retrofire_amd/csrc/rf_copy.cpp"

static long check(rf::CopyPool& pool, unsigned seed, int rounds) {
    std::mt19937_64 rng(seed);
    long bad = 0;
    for (int i = 0; i < rounds; ++i) {
        const size_t row = i % 3 == 0 ? 4096 : 1 + rng() % 9000, rows = rng() % (i % 2 ? 40 : 700);
        const size_t sp = row + (i % 4 ? rng() % 70 : 0), dp = row + (i % 5 ? rng() % 70 : 0);
        std::vector<uint8_t> src(sp * rows + 1), dst(dp * rows + 1, 0xA5), want = dst;
        for (uint8_t& b : src) b = (uint8_t)rng();
        for (size_t r = 0; r < rows; ++r) std::memcpy(&want[r * dp], &src[r * sp], row);
        pool.run({dst.data(), src.data(), dp, sp, row, rows});
        bad += dst != want;
    }
    return bad;
}

int main() {
    long total = 0, bad = 0;
    for (int k = 0; k < 4; ++k) {
        rf::CopyPool pool;
        long b[3] = {0, 0, 0};
        std::vector<std::thread> callers;
        for (int c = 0; c < 3; ++c)
            callers.emplace_back([&, c] { b[c] = check(pool, 10 * k + c, 120); });
        for (std::thread& t : callers) t.join();
        total += 360;
        bad += b[0] + b[1] + b[2];
    }
    std::printf("%ld %ld\n", total, bad);
    return bad != 0;
}
