// Host copies by several threads, from the serving loop's pinned read-back
// block into its callers' pageable memory: one thread copies at about 20 GB/s,
// less where pages are touched for the first time, and the frames come down the
// link at 57. A burst of 24 mixed frames (139 MB), submitted and polled: 6.3 ms
// with the caller alone, 5.0 with one thread more, 4.0 with four (65, 43 and
// 22 ms into fresh memory). rf_render's single frames gain less (1920 x 1080:
// 0.84 to 0.76 ms) and lose in fresh memory (1.5 to 3.1 ms): not used there.
#include <algorithm>
#include <chrono>
#include <cstring>

#if defined(__x86_64__)
#include <immintrin.h>
#endif

#include "rf_internal.hpp"

namespace rf {

static inline void relax() {
#if defined(__x86_64__)
    _mm_pause();
#else
    std::this_thread::yield();
#endif
}

void copy_rows(const CopyRows& c, size_t r0, size_t r1) {
    if (c.dst_pitch == c.row && c.src_pitch == c.row) {
        std::memcpy(c.dst + r0 * c.row, c.src + r0 * c.row, (r1 - r0) * c.row);
        return;
    }
    for (size_t r = r0; r < r1; ++r) std::memcpy(c.dst + r * c.dst_pitch, c.src + r * c.src_pitch, c.row);
}

// Pieces of about PIECE bytes, taken from a counter by whoever is free: a
// thread that is scheduled late takes fewer.
constexpr size_t PIECE = 256 << 10;
// Below this the caller copies alone: the others would not be awake in time.
constexpr size_t ALONE = 512 << 10;
// How long a thread that ran out of work looks for more before it sleeps.
constexpr auto LINGER = std::chrono::microseconds(200);

CopyPool::CopyPool() {
    const unsigned cores = std::thread::hardware_concurrency();
    const unsigned n = std::min(4u, cores > 1 ? cores - 1 : 0u);
    try {
        for (unsigned i = 0; i < n; ++i) threads.emplace_back([this] { worker(); });
    } catch (...) {  // fewer threads, or none: the caller copies what they do not
    }
}

CopyPool::~CopyPool() {
    {
        std::lock_guard<std::mutex> g(m);
        stop = true;
    }
    cv.notify_all();
    for (std::thread& t : threads) t.join();
}

void CopyPool::work() {
    for (;;) {
        const size_t k = next.fetch_add(1);
        if (k >= pieces) return;
        const size_t r0 = k * rows_per_piece, r1 = std::min(r0 + rows_per_piece, job.rows);
        copy_rows(job, r0, r1);
    }
}

void CopyPool::worker() {
    uint64_t seen = 0;
    for (;;) {
        const auto until = std::chrono::steady_clock::now() + LINGER;
        while (epoch.load() == seen && std::chrono::steady_clock::now() < until)
            for (int i = 0; i < 32; ++i) relax();
        {
            std::unique_lock<std::mutex> lk(m);
            cv.wait(lk, [&] { return stop || epoch.load() != seen; });
            if (stop) return;
            seen = epoch.load();
            if (!open) continue;  // a copy that is done already
            ++inside;
        }
        work();
        inside.fetch_sub(1);
    }
}

void CopyPool::run(const CopyRows& c) {
    if (c.rows == 0 || c.row == 0) return;
    std::unique_lock<std::mutex> one(user, std::defer_lock);
    // small, nobody to help, or the threads are another caller's just now
    if (c.rows * c.row < ALONE || threads.empty() || !one.try_lock()) {
        copy_rows(c, 0, c.rows);
        return;
    }
    {
        std::lock_guard<std::mutex> g(m);
        job = c;
        rows_per_piece = std::max<size_t>(1, PIECE / c.row);
        pieces = (c.rows + rows_per_piece - 1) / rows_per_piece;
        next.store(0);
        open = true;
        epoch.fetch_add(1);
    }
    cv.notify_all();
    work();
    {
        std::lock_guard<std::mutex> g(m);
        open = false;  // nobody enters any more
    }
    while (inside.load() != 0) relax();
}

}  // namespace rf
