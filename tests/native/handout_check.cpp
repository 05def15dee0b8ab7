// rf::Handout (rf_handout.hpp): room for read-back that a poll gives back reaches
// a worker that found none. Built as host code by tests/test_handout.py; prints
// "cases failures".
#include <atomic>
#include <cstdio>
#include <thread>
#include <vector>

#include "rf_handout.hpp"

using namespace std::chrono_literals;
constexpr uint64_t BLOCK = 1 << 20;
static uint8_t mem[BLOCK];

// The poll gives the block's only buffer back after the worker has found no room
// and before it waits, as far as the lock allows. What the worker then does is
// what the serving loop's worker does: wait, and look again when woken.
static bool late_return() {
    rf::Handout h;
    h.pin.init(mem, BLOCK);
    rf::Done d{};
    d.pixels = h.pin_take(BLOCK);
    d.pix_bytes = BLOCK;
    h.done.push_back(d);
    std::atomic<bool> copying{false}, looked{false}, polled{false};
    std::thread client([&] {
        h.hand_out(8, 0, [&](uint32_t, const rf::Done&) {
            copying = true;
            while (!looked) std::this_thread::yield();
        });
        polled = true;
    });
    while (!copying) std::this_thread::yield();
    std::unique_lock<std::mutex> lk(h.m);
    uint8_t* p = h.pin_take(BLOCK);
    bool ok = p == nullptr;
    looked = true;
    for (int i = 0; i < 200 && !polled; ++i) std::this_thread::sleep_for(1ms);
    while (!p && h.cv_work.wait_for(lk, 2s) == std::cv_status::no_timeout) p = h.pin_take(BLOCK);
    ok = ok && p == mem;
    lk.unlock();
    client.join();
    return ok;
}

// A worker that serves `n` requests through a block with room for two results,
// and `clients` that poll until all have come.
static bool stream(uint64_t n, int clients) {
    rf::Handout h;
    h.pin.init(mem, BLOCK);
    std::atomic<uint64_t> got{0};
    std::atomic<bool> lost{false};
    std::thread worker([&] {
        std::unique_lock<std::mutex> lk(h.m);
        for (uint64_t i = 0; i < n;) {
            rf::Done d{};
            d.res.id = i;
            d.pixels = h.pin_take(BLOCK / 2);
            d.pix_bytes = BLOCK / 2;
            if (d.pixels) {
                h.done.push_back(d);
                h.cv_done.notify_all();
                ++i;
            } else if (h.cv_work.wait_for(lk, 5s) == std::cv_status::timeout) {
                lost = true;
                return;
            }
        }
    });
    std::vector<std::thread> polls;
    for (int c = 0; c < clients; ++c)
        polls.emplace_back([&] {
            while (got < n && !lost) got += h.hand_out(3, 1, [](uint32_t, const rf::Done&) {});
        });
    worker.join();
    for (std::thread& t : polls) t.join();
    return !lost && got == n && h.pin.used == 0 && h.pin.largest() == BLOCK;
}

int main() {
    int cases = 0, bad = 0;
    for (int i = 0; i < 3; ++i, ++cases) bad += !late_return();
    for (int clients : {1, 2, 4}) {
        bad += !stream(20000, clients);
        ++cases;
    }
    std::printf("%d %d\n", cases, bad);
    return bad != 0;
}
