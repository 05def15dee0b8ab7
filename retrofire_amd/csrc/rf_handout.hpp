// What the serving loop's threads and the callers of rf_serve_poll hand to each
// other: finished results, and the read-back buffers their pixels lie in.
// Host code only (tests/native/handout_check.cpp builds it by itself).
#pragma once

#include <algorithm>
#include <chrono>
#include <condition_variable>
#include <cstdint>
#include <deque>
#include <map>
#include <mutex>

#include "../../include/retrofire_amd.h"

namespace rf {

// Device blocks and read-back buffers are whole multiples of this.
constexpr uint64_t ARENA_ALIGN = 256;
inline uint64_t align_up(uint64_t x) { return (x + ARENA_ALIGN - 1) & ~(ARENA_ALIGN - 1); }

// First-fit allocator over a byte range; free ranges coalesce. Not locked.
struct Arena {
    uint8_t* base = nullptr;
    uint64_t size = 0, used = 0;
    std::map<uint64_t, uint64_t> free_;  // offset -> bytes
    void init(uint8_t* b, uint64_t n) {
        base = b;
        size = n;
        used = 0;
        free_.clear();
        if (n) free_[0] = n;
    }
    uint64_t largest() const {
        uint64_t m = 0;
        for (const auto& kv : free_) m = std::max(m, kv.second);
        return m;
    }
    bool alloc(uint64_t bytes, uint64_t& off) {
        for (auto it = free_.begin(); it != free_.end(); ++it) {
            if (it->second < bytes) continue;
            off = it->first;
            const uint64_t rest = it->second - bytes;
            free_.erase(it);
            if (rest) free_[off + bytes] = rest;
            used += bytes;
            return true;
        }
        return false;
    }
    void release(uint64_t off, uint64_t bytes) {
        used -= bytes;
        auto it = free_.emplace(off, bytes).first;
        auto nx = std::next(it);
        if (nx != free_.end() && it->first + it->second == nx->first) {
            it->second += nx->second;
            free_.erase(nx);
        }
        if (it != free_.begin()) {
            auto pv = std::prev(it);
            if (pv->first + pv->second == it->first) {
                pv->second += it->second;
                free_.erase(it);
            }
        }
    }
};

struct Done {
    rf_result res;
    uint8_t* pixels = nullptr;  // pinned, width * height * bpp
    size_t pix_bytes = 0;
};

struct Handout {
    std::mutex m;  // guards all below, and the loop's own state
    std::condition_variable cv_work, cv_done;
    std::deque<Done> done;
    Arena pin;  // read-back buffers in the pinned block

    bool pin_in_block(const uint8_t* p) const { return p >= pin.base && p < pin.base + pin.size; }
    // Read-back buffer of `bytes` from the pinned block (nullptr if it does not
    // fit now). Called with `m` held.
    uint8_t* pin_take(size_t bytes) {
        uint64_t off = 0;
        return pin.alloc(align_up(bytes), off) ? pin.base + off : nullptr;
    }
    // Returns one of the block's buffers. Called with `m` held: the worker tests
    // for room and then waits on cv_work in one hold of `m`, so a return that
    // the test missed comes after the wait has begun, and its notification is
    // not lost.
    void pin_put(uint8_t* p, size_t bytes) {
        if (p) pin.release((uint64_t)(p - pin.base), align_up(bytes));
    }
    // Hands out up to `max` of the results that are finished, waiting up to
    // timeout_ms for the first. `deliver(k, result)` runs without `m`, so the
    // worker admits and the waiters report meanwhile; buffers outside the block
    // are its to free. What finishes meanwhile is the next call's: the caller's
    // own work on these results overlaps it (a burst of 24 mixed
    // requests: about 30 us).
    template <class Deliver>
    uint32_t hand_out(uint32_t max, uint32_t timeout_ms, Deliver&& deliver) {
        std::unique_lock<std::mutex> lk(m);
        if (done.empty() && timeout_ms)
            cv_done.wait_for(lk, std::chrono::milliseconds(timeout_ms), [&] { return !done.empty(); });
        max = (uint32_t)std::min<size_t>(max, done.size());
        uint32_t n = 0;
        for (; n < max && !done.empty(); ++n) {
            const Done d = done.front();
            done.pop_front();
            lk.unlock();
            deliver(n, d);
            lk.lock();
            if (pin_in_block(d.pixels)) pin_put(d.pixels, d.pix_bytes);
        }
        lk.unlock();
        if (n) cv_work.notify_all();  // admissions may wait for read-back space
        return n;
    }
};

}  // namespace rf
