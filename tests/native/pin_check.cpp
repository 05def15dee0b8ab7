// rf::PinBuf (rf_pin.cpp) over a host memory allocator that can fail. Built as host
// code by tests/test_pin.py; prints "checks failures".
#include <cstdio>
#include <cstdlib>
#include <set>

#include "../../retrofire_amd/csrc/rf_pin.cpp"

static size_t limit;              // larger requests fail
static hipError_t last_error;     // what hipGetLastError reports
static std::set<void*> blocks;

extern "C" hipError_t hipHostMalloc(void** p, size_t n, unsigned int) {
    if (n > limit) return last_error = hipErrorOutOfMemory;
    blocks.insert(*p = std::malloc(1));
    return hipSuccess;  // a success leaves an earlier error where it is
}
extern "C" hipError_t hipHostFree(void* p) {
    if (!blocks.erase(p)) return last_error = hipErrorInvalidValue;
    std::free(p);
    return hipSuccess;
}
extern "C" hipError_t hipGetLastError() {
    const hipError_t e = last_error;
    last_error = hipSuccess;
    return e;
}

static int checks = 0, bad = 0;
#define CHECK(c) (++checks, (c) ? 0 : (++bad, std::printf("%s\n", #c)))

int main() {
    rf::PinBuf b;
    limit = size_t(1) << 40;
    CHECK(b.ensure(100000) && b.p && b.cap >= 100000 && b.cap <= 130000);
    uint8_t* const first = b.p;
    CHECK(b.ensure(100001) && b.p == first);  // within what is held
    const size_t held = b.cap;
    limit = 1 << 20;
    CHECK(!b.ensure(2 << 20));
    CHECK(b.p == first && b.cap == held && blocks.size() == 1);  // a failed growth loses nothing
    CHECK(hipGetLastError() == hipSuccess);                      // and leaves no error for the next launch
    CHECK(b.ensure(held) && b.p == first);
    limit = size_t(1) << 40;
    CHECK(b.ensure(256 << 20) && b.cap >= (256u << 20) && b.cap <= (256u << 20) + rf::PIN_SLACK + 4096);
    CHECK(blocks.size() == 1);
    b.release();
    CHECK(blocks.empty() && !b.p && b.cap == 0);
    limit = 0;
    CHECK(!b.ensure(1) && !b.p && b.cap == 0 && hipGetLastError() == hipSuccess);
    std::printf("%d %d\n", checks, bad);
    return bad != 0;
}
