// Pinned host memory, grow-only (rf_render's staging).
#include <algorithm>

#include "rf_internal.hpp"

namespace rf {

bool PinBuf::ensure(size_t bytes) {
    if (bytes <= cap) return true;
    const size_t want = (bytes + std::min(bytes / 4, PIN_SLACK) + 4095) & ~size_t(4095);
    uint8_t* q = nullptr;
    if (hipHostMalloc((void**)&q, want, 0)) {
        // The caller goes on without: the error is settled here, or the check
        // behind the next launch would report it as that launch's.
        (void)hipGetLastError();
        return false;
    }
    release();
    p = q;
    cap = want;
    return true;
}

void PinBuf::release() {
    if (p) (void)hipHostFree(p);
    p = nullptr;
    cap = 0;
}

}  // namespace rf
