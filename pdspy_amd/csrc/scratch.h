// Device scratch kept between calls.  The device is a template parameter, so
// that the rules are checked on the host (tests/sanitize/scratch_check.cpp).
#pragma once
#include <cstddef>

// One buffer that grows.  Its users ask by size: an allocation that failed, or a
// smaller one made after it, leaves a buffer that a larger user must not get.
// Dev: static void *alloc(size_t) (NULL if there is no memory), static void free(void *).
template <class Dev>
struct GrowBuffer {
    void *p = nullptr;
    size_t cap = 0;

    void grow(size_t need) {
        if (cap >= need) return;
        release();
        p = Dev::alloc(need);
        if (p) cap = need;
    }
    // the buffer, if it holds `need` bytes
    void *get(size_t need) const { return need > 0 && need <= cap ? p : nullptr; }
    void release() {
        if (p) Dev::free(p);
        p = nullptr;
        cap = 0;
    }
};
