// Device scratch kept between calls.  The device is a template parameter, so
// that the rules are checked on the host (tests/sanitize/scratch_check.cpp).
#pragma once
#include <cstddef>
#include <mutex>

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

// One buffer that calls on any stream and from any thread share.  A call's work is
// ordered behind that of the call before it by an event, always: an equal stream
// handle does not mean the same queue (a destroyed stream's handle may come back, and
// the per-thread default stream is one handle for all threads).
// Dev, besides alloc and free: types Stream and Event (falsy until made); static bool
// make(Event &), drop(Event), wait_host(Event), wait(Stream, Event), record(Event,
// Stream), drain(Stream); each leaves no error behind.
template <class Dev>
class SharedScratch {
    GrowBuffer<Dev> buf_;
    typename Dev::Event ev_{};
    bool used_ = false;
    std::mutex mu_;

    void *take(typename Dev::Stream s, size_t need) {
        if (!ev_ && !Dev::make(ev_)) return nullptr;
        if (buf_.cap < need) {
            if (used_ && !Dev::wait_host(ev_)) return nullptr;
            used_ = false;
            buf_.grow(need);
        }
        if (used_ && !Dev::wait(s, ev_)) return nullptr;
        return buf_.get(need);
    }

public:
    // f(p) enqueues work on s that uses p[0 .. need); false: no scratch, nothing done
    template <class F>
    bool with(typename Dev::Stream s, size_t need, F f) {
        std::lock_guard<std::mutex> lock(mu_);
        void *p = take(s, need);
        if (!p) return false;
        f(p);
        used_ = Dev::record(ev_, s);
        if (!used_) Dev::drain(s);  // nothing to wait on: wait here
        return true;
    }
    void release() {
        buf_.release();
        if (ev_) Dev::drop(ev_);
        ev_ = {};
        used_ = false;
    }
};
