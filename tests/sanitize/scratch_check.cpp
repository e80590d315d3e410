// The rules of the device scratch (pdspy_amd/csrc/scratch.h) on host memory,
// under AddressSanitizer and UBSan.  Prints "scratch_check ok" and exits 0, or
// names the first violation and exits 1.
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <initializer_list>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

#include "../../pdspy_amd/csrc/scratch.h"

static int fail(const char *what) {
    std::printf("scratch_check FAILED: %s\n", what);
    return 1;
}

// host memory with a limit on one allocation
struct Mem {
    static size_t limit;
    static int live;
    static void *alloc(size_t n) {
        if (n > limit) return nullptr;
        ++live;
        return std::malloc(n);
    }
    static void free(void *p) {
        --live;
        std::free(p);
    }
};
size_t Mem::limit = 0;
int Mem::live = 0;

// A batch's items on one stream share a buffer and grow it in turn; each then
// writes what it asked for.  Whatever allocations fail, no item may be given a
// buffer smaller than that.
static int check_growing() {
    const size_t needs[][4] = {{64, 1, 0, 0}, {1, 64, 2, 64}, {8, 64, 8, 0}, {64, 8, 65, 9}};
    for (size_t limit : {0, 1, 8, 63, 64, 100})
        for (const size_t *n : needs) {
            Mem::limit = limit;
            GrowBuffer<Mem> b;
            for (int i = 0; i < 4; ++i) b.grow(n[i]);
            if (b.get(0)) return fail("a buffer for nothing");
            for (int i = 0; i < 4; ++i) {
                void *p = b.get(n[i]);
                if (p) std::memset(p, 1, n[i]);
                if (p && n[i] > limit) return fail("a buffer that could not be allocated");
            }
            b.release();
            if (Mem::live) return fail("a buffer left");
        }
    return 0;
}

// a stream: tasks run in order on a thread of its own
struct Queue {
    std::mutex mu;
    std::condition_variable cv;
    std::deque<std::function<void()>> todo;
    bool busy = false, stop = false;
    std::thread th{[this] {
        std::unique_lock<std::mutex> l(mu);
        for (;;) {
            cv.wait(l, [&] { return stop || !todo.empty(); });
            if (todo.empty()) return;
            auto f = todo.front();
            todo.pop_front();
            busy = true;
            l.unlock();
            f();
            l.lock();
            busy = false;
            cv.notify_all();
        }
    }};
    void push(std::function<void()> f) {
        std::lock_guard<std::mutex> l(mu);
        todo.push_back(f);
        cv.notify_all();
    }
    void drain() {
        std::unique_lock<std::mutex> l(mu);
        cv.wait(l, [&] { return todo.empty() && !busy; });
    }
    ~Queue() {
        drain();
        {
            std::lock_guard<std::mutex> l(mu);
            stop = true;
            cv.notify_all();
        }
        th.join();
    }
};

struct Flag {
    std::mutex mu;
    std::condition_variable cv;
    bool set = false;
    void raise() {
        std::lock_guard<std::mutex> l(mu);
        set = true;
        cv.notify_all();
    }
    void wait() {
        std::unique_lock<std::mutex> l(mu);
        cv.wait(l, [&] { return set; });
    }
};
struct Ev {
    std::shared_ptr<Flag> last;
};

// Every stream has the same handle, and which queue it is depends on the thread:
// the per-thread default stream, or a handle that came back.
static thread_local Queue *mine = nullptr;
struct Host : Mem {
    using Stream = int;
    using Event = Ev *;
    static std::atomic<int> fail_wait, fail_make, fail_record;
    static bool make(Event &e) {
        if (fail_make) return false;
        e = new Ev();
        return true;
    }
    static void drop(Event e) { delete e; }
    static bool wait_host(Event e) {
        if (fail_wait) return false;
        e->last->wait();
        return true;
    }
    static bool wait(Stream, Event e) {
        if (fail_wait) return false;
        auto f = e->last;
        mine->push([f] { f->wait(); });
        return true;
    }
    static bool record(Event e, Stream) {
        if (fail_record) return false;
        auto f = std::make_shared<Flag>();
        e->last = f;
        mine->push([f] { f->raise(); });
        return true;
    }
    static void drain(Stream) { mine->drain(); }
};
std::atomic<int> Host::fail_wait{0}, Host::fail_make{0}, Host::fail_record{0};

// Calls of growing and shrinking sizes from several threads: what a call has
// written is there when its own later work reads it, and the buffer lives until then.
static int check_sharing() {
    Mem::limit = 1 << 20;
    SharedScratch<Host> sc;
    std::atomic<int> bad{0}, ran{0};
    std::vector<std::thread> ts;
    for (int t = 0; t < 4; ++t)
        ts.emplace_back([&, t] {
            Queue q;
            mine = &q;
            for (int i = 0; i < 24; ++i) {
                const size_t n = 64 + (size_t)((i * 37 + t * 91) % 400) * (i / 8 + 1);
                sc.with(0, n, [&](void *p) {
                    unsigned char *c = (unsigned char *)p;
                    const int v = 1 + t;
                    q.push([c, n, v] { std::memset(c, v, n); });
                    q.push([] { std::this_thread::sleep_for(std::chrono::microseconds(300)); });
                    q.push([c, n, v, &bad, &ran] {
                        for (size_t k = 0; k < n; ++k) bad += c[k] != v;
                        ++ran;
                    });
                });
            }
            q.drain();
        });
    for (auto &t : ts) t.join();
    sc.release();
    if (ran != 4 * 24) return fail("calls left out");
    if (bad) return fail("a call's scratch written by another");
    return Mem::live ? fail("a shared buffer left") : 0;
}

// Each thing that can fail: the call is told to do without, or is waited for
static int check_failures() {
    Queue q;
    mine = &q;
    SharedScratch<Host> sc;
    int n = 0;
    auto f = [&](void *) { ++n; };
    Host::fail_make = 1;
    if (sc.with(0, 8, f) || n) return fail("no event, but a buffer");
    Host::fail_make = 0;
    Mem::limit = 4;
    if (sc.with(0, 8, f) || n) return fail("no memory, but a buffer");
    if (!sc.with(0, 4, f) || n != 1) return fail("a smaller buffer refused");
    Mem::limit = 100;
    Host::fail_wait = 1;
    if (sc.with(0, 4, f) || sc.with(0, 8, f) || n != 1) return fail("a buffer still in use");
    Host::fail_wait = 0;
    Host::fail_record = 1;
    std::atomic<int> done{0};
    if (!sc.with(0, 8, [&](void *) {
            q.push([&] { std::this_thread::sleep_for(std::chrono::milliseconds(5)); ++done; });
        }) || !done)
        return fail("no event to wait on, but no wait");
    Host::fail_record = 0;
    sc.release();
    q.drain();
    return 0;
}

int main() {
    if (check_growing() || check_failures() || check_sharing()) return 1;
    std::printf("scratch_check ok\n");
    return 0;
}
