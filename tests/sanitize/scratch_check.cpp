// The rules of the device scratch (pdspy_amd/csrc/scratch.h) on host memory,
// under AddressSanitizer and UBSan.  Prints "scratch_check ok" and exits 0, or
// names the first violation and exits 1.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <initializer_list>

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

int main() {
    if (check_growing()) return 1;
    std::printf("scratch_check ok\n");
    return 0;
}
