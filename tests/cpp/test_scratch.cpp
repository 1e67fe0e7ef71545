// The library's scratch where the allocator has less than a call would run best with: the call gets what it needs.
#include <cstdio>
#include <cstdlib>

#include "../../oxillama_amd/csrc/oxq_scratch.hpp"

static int failed = 0;
#define CHECK(x)                                                \
    do {                                                        \
        if (!(x)) {                                             \
            std::printf("%s:%d: %s\n", __FILE__, __LINE__, #x); \
            failed++;                                           \
        }                                                       \
    } while (0)

struct Device {  // one allocation at a time of at most `room` bytes
    size_t room;
    int held = 0;
    size_t grow(oxq::ScratchBuffer &b, size_t best, size_t need, int &status) {
        return b.grow(best, need, status,
                      [&](void **p, size_t n) {
                          if (held || n > room) return 2;
                          *p = std::malloc(1);
                          held++;
                          return 0;
                      },
                      [&](void *p) { std::free(p), held--; });
    }
};

int main() {
    int status = 0;
    {  // room for all of it; a second call finds it there
        Device d{1000000};
        oxq::ScratchBuffer b;
        CHECK(d.grow(b, 64000, 3000, status) == 64000 && status == 0 && b.cap >= 64000);
        void *const p = b.ptr;
        CHECK(d.grow(b, 5000, 5000, status) == 5000 && b.ptr == p);
        CHECK(d.grow(b, 200000, 200000, status) == 200000 && b.cap >= 200000 && d.held == 1);
    }
    {  // not for what it would run best with
        Device d{10000};
        oxq::ScratchBuffer b;
        CHECK(d.grow(b, 64000, 3000, status) == 3000 && status == 0 && b.cap >= 3000 && d.held == 1);
        CHECK(d.grow(b, 64000, 9900, status) == 9900 && b.cap >= 9900 && d.held == 1);
    }
    {  // exactly for it, without the margin
        Device d{64000};
        oxq::ScratchBuffer b;
        CHECK(d.grow(b, 64000, 3000, status) == 64000 && b.cap == 64000);
    }
    {  // not even for what it needs: nothing is kept, and a smaller call is served again
        Device d{1000};
        oxq::ScratchBuffer b;
        CHECK(d.grow(b, 64000, 3000, status) == 0 && status == 2 && b.ptr == nullptr && b.cap == 0 && d.held == 0);
        CHECK(d.grow(b, 700, 700, status) == 700 && status == 0);
    }
    std::printf("%d failed\n", failed);
    return failed != 0;
}
