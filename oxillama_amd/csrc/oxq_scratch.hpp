// A growable device buffer of the library's own, and how it grows: to the size that a call runs best with, and where that is
// not to be had to the size that it needs.  (No HIP header here: a host test stands in for the allocator.)
#pragma once
#include <cstddef>

namespace oxq {

struct ScratchBuffer {
    void *ptr = nullptr;
    size_t cap = 0;

    // alloc(&p, bytes): 0 on success; drop(p) frees.  What the buffer serves from now on: best, else need, else 0 (and then `status`
    // is the allocator's last answer).
    template <class Alloc, class Drop>
    size_t grow(size_t best, size_t need, int &status, Alloc alloc, Drop drop) {
        status = 0;
        if (best <= cap) return best;
        release(drop);
        const size_t tries[] = {best + best / 4 + 256, best, need + need / 4 + 256, need};
        for (size_t i = best == need ? 2 : 0; i < 4; i++) {
            status = alloc(&ptr, tries[i]);
            if (status == 0) {
                cap = tries[i];
                return i < 2 ? best : need;
            }
            ptr = nullptr;
        }
        return 0;
    }
    template <class Drop>
    void release(Drop drop) {
        if (ptr) drop(ptr);
        ptr = nullptr;
        cap = 0;
    }
};

}  // namespace oxq
