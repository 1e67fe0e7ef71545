// How much dynamic LDS the kernels are opted in to.  The runtime keeps one limit per kernel and device for the whole
// process, while the launches of one kernel ask for amounts that depend on their row length: the limit is only ever
// raised, whichever thread asks, so that no thread's launch finds it below what it was told it has.
// (No HIP header here: a host test counts the calls that would go to the runtime.)
#pragma once
#include <cstddef>
#include <cstdint>
#include <mutex>
#include <unordered_map>

namespace oxq {

class LdsOptIn {  // (one per process)
    struct Key {
        const void *kern;
        int device;
        bool operator==(const Key &o) const { return kern == o.kern && device == o.device; }
    };
    struct Hash {
        size_t operator()(const Key &k) const { return reinterpret_cast<uintptr_t>(k.kern) ^ (size_t)k.device * 0x9E3779B97F4A7C15ull; }
    };
    std::mutex mu;
    std::unordered_map<Key, size_t, Hash> limit;

public:
    // set(bytes): the runtime's call for this kernel and device, 0 on success.  Returns its status; a failed call
    // leaves the limit as it was; `no_memory` if the table cannot grow.
    template <class Set>
    int raise(const void *kern, int device, size_t bytes, int no_memory, Set set) {
        // what this thread knows to be allowed at least, by (kernel, device): true for good, as no limit is lowered; a
        // slot that another pair took only costs the way through the lock
        struct Known {
            const void *kern = nullptr;
            int device = -1;
            size_t bytes = 0;
        };
        static thread_local Known known[256];
        Known &t = known[((reinterpret_cast<uintptr_t>(kern) >> 4) ^ (uintptr_t)device * 31) & 255];
        if (t.kern == kern && t.device == device && t.bytes >= bytes) return 0;
        std::lock_guard<std::mutex> lock(mu);
        size_t *have = nullptr;
        try {
            have = &limit[Key{kern, device}];
        } catch (...) {
            return no_memory;
        }
        if (*have < bytes) {
            const int status = set(bytes);
            if (status != 0) return status;
            *have = bytes;
        }
        t = Known{kern, device, *have};
        return 0;
    }
};

}  // namespace oxq
