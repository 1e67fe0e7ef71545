// The process-wide LDS limit of a kernel, with a counted stand-in for the runtime's call: launches of one kernel from
// two threads with different row lengths must never find the limit below what they asked for.
#include <algorithm>
#include <cstdio>
#include <thread>
#include <vector>

#include "../../oxillama_amd/csrc/oxq_lds_opt_in.hpp"

static int failed = 0;
#define CHECK(x)                                                     \
    do {                                                             \
        if (!(x)) {                                                  \
            std::printf("%s:%d: %s\n", __FILE__, __LINE__, #x);      \
            failed++;                                                \
        }                                                            \
    } while (0)

struct Runtime {  // one limit per process, as the runtime has it (one kernel, two devices)
    size_t limit[2] = {0, 0};
    int calls = 0, status = 0;
    int launch(oxq::LdsOptIn &o, int device, size_t bytes) {  // 0: the launch fits under the limit of its time
        const int st = o.raise(this, device, bytes, 99, [&](size_t n) {
            calls++;
            if (status == 0) limit[device] = n;
            return status;
        });
        return st ? st : bytes <= limit[device] ? 0 : -1;
    }
};

int main() {
    oxq::LdsOptIn o;
    Runtime first, second;
    {
        Runtime &r = first;
        CHECK(r.launch(o, 0, 100 << 10) == 0);
        std::thread([&] { CHECK(r.launch(o, 0, 50 << 10) == 0); }).join();  // a thread with shorter rows
        CHECK(r.launch(o, 0, 100 << 10) == 0);
        CHECK(r.calls == 1 && r.limit[0] == 100 << 10);
        std::thread([&] { CHECK(r.launch(o, 0, 150 << 10) == 0); }).join();
        CHECK(r.launch(o, 0, 120 << 10) == 0 && r.calls == 2);
        CHECK(r.launch(o, 1, 40 << 10) == 0 && r.limit[1] == 40 << 10 && r.calls == 3);  // the other device has its own
        CHECK(r.launch(o, 0, 150 << 10) == 0 && r.calls == 3);
    }
    {  // a refused call leaves the limit where it was, and is made again
        Runtime &r = second;
        CHECK(r.launch(o, 0, 64 << 10) == 0);
        r.status = 7;
        CHECK(r.launch(o, 0, 200 << 10) == 7 && r.launch(o, 0, 200 << 10) == 7 && r.calls == 3);
        r.status = 0;
        CHECK(r.launch(o, 0, 64 << 10) == 0 && r.launch(o, 0, 160 << 10) == 0 && r.calls == 4);
    }
    {  // many kernels that share slots of the threads' tables, from several threads
        std::vector<Runtime> kernels(600);
        std::mutex mu;
        auto work = [&](size_t first) {
            for (int round = 0; round < 3; round++)
                for (size_t i = 0; i < kernels.size(); i++) {
                    const size_t bytes = ((first + i * 7 + round * 13) % 160 + 1) << 10;
                    const int st = o.raise(&kernels[i], 0, bytes, 99, [&](size_t n) {
                        kernels[i].limit[0] = n;
                        return 0;
                    });
                    std::lock_guard<std::mutex> lock(mu);
                    CHECK(st == 0);
                }
        };
        std::vector<std::thread> pool;
        for (size_t t = 0; t < 4; t++) pool.emplace_back(work, t * 40);
        for (auto &t : pool) t.join();
        for (size_t i = 0; i < kernels.size(); i++) {
            size_t most = 0;
            for (size_t t = 0; t < 4; t++)
                for (int round = 0; round < 3; round++) most = std::max(most, ((t * 40 + i * 7 + round * 13) % 160 + 1) << 10);
            CHECK(kernels[i].limit[0] == most);
        }
    }
    std::printf("%d failed\n", failed);
    return failed != 0;
}
