// engine_amd/csrc/per_device.hpp: set-up runs once on each device, again after a failure,
// and on every call past the 64th device.
#include "per_device.hpp"

#include <cstdio>
#include <thread>
#include <vector>

#define CHECK(x)                                                  \
    do {                                                          \
        if (!(x)) {                                               \
            std::printf("line %d: %s\n", __LINE__, #x);           \
            return 1;                                             \
        }                                                         \
    } while (0)

int main() {
    ribn_amd::PerDevice p;
    int calls = 0, result = 0;
    auto setup = [&] { ++calls; return result; };
    CHECK(p.once(0, setup) == 0 && calls == 1);
    CHECK(p.once(0, setup) == 0 && calls == 1);
    result = 7;  // a second device: its own set-up, repeated while it fails
    CHECK(p.once(1, setup) == 7 && calls == 2);
    CHECK(p.once(1, setup) == 7 && calls == 3);
    CHECK(p.once(0, setup) == 0 && calls == 3);
    result = 0;
    CHECK(p.once(1, setup) == 0 && calls == 4);
    CHECK(p.once(1, setup) == 0 && calls == 4);
    CHECK(p.once(63, setup) == 0 && p.once(63, setup) == 0 && calls == 5);
    CHECK(p.once(64, setup) == 0 && p.once(64, setup) == 0 && calls == 7);
    CHECK(p.once(0, setup) == 0 && calls == 7);

    ribn_amd::PerDevice q;
    std::vector<std::thread> threads;
    std::atomic<int> done{0}, early{0};
    for (int t = 0; t < 8; ++t)
        threads.emplace_back([&, t] {
            std::atomic<int>* mine = &done;
            q.once(t & 1, [&] { mine->fetch_or(1 << (t & 1)); return 0; });
            if (!(mine->load() & (1 << (t & 1)))) ++early;
        });
    for (auto& t : threads) t.join();
    CHECK(early == 0 && done == 3);
    std::puts("ok");
    return 0;
}
