// One-time set-up of a process-wide object on each device it is used on.
#pragma once

#include <atomic>
#include <cstdint>

namespace ribn_amd {

// A kernel's function attributes (its largest dynamic LDS) belong to the
// device that was current when they were set, so a kernel that a second context
// launches on another GPU needs them there too.
class PerDevice {
  public:
    // setup() the first time on `device`, until it returns 0 (success) there;
    // devices past the 64th set up on every call. Threads may race: setup() is
    // then called more than once, and none returns before it has succeeded.
    template <class F>
    auto once(int device, F&& setup) -> decltype(setup()) {
        const uint64_t bit = device >= 0 && device < 64 ? uint64_t{1} << device : 0;
        if (done_.load(std::memory_order_acquire) & bit) return decltype(setup()){};
        const auto e = setup();
        if (e == decltype(setup()){}) done_.fetch_or(bit, std::memory_order_release);
        return e;
    }

  private:
    std::atomic<uint64_t> done_{0};
};

}  // namespace ribn_amd
