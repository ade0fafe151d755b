// What a kernel has to be told before its first launch on a device, told once a device and not once a process: plain C++.
#pragma once
#include <atomic>
#include <cstdint>

namespace nh {

// One object a kernel, of static storage.  Threads that meet here may tell the same thing twice, which is harmless.
class OnceADevice {
    std::atomic<uint64_t> told{0};

public:
    // `tell` answers zero where it succeeded; what failed is told again.  (Devices past the word's bits: every time.)
    template <class Tell>
    auto operator()(int32_t device, Tell tell) -> decltype(tell()) {
        const uint64_t bit = device >= 0 && device < 64 ? uint64_t(1) << device : 0u;
        if (told.load(std::memory_order_acquire) & bit) return decltype(tell())(0);
        const auto status = tell();
        if (status == decltype(tell())(0)) told.fetch_or(bit, std::memory_order_release);
        return status;
    }
};

}  // namespace nh
