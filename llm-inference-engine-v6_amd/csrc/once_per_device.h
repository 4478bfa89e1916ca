// Something that has to be done once for every device of the process before its first use there (telling a kernel how much LDS
// its launches ask for). Plain C++: it knows nothing of the GPU runtime.
#pragma once

#include <atomic>
#include <mutex>

namespace llme {

class OncePerDevice {
public:
    static constexpr int kDevices = 64;

    // Runs act() -> status (0: done) unless it has succeeded for this device before; a failure is returned and tried again by the
    // next call. A thread that comes while another one acts waits for it, so that nobody goes on before it is done. `at_least`: an
    // amount that act() asks for; it runs again where a call asks for more than was granted.
    template <typename ACT>
    int operator()(int device, int at_least, ACT&& act) {
        if (device < 0 || device >= kDevices) return act();
        if (granted_[device].load(std::memory_order_acquire) >= at_least) return 0;
        std::lock_guard<std::mutex> guard(mutex_);
        if (granted_[device].load(std::memory_order_relaxed) >= at_least) return 0;
        const int status = act();
        if (status == 0) granted_[device].store(at_least, std::memory_order_release);
        return status;
    }

private:
    std::atomic<int> granted_[kDevices] = {};
    std::mutex mutex_;
};

}  // namespace llme
