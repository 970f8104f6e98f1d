// ff_per_device.hpp -- set-up that is needed once on every device of the process.
// Host only and without GPU calls.
#pragma once

#include <mutex>
#include <set>

namespace ffamd {

// run(device, f): f() if it has not run for that device yet (or threw when it
// did). Safe from several threads.
class OncePerDevice {
public:
    template <class F>
    void run(int device, F f) {
        std::lock_guard<std::mutex> lk(mu_);
        if (done_.count(device)) return;
        f();
        done_.insert(device);
    }

private:
    std::mutex mu_;
    std::set<int> done_;
};

}  // namespace ffamd
