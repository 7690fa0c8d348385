// Mutual exclusion of the calls that run grid-synchronizing kernels on a device.
#pragma once

#include <mutex>

namespace snhip {

// A grid of such a kernel fills the device, and two of them, each with part of its
// workgroups resident, would wait for each other. One call at a time holds the
// device's gate, from before its launch until its kernel has finished. Who waits
// holds the turnstile (next_), so that a caller in a loop cannot pass through again
// before it.
class DeviceGate {
public:
    void enter() {
        next_.lock();
        hold_.lock();
        next_.unlock();
    }
    void leave() { hold_.unlock(); }

private:
    std::mutex next_, hold_;
};

}  // namespace snhip
