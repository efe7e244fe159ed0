// grx_once.h - work done once for each device of the process.
#pragma once
#include <atomic>

// A kernel's attributes belong to one device's copy of it, so a limit raised
// on the first GPU that ran the kernel is not raised on the second.  run()
// calls f for the first call on a device and again after a call that returned
// false; threads that meet there may call it twice.  Devices past the table
// call it every time.
class GrxDeviceOnce {
    static constexpr int kDevices = 64;
    std::atomic<bool> done_[kDevices] = {};

  public:
    template <typename F>
    bool run(int device, F &&f) {
        if (device < 0 || device >= kDevices) return f();
        if (done_[device].load(std::memory_order_acquire)) return true;
        if (!f()) return false;
        done_[device].store(true, std::memory_order_release);
        return true;
    }
};
