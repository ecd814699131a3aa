// The device a thread's HIP calls go to.
#pragma once

#include <hip/hip_runtime.h>

namespace tamd {

// 0 where there is none (the call that follows fails by itself).
inline int current_device() {
    int d = 0;
    return hipGetDevice(&d) == hipSuccess ? d : 0;
}

// Makes `device` the thread's current one for the scope.  A thread starts on
// device 0, whichever one the process works on, and a launch goes to the current
// device, where memory of another one need not be mapped; a copy finds the
// device from its pointers.
class device_scope {
public:
    explicit device_scope(int device) : before_(current_device()), changed_(device != before_) {
        status = changed_ ? hipSetDevice(device) : hipSuccess;
    }
    device_scope(const device_scope&) = delete;
    device_scope& operator=(const device_scope&) = delete;
    ~device_scope() {
        if (changed_) (void)hipSetDevice(before_);
    }
    hipError_t status;

private:
    const int before_;
    const bool changed_;
};

}  // namespace tamd
