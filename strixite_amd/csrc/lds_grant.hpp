// A kernel's dynamic LDS above the default limit has to be allowed once on each device that runs it.
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <mutex>
#include <vector>

namespace strix::kernels {

// Allows `kernel` `bytes` of dynamic LDS on the current device, unless that much is allowed there already (so a launch
// that needs no more than before makes no runtime call but the device's lookup). A refusal is returned and not kept:
// the next call asks again.
inline hipError_t allow_lds(const void *kernel, size_t bytes) {
    struct Grant {
        int device;
        const void *kernel;
        size_t bytes;
    };
    static std::mutex mu;
    static std::vector<Grant> granted;
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) return e;
    std::lock_guard<std::mutex> lock(mu);
    Grant *g = nullptr;
    for (Grant &i : granted)
        if (i.device == device && i.kernel == kernel) g = &i;
    if (g != nullptr && g->bytes >= bytes) return hipSuccess;
    e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
    if (e != hipSuccess) return e;
    if (g != nullptr) g->bytes = bytes;
    else granted.push_back({device, kernel, bytes});
    return hipSuccess;
}

}  // namespace strix::kernels
