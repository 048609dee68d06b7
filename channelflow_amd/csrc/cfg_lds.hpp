// The dynamic-LDS opt-in of kernels that take more than 64 KB.
#pragma once

#include <hip/hip_runtime.h>

#include <map>
#include <stdexcept>
#include <string>
#include <utility>

namespace cfg {

// Raises a kernel's dynamic-LDS limit once per (device, kernel, size), so that
// launches recorded into a graph make no attribute calls.
template <class K>
inline void allow_lds(K kernel, size_t bytes) {
    if (bytes <= 64 * 1024) return;
    static std::map<std::pair<int, const void*>, size_t> done;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) throw std::runtime_error(std::string("hipGetDevice: ") + hipGetErrorString(e));
    size_t& d = done[std::make_pair(dev, (const void*)kernel)];
    if (d >= bytes) return;
    e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
    if (e != hipSuccess)  // the launch that follows would fail without saying why
        throw std::runtime_error("hipFuncSetAttribute(MaxDynamicSharedMemorySize, " + std::to_string(bytes) +
                                 " B): " + hipGetErrorString(e));
    d = bytes;
}

}  // namespace cfg
