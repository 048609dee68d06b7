// The library's process-wide caches over a fake HIP with several devices: memory is
// the host's, and hipGetDevice returns what fake_device says. Built by
// tests/test_device_caches.py with g++.
#include <cstdlib>
#include <cstring>
#include <vector>

#include "../../channelflow_amd/csrc/cfg_host.hpp"
#include "../../channelflow_amd/csrc/cfg_lds.hpp"

static int fake_device = 0, raised = 0, set_ups = 0;

extern "C" {
hipError_t hipGetDevice(int* d) { *d = fake_device; return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) { *p = std::calloc(1, n); return hipSuccess; }
hipError_t hipFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return ""; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = nullptr; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t*) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float*, hipEvent_t, hipEvent_t) { return hipSuccess; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { ++raised; return hipSuccess; }
}

namespace cfg {
void launch_tau_setup(const Geom&, const TauSet&, double, bool, hipStream_t) { ++set_ups; }
}  // namespace cfg

extern "C" {

// Geometry, tau set and constants of one grid made on `first` and kept, then asked for
// on `second`: how many of the three are the kept ones.
int shared_between(int first, int second) {
    const cfg_grid g{16, 9, 16, 0, 2.0, 1.0, -1.0, 1.0};
    cfg::DevPool pool;
    fake_device = first;
    const auto geo = cfg::geometry_for(g, true);
    const auto tau = cfg::tau_for(*geo, 0.01, 5.0, true, nullptr, pool, nullptr);
    const auto con = cfg::shared_consts({1.0, 2.0});
    fake_device = second;
    const auto geo2 = cfg::geometry_for(g, true);
    const auto tau2 = cfg::tau_for(*geo2, 0.01, 5.0, true, nullptr, pool, nullptr);
    const auto con2 = cfg::shared_consts({1.0, 2.0});
    return (geo == geo2) + (tau == tau2) + (con == con2);
}

static void kernel() {}

// attribute calls of two launches with `bytes` of dynamic LDS on each device
int raises(int devices, long bytes) {
    raised = 0;
    for (int i = 0; i < 2 * devices; ++i) {
        fake_device = i / 2;
        cfg::allow_lds(kernel, (size_t)bytes);
    }
    return raised;
}

}  // extern "C"
