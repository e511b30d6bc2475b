// SPDX-License-Identifier: Apache-2.0
#include <hip/hip_runtime.h>

#include <functional>
#include <mutex>
#include <stdexcept>

#include "pcg_resident.hpp"

namespace chysx_amd {

[[noreturn]] void throw_hip(hipError_t err, const char* what);

namespace {

// Launches whose instances span more than kFreeCluster workgroups run one
// after the other on a device, whatever their streams: two that each hold part
// of the compute units while they wait for the rest would not meet.  Smaller
// ones never hold enough of them (at most 32 hardware queues with 7 waiting
// workgroups each, of 256 compute units) and stay free.
constexpr int kFreeCluster = 8;
constexpr int kMaxDevices = 64;
struct Gate {
    std::mutex lock;
    hipEvent_t last = nullptr;  // the latest gated launch
    hipStream_t stream = nullptr;
};
Gate& gate_of_device() {
    static Gate gates[kMaxDevices];
    int dev = 0;
    const hipError_t err = hipGetDevice(&dev);
    if (err != hipSuccess) throw_hip(err, "hipGetDevice");
    if (dev < 0 || dev >= kMaxDevices) throw std::runtime_error("chysx: device index out of range");
    return gates[dev];
}

}  // namespace

void with_resident_gate(int max_cluster, hipStream_t s, const std::function<void()>& enqueue) {
    if (max_cluster <= kFreeCluster) {
        enqueue();
        return;
    }
    auto check = [](hipError_t err, const char* what) {
        if (err != hipSuccess) throw_hip(err, what);
    };
    Gate& G = gate_of_device();
    const std::lock_guard<std::mutex> hold(G.lock);
    if (!G.last) check(hipEventCreateWithFlags(&G.last, hipEventDisableTiming), "hipEventCreate(resident solve)");
    else if (G.stream != s) check(hipStreamWaitEvent(s, G.last, 0), "hipStreamWaitEvent(resident solve)");
    enqueue();
    check(hipEventRecord(G.last, s), "hipEventRecord(resident solve)");
    G.stream = s;
}

}  // namespace chysx_amd
