// SPDX-License-Identifier: Apache-2.0
#include "resident_gate.hpp"

#include <hip/hip_runtime.h>

#include <functional>
#include <mutex>
#include <stdexcept>

#include "pcg_resident.hpp"

namespace chysx_amd {

[[noreturn]] void throw_hip(hipError_t err, const char* what);

namespace {

constexpr int kMaxDevices = 64;
struct Gate {
    std::mutex lock;
    GateBook<hipEvent_t> book;
};
Gate& gate_of(int device) {
    static Gate gates[kMaxDevices];
    if (device < 0 || device >= kMaxDevices) throw std::runtime_error("chysx: device index out of range");
    return gates[device];
}

}  // namespace

void with_resident_gate(const GatedLaunch& L, hipStream_t s, const std::function<void()>& enqueue) {
    if (L.weight <= 0) {
        enqueue();
        return;
    }
    auto check = [](hipError_t err, const char* what) {
        if (err != hipSuccess) throw_hip(err, what);
    };
    Gate& G = gate_of(L.device);
    const std::lock_guard<std::mutex> hold(G.lock);
    const auto waits = G.book.admit(L.owner, L.done, L.weight, L.room, [&](hipEvent_t e) {
        const hipError_t err = hipEventQuery(e);
        if (err == hipSuccess) return true;
        if (err != hipErrorNotReady) throw_hip(err, "hipEventQuery(solve in flight)");
        (void)hipGetLastError();  // not an error of a later launch
        return false;
    });
    for (hipEvent_t e : waits) check(hipStreamWaitEvent(s, e, 0), "hipStreamWaitEvent(solve in flight)");
    enqueue();
    check(hipEventRecord(L.done, s), "hipEventRecord(solve)");
}

void leave_resident_gate(int device, const void* owner) {
    Gate& G = gate_of(device);
    const std::lock_guard<std::mutex> hold(G.lock);
    G.book.forget(owner);
}

}  // namespace chysx_amd
