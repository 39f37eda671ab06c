// Facts about an AMD GPU that launch heuristics need, looked up once per device and cached for the
// life of the process. (The reference keeps the equivalent cudaDeviceProp fields inside its nvidia
// handle, src/infiniop/devices/nvidia/nvidia_common.cu:15-63.)
#ifndef INFINICORE_AMD_DEVICE_H
#define INFINICORE_AMD_DEVICE_H

#include <atomic>
#include <chrono>

namespace device::amd {

struct DeviceInfo {
    int compute_units;   // CUs on the device (256 on MI355X)
    int wavefront_size;  // lanes per wavefront (64 on CDNA)
    bool queried;        // false when HIP could not see the device and defaults were used
};

// Never fails: if the device cannot be queried (no GPU visible to this process) it returns MI355X
// defaults with queried == false, so descriptors can still be created and validated on a host
// without a GPU.
const DeviceInfo &deviceInfo(int device_id);

// A 64-bit value no earlier call of this process has used and that is never 0 (the value of a cleared flag):
// a counter that starts at a point of the clock, spread over the word by an odd multiplier. What a workspace
// holds before its first use can only be mistaken for it by a 2^-64 accident.
inline unsigned long long nextToken() {
    static std::atomic<unsigned long long> counter{
        static_cast<unsigned long long>(std::chrono::steady_clock::now().time_since_epoch().count()) | 1ull};
    unsigned long long t = counter.fetch_add(1, std::memory_order_relaxed) * 0x9e3779b97f4a7c15ull;
    return t != 0 ? t : 0x9e3779b97f4a7c15ull;
}

} // namespace device::amd

#endif
