// The host's read of a device-resident key and H (the kernel-level calls).
#include <hip/hip_runtime.h>

#include <cstdint>
#include <mutex>
#include <new>

#include "si_kernels.h"

namespace si {

namespace {

// 16 bytes of the current device's own memory?
bool own_device_bytes(const void* p, int dev)
{
    hipPointerAttribute_t a;
    hipDeviceptr_t base = nullptr;
    size_t size = 0;
    if (hipPointerGetAttributes(&a, p) != hipSuccess || a.type != hipMemoryTypeDevice || a.device != dev ||
        hipMemGetAddressRange(&base, &size, const_cast<void*>(p)) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    const uintptr_t off = reinterpret_cast<uintptr_t>(p) - reinterpret_cast<uintptr_t>(base);
    return off <= size && size - off >= 16;
}

}  // namespace

// The kernel-level calls take the key and H as device pointers and need their
// values on the host (which context?).  Two device-to-host copies and a stream
// synchronisation cost such a call about 30 us beyond its record kernel; one
// wave that stores both into pinned host memory, and a host that watches for
// its flag, costs a launch and a PCIe write.  MI355X, a 100,003-byte record
// sealed and then opened: 87.0 -> 40.1 us for the pair.  Only a wait longer than the spin (earlier
// work on the stream) falls back to synchronising the stream.
hipError_t fetch_key(hipStream_t stream, const void* key, const void* h, uint8_t out[32])
{
    struct Box {
        uint8_t bytes[32];
        uint32_t flag;
    };
    static std::mutex m;
    static Box* box = nullptr;
    static uint32_t seq = 0;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return hipErrorNotSupported;
    if (!own_device_bytes(key, dev) || (h && !own_device_bytes(h, dev))) return hipErrorNotSupported;
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone) {
        (void)hipGetLastError();
        return hipErrorNotSupported;
    }
    std::lock_guard<std::mutex> g(m);
    if (!box) {
        void* b = nullptr;
        if (hipHostMalloc(&b, sizeof(Box), hipHostMallocPortable | hipHostMallocMapped) != hipSuccess)
            return hipErrorNotSupported;
        box = new (b) Box();
    }
    void* dbox = nullptr;
    hipError_t e = hipHostGetDevicePointer(&dbox, box, 0);
    if (e != hipSuccess) return e;
    Box* const db = static_cast<Box*>(dbox);
    ++seq;
    e = launch_key_fetch(stream, static_cast<const uint8_t*>(key), static_cast<const uint8_t*>(h), db->bytes, &db->flag,
                         seq);
    if (e != hipSuccess) return e;
    constexpr int kSpins = 20000;
    int i = 0;
    while (__atomic_load_n(&box->flag, __ATOMIC_ACQUIRE) != seq && ++i < kSpins) __builtin_ia32_pause();
    if (i == kSpins) {
        e = hipStreamSynchronize(stream);
        if (e == hipSuccess && __atomic_load_n(&box->flag, __ATOMIC_ACQUIRE) != seq) e = hipErrorUnknown;
    }
    volatile uint8_t* const w = box->bytes;
    for (int k = 0; k < 32; ++k) {
        if (e == hipSuccess && (k < 16 || h)) out[k] = w[k];
        w[k] = 0;
    }
    return e;
}

}  // namespace si
