// The host's read of a device-resident key and H (the kernel-level calls).
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdint>
#include <mutex>
#include <new>

#include "si_kernels.h"
#include "si_launch.h"

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

// Where a fetch lands: pinned memory that the device can write.
struct Box {
    uint8_t bytes[32];
    uint32_t flag;
};

// The boxes.  One in use at a time (the lock); a fetch whose end was not seen
// (its stream could not be waited for) may still write its own, so that box is
// left until its flag shows that the kernel has ended.
struct Slot {
    Box* box = nullptr;
    uint32_t unseen = 0;  // the sequence number of a fetch not seen to end
};
constexpr int kSlots = 16;
std::mutex g_boxes_lock;
Slot g_boxes[kSlots];
uint32_t g_seq = 0;  // never 0 in a fetch
std::atomic<uint64_t> g_fetches{0};

bool landed(const Box* b, uint32_t seq) { return __atomic_load_n(&b->flag, __ATOMIC_ACQUIRE) == seq; }

void wipe(Box* b)
{
    volatile uint8_t* const w = b->bytes;
    for (size_t k = 0; k < sizeof(b->bytes); ++k) w[k] = 0;
}

// A slot that no kernel can write, with its box (nullptr: none free, or no
// memory; no error stays pending).  Unseen fetches that have ended since give theirs back, wiped.
Slot* take_slot()
{
    Slot* free_slot = nullptr;
    for (Slot& s : g_boxes) {
        if (s.unseen && landed(s.box, s.unseen)) {
            wipe(s.box);
            s.unseen = 0;
        }
        if (!s.unseen && (!free_slot || (!free_slot->box && s.box))) free_slot = &s;
    }
    if (free_slot && !free_slot->box) {
        void* b = nullptr;
        if (!granted(hipHostMalloc(&b, sizeof(Box), hipHostMallocPortable | hipHostMallocMapped))) return nullptr;
        free_slot->box = new (b) Box();
    }
    return free_slot;
}

}  // namespace

// The kernel-level calls take the key and H as device pointers and need their
// values on the host (which context?).  Two device-to-host copies and a stream
// synchronisation cost such a call about 30 us beyond its record kernel; one
// wave that stores both into pinned host memory, and a host that watches for
// its flag, costs a launch and a PCIe write.  MI355X, a 100,003-byte record
// sealed and then opened: 87.0 -> 40.1 us for the pair.  Only a wait longer than
// the spin (earlier work on the stream) falls back to synchronising the stream.
hipError_t fetch_key(hipStream_t stream, const void* key, const void* h, uint8_t out[32])
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) {
        (void)hipGetLastError();
        return hipErrorNotSupported;
    }
    if (!own_device_bytes(key, dev) || (h && !own_device_bytes(h, dev))) return hipErrorNotSupported;
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone) {
        (void)hipGetLastError();
        return hipErrorNotSupported;
    }
    std::lock_guard<std::mutex> g(g_boxes_lock);
    Slot* const slot = take_slot();
    if (!slot) return hipErrorNotSupported;
    Box* const box = slot->box;
    void* dbox = nullptr;
    if (hipHostGetDevicePointer(&dbox, box, 0) != hipSuccess) {
        (void)hipGetLastError();
        return hipErrorNotSupported;
    }
    Box* const db = static_cast<Box*>(dbox);
    if (++g_seq == 0) g_seq = 1;
    const uint32_t seq = g_seq;
    hipError_t e = launch_key_fetch(stream, static_cast<const uint8_t*>(key), static_cast<const uint8_t*>(h), db->bytes,
                                    &db->flag, seq);
    if (e != hipSuccess) return e;
    constexpr int kSpins = 20000;
    int i = 0;
    while (!landed(box, seq) && ++i < kSpins) __builtin_ia32_pause();
    if (i == kSpins) {
        e = hipStreamSynchronize(stream);
        if (!landed(box, seq)) {
            slot->unseen = seq;
            return e != hipSuccess ? e : hipErrorUnknown;
        }
    }
    const volatile uint8_t* const w = box->bytes;
    if (e == hipSuccess)
        for (int k = 0; k < (h ? 32 : 16); ++k) out[k] = w[k];
    wipe(box);
    if (e == hipSuccess) g_fetches.fetch_add(1, std::memory_order_relaxed);
    return e;
}

uint64_t key_fetches() { return g_fetches.load(std::memory_order_relaxed); }

}  // namespace si
