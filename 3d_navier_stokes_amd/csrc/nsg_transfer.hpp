// nsg_transfer.hpp -- copies between the caller's (pageable) host arrays and the device, through
// pinned slots and several host threads; not part of the C ABI.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <functional>

namespace nsgx {

// Handles that copy (contexts, increment statistics) hold the slot pool while they live; the last
// one gives its pinned memory back.
void pool_ref();
void pool_unref();

// host side of the bytes [off, off + len) of the device array: fills the slot from the caller's array
// (upload) or empties it into that array (download).  Called from several threads on disjoint ranges.
using HostPart = std::function<void(size_t off, size_t len, char* slot)>;
// further host work of a download, split into `parts` (called once for each part)
using SidePart = std::function<void(int part, int parts)>;

// Uploads `bytes` to dst / downloads them from src on the stream (of the current device), in chunks
// that are multiples of `unit` bytes (but for the last).  host_bytes: what the host side reads or
// writes in all (it sets the number of threads).  Both return when every copy and host part is done.
hipError_t upload(hipStream_t s, void* dst, size_t bytes, size_t unit, size_t host_bytes, const HostPart& fill);
hipError_t download(hipStream_t s, const void* src, size_t bytes, size_t unit, size_t host_bytes, const HostPart& drain,
                    const SidePart& side = SidePart());
// the same for plain arrays
hipError_t upload(hipStream_t s, void* dst, const void* host, size_t bytes);
hipError_t download(hipStream_t s, const void* src, void* host, size_t bytes);

// one slot of the pool, for what is small enough that a kernel writes it to the host by itself
constexpr size_t kSlotBytes = 2u << 20;
struct Slot {
    char* p = nullptr;
    bool pinned = false;  // else plain memory, which no kernel can write
};
struct SlotGuard {
    Slot slot;
    SlotGuard();
    ~SlotGuard();
    SlotGuard(const SlotGuard&) = delete;
    SlotGuard& operator=(const SlotGuard&) = delete;
};

}  // namespace nsgx
