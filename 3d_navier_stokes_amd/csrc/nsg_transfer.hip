// nsg_transfer.hip -- see nsg_transfer.hpp.  Host code only.
//
// A pageable copy runs at 29 GB/s to the device and 10-17 GB/s from it (one thread of the runtime
// stages it), a pinned one at 57 GB/s both ways, and the caller's array is usually fresh: its page
// faults cost as much as the copy.  So the array goes chunk by chunk through a ring of pinned slots:
// the calling thread makes every HIP call (a thread's first one costs it some 100 us), and from
// kThreadedBytes on, worker threads move the chunks between slots and array, faulting the pages in.
// Smaller arrays stay on the calling thread: a worker that has to share a core with the caller's own
// (often spinning) thread pool can lose milliseconds (12 boxes of 0.8 to 22 MB: 44 -> 58 ms).
#include "nsg_transfer.hpp"

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <system_error>
#include <thread>
#include <vector>

namespace {

constexpr int kMaxSlots = 32;                   // 64 MiB of pinned memory at most
constexpr int kMaxThreads = 8;
constexpr size_t kThreadedBytes = 32u << 20, kBytesPerThread = 8u << 20;

using nsgx::kSlotBytes;
using nsgx::Slot;

struct Pool {
    std::mutex mu;
    std::condition_variable freed;
    std::vector<Slot> idle;
    int made = 0, refs = 0;
};
Pool& pool() {
    static Pool p;
    return p;
}

void release_memory(const Slot& s) {
    if (s.pinned) (void)hipHostFree(s.p);
    else std::free(s.p);
}

// 1 to n slots (as many as there are without waiting; waits for one if other threads hold all)
std::vector<Slot> acquire(int n) {
    Pool& q = pool();
    std::vector<Slot> got;
    got.reserve(n);
    std::unique_lock<std::mutex> lk(q.mu);
    for (;;) {
        while ((int)got.size() < n && !q.idle.empty()) {
            got.push_back(q.idle.back());
            q.idle.pop_back();
        }
        while ((int)got.size() < n && q.made < kMaxSlots) {
            Slot s;
            void* p = nullptr;
            if (hipHostMalloc(&p, kSlotBytes, hipHostMallocDefault) == hipSuccess) {
                s.pinned = true;
            } else {
                (void)hipGetLastError();
                p = std::malloc(kSlotBytes);  // no pinned memory left: the runtime stages the copies
            }
            if (!p) break;
            s.p = (char*)p;
            ++q.made;
            q.idle.reserve(q.made);  // giving a slot back never allocates
            got.push_back(s);
        }
        if (!got.empty() || q.made == 0) return got;
        q.freed.wait(lk);
    }
}
void give_back(const std::vector<Slot>& slots) {
    Pool& q = pool();
    std::lock_guard<std::mutex> lk(q.mu);
    for (const Slot& s : slots) {
        if (q.refs > 0) {
            q.idle.push_back(s);
        } else {
            release_memory(s);
            --q.made;
        }
    }
    q.freed.notify_all();
}

// Chunk k lives in slot k % S.  Uploads: host part (slot free) -> copy; downloads: copy -> host part.
// moved[k] is set when the host part of chunk k is done; open = number of chunks whose host part may
// start (uploads: their slots are free; downloads: their copies are done).
struct Transfer {
    hipStream_t s;
    char* dev;
    size_t bytes, chunk, nchunk;
    bool up;
    const nsgx::HostPart& part;
    const nsgx::SidePart& side;
    std::vector<Slot> slots;
    std::vector<hipEvent_t> ev;
    std::unique_ptr<std::atomic<bool>[]> moved;
    std::atomic<size_t> open{0};
    std::atomic<bool> stop{false};

    size_t off(size_t k) const { return k * chunk; }
    size_t len(size_t k) const { return std::min(chunk, bytes - k * chunk); }
    size_t S() const { return slots.size(); }

    void host(size_t k) {
        part(off(k), len(k), slots[k % S()].p);
        moved[k].store(true, std::memory_order_release);
    }
    // worker w of n: its share of the side work, then chunks w, w + n, ...
    void worker(int w, int n) {
        if (side) side(w, n);
        for (size_t k = w; k < nchunk; k += n) {
            while (open.load(std::memory_order_acquire) <= k) {
                if (stop.load(std::memory_order_relaxed)) return;
                std::this_thread::yield();
            }
            host(k);
        }
    }
    hipError_t copy(size_t k) {
        const hipError_t e = up ? hipMemcpyAsync(dev + off(k), slots[k % S()].p, len(k), hipMemcpyHostToDevice, s)
                                : hipMemcpyAsync(slots[k % S()].p, dev + off(k), len(k), hipMemcpyDeviceToHost, s);
        return e != hipSuccess || !ev[k % S()] ? e : hipEventRecord(ev[k % S()], s);
    }
    // a single chunk has no event: the stream holds nothing after it
    hipError_t wait(size_t k) { return ev[k % S()] ? hipEventSynchronize(ev[k % S()]) : hipStreamSynchronize(s); }
    // all chunks, the host parts by this thread (alone) or by workers; every slot is idle afterwards
    hipError_t run(bool alone) {
        hipError_t e = hipSuccess;
        auto host_done = [&](size_t k) {
            if (alone) {
                host(k);
                return;
            }
            while (!moved[k].load(std::memory_order_acquire)) std::this_thread::yield();
        };
        if (up) {
            open.store(std::min(S(), nchunk), std::memory_order_release);
            for (size_t k = 0; k < nchunk; ++k) {
                // chunk k - S / 2's copy frees its slot for chunk k + S - S / 2
                const size_t lag = std::max<size_t>(1, S() / 2);
                if (k >= lag) {
                    if ((e = wait(k - lag)) != hipSuccess) break;
                    open.store(std::min(k - lag + 1 + S(), nchunk), std::memory_order_release);
                }
                host_done(k);
                if ((e = copy(k)) != hipSuccess) break;
            }
        } else {
            size_t next = 0;
            for (; next < std::min(S(), nchunk) && e == hipSuccess; ++next) e = copy(next);
            if (alone && side) side(0, 1);
            for (size_t k = 0; k < nchunk && e == hipSuccess; ++k) {
                if ((e = wait(k)) != hipSuccess) break;
                open.store(k + 1, std::memory_order_release);
                if (alone) host(k);
                // refill the slot of the oldest chunk once it is empty
                while (e == hipSuccess && next < nchunk && moved[next - S()].load(std::memory_order_acquire)) e = copy(next++);
                if (e == hipSuccess && k + 1 == next && next < nchunk) {  // nothing in flight: wait for a slot
                    host_done_wait(next - S());
                    e = copy(next++);
                }
            }
        }
        if (e != hipSuccess) stop.store(true);
        const hipError_t w = hipStreamSynchronize(s);  // no copy touches a slot any more
        return e != hipSuccess ? e : w;
    }
    void host_done_wait(size_t k) {
        while (!moved[k].load(std::memory_order_acquire)) std::this_thread::yield();
    }
};

hipError_t transfer(hipStream_t s, void* dev, size_t bytes, size_t unit, size_t host_bytes, bool up,
                    const nsgx::HostPart& part, const nsgx::SidePart& side) {
    if (bytes == 0) return hipSuccess;
    hipError_t e = hipSuccess;
    std::vector<std::thread> th;
    std::vector<Slot> slots;
    std::vector<hipEvent_t> ev;
    try {
        const int cores = (int)std::max(1u, std::thread::hardware_concurrency());
        const int want = host_bytes < kThreadedBytes ? 0 : (int)std::min<size_t>(std::min(kMaxThreads, cores), host_bytes / kBytesPerThread);
        // at least four chunks, so that copies and host parts overlap
        const size_t per = std::max<size_t>(bytes / (want ? 4 * want : 4) + 1, 256u << 10);
        const size_t chunk = std::max(unit, std::min(per, kSlotBytes) / unit * unit);
        Transfer t{s, (char*)dev, bytes, chunk, (bytes + chunk - 1) / chunk, up, part, side, {}, {}, nullptr};
        th.reserve(want);
        slots.reserve(2 * want + 3);
        slots = acquire((int)std::min<size_t>(t.nchunk, want ? 2 * want : 3));
        if (slots.empty()) return hipErrorOutOfMemory;
        t.slots = slots;
        ev.assign(slots.size(), nullptr);
        for (auto& v : ev)
            if (e == hipSuccess && t.nchunk > 1) e = hipEventCreateWithFlags(&v, hipEventDisableTiming);
        t.ev = ev;
        t.moved.reset(new std::atomic<bool>[t.nchunk]);
        for (size_t k = 0; k < t.nchunk; ++k) t.moved[k].store(false);
        if (e == hipSuccess) {
            int n = 0;
            std::atomic<int> go{0};  // workers start when their number is known; < 0: none
            try {
                for (; n < want; ++n)
                    th.emplace_back([&t, &go, n] {
                        int g;
                        while ((g = go.load(std::memory_order_acquire)) == 0) std::this_thread::yield();
                        if (g > 0) t.worker(n, g);
                    });
            } catch (const std::system_error&) {  // fewer threads, or none
            }
            go.store(n ? n : -1, std::memory_order_release);
            e = t.run(n == 0);
            for (auto& x : th) x.join();
        }
    } catch (const std::bad_alloc&) {
        e = hipErrorOutOfMemory;
    }
    for (hipEvent_t v : ev)
        if (v) (void)hipEventDestroy(v);
    if (!slots.empty()) give_back(slots);
    return e;
}

}  // namespace

namespace nsgx {

void pool_ref() {
    Pool& q = pool();
    std::lock_guard<std::mutex> lk(q.mu);
    ++q.refs;
}

void pool_unref() {
    Pool& q = pool();
    std::lock_guard<std::mutex> lk(q.mu);
    if (--q.refs > 0) return;
    for (const Slot& s : q.idle) release_memory(s);
    q.made -= (int)q.idle.size();
    q.idle.clear();
}

SlotGuard::SlotGuard() {
    try {
        std::vector<Slot> v = acquire(1);
        if (!v.empty()) slot = v[0];
    } catch (const std::bad_alloc&) {
    }
}
SlotGuard::~SlotGuard() {
    if (!slot.p) return;
    Pool& q = pool();
    std::lock_guard<std::mutex> lk(q.mu);
    if (q.refs > 0) {
        q.idle.push_back(slot);
    } else {
        release_memory(slot);
        --q.made;
    }
    q.freed.notify_all();
}

hipError_t upload(hipStream_t s, void* dst, size_t bytes, size_t unit, size_t host_bytes, const HostPart& fill) {
    return transfer(s, dst, bytes, unit, host_bytes, true, fill, SidePart());
}
hipError_t download(hipStream_t s, const void* src, size_t bytes, size_t unit, size_t host_bytes, const HostPart& drain,
                    const SidePart& side) {
    return transfer(s, const_cast<void*>(src), bytes, unit, host_bytes, false, drain, side);
}
// An array that crosses as it is needs no host part: below kThreadedBytes the runtime's own staging is the
// faster one (increment statistics of a host snapshot, two uploads, slots -> runtime: 64^3 906 -> 613 us,
// 110^3 (32 MB) 4426 -> 2842; with the worker threads 115^3 (37 MB) 3254 -> 2775, 150^3 6260 -> 5270).  The
// callers wait for the stream before they return
hipError_t upload(hipStream_t s, void* dst, const void* host, size_t bytes) {
    if (bytes < kThreadedBytes) return hipMemcpyAsync(dst, host, bytes, hipMemcpyHostToDevice, s);
    return upload(s, dst, bytes, 4096, bytes,
                  [host](size_t off, size_t len, char* slot) { std::memcpy(slot, (const char*)host + off, len); });
}
hipError_t download(hipStream_t s, const void* src, void* host, size_t bytes) {
    if (bytes < kThreadedBytes) {
        const hipError_t e = hipMemcpyAsync(host, src, bytes, hipMemcpyDeviceToHost, s);
        return e != hipSuccess ? e : hipStreamSynchronize(s);
    }
    return download(s, src, bytes, 4096, bytes,
                    [host](size_t off, size_t len, char* slot) { std::memcpy((char*)host + off, slot, len); });
}

}  // namespace nsgx
