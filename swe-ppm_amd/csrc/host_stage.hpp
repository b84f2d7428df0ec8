// host_stage.hpp -- large copies between pageable host arrays and the GPU
// through a ring of pinned slots, the host side done by several threads.
//
// The runtime's own copy of a pageable array runs at 17 to 23 GB/s, and where the
// destination is fresh memory one thread also takes its page faults; the link
// itself moves 55 GB/s to and from pinned memory.  Here the calling thread
// queues the DMA transfers of one slot after the other and the workers copy
// between the slots and the arrays, faults included.
// The calling thread alone talks to the GPU.  Every wait ends: there is at least
// one worker, and a failed transfer raises `stop`, which each waiting loop tests.
#pragma once

#include <hip/hip_runtime.h>
#include <sched.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <thread>

namespace swe {

struct HostCopy {
    void* host;
    void* dev;
    size_t bytes;
};

class HostStage {
   public:
    static constexpr int kSlots = 12, kWorkers = 8;
    static constexpr size_t kSlotBytes = size_t(4) << 20;
    // Bytes in all from which the ring is used.  ms straight and through the ring,
    // arrays of one square block: to fresh host memory 4 MiB 0.29 / 0.33, 11.5
    // 0.73 / 0.54, 48 3.05 / 1.45, 96 10.5 / 3.2, 343 36 / 8.0; to the device 64 MiB
    // 2.35 / 2.05, 128 4.55 / 3.55, 456 14.9 / 10.3, but the first time (the slots'
    // own page faults) 64 MiB 2.6 / 4.9, 128 4.9 / 6.3, 456 18.1 / 17.0.  Slots of
    // 1 / 2 / 4 / 8 MiB: 11.1 / 9.0 / 8.0 / 7.7 ms for 343 MB to the host.  Making the
    // ring takes about 5 ms, which a download of 48 MiB does not win back.
    static constexpr size_t kLeastToHost = size_t(64) << 20, kLeastToDevice = size_t(256) << 20;

    // Pinned memory and events for transfers of `bytes` in all to the host; without
    // them (too small, no memory, too few CPUs) copies go straight.
    void create(size_t bytes) {
        if (bytes < kLeastToHost || cpus() < 3) return;
        bool ok = hipHostMalloc((void**)&slots_, kSlots * kSlotBytes, hipHostMallocDefault) == hipSuccess;
        for (int i = 0; i < kSlots && ok; ++i)
            ok = hipEventCreateWithFlags(&done_[i], hipEventDisableTiming) == hipSuccess;
        if (!ok) {
            destroy();
            (void)hipGetLastError();
        }
    }
    void destroy() {
        for (hipEvent_t& e : done_) {
            if (e) (void)hipEventDestroy(e);
            e = nullptr;
        }
        if (slots_) (void)hipHostFree(slots_);
        slots_ = nullptr;
    }

    // Queues / performs the copies in stream order; the host arrays are complete
    // (to host) or read (to device) when the stream has been synchronised.
    hipError_t to_device(const HostCopy* copies, int count, hipStream_t stream) {
        return run(copies, count, stream, true);
    }
    hipError_t to_host(const HostCopy* copies, int count, hipStream_t stream) {
        return run(copies, count, stream, false);
    }

   private:
    struct Piece {
        char *host, *dev;
        size_t bytes;
    };
    static int pieces(const HostCopy& c) { return (int)((c.bytes + kSlotBytes - 1) / kSlotBytes); }
    static Piece piece(const HostCopy* c, int i) {
        for (; i >= pieces(*c); ++c) i -= pieces(*c);
        const size_t at = (size_t)i * kSlotBytes;
        return Piece{(char*)c->host + at, (char*)c->dev + at, std::min(kSlotBytes, c->bytes - at)};
    }

    static int cpus() {
        cpu_set_t set;
        return sched_getaffinity(0, sizeof(set), &set) == 0 ? CPU_COUNT(&set) : 1;
    }
    // memory the runtime does not know (a device, managed or pinned array is
    // copied straight)
    static bool pageable(const void* p) {
        hipPointerAttribute_t a{};
        if (hipPointerGetAttributes(&a, p) != hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
        return a.type == hipMemoryTypeUnregistered;
    }
    static hipError_t straight(const HostCopy* copies, int count, hipStream_t stream, bool toDevice) {
        for (int i = 0; i < count; ++i) {
            const HostCopy& c = copies[i];
            const hipError_t e = toDevice ? hipMemcpyAsync(c.dev, c.host, c.bytes, hipMemcpyHostToDevice, stream)
                                          : hipMemcpyAsync(c.host, c.dev, c.bytes, hipMemcpyDeviceToHost, stream);
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    }

    hipError_t run(const HostCopy* copies, int count, hipStream_t stream, bool toDevice) {
        size_t total = 0;
        int n = 0;
        bool staged = slots_ != nullptr;
        for (int i = 0; i < count; ++i) {
            const HostCopy& c = copies[i];
            total += c.bytes;
            n += pieces(c);
            staged = staged && pageable(c.host);
            // arrays that share memory are written one after the other
            for (int j = 0; j < i && !toDevice; ++j)
                staged = staged && ((char*)c.host + c.bytes <= (char*)copies[j].host ||
                                    (char*)copies[j].host + copies[j].bytes <= (char*)c.host);
        }
        if (!staged || total < (toDevice ? kLeastToDevice : kLeastToHost))
            return straight(copies, count, stream, toDevice);

        // piece i uses slot i % kSlots.  open: pieces whose slot a worker may use
        // (to host: the transfer has arrived; to device: the slot's last transfer
        // has left); filled[slot]: pieces the workers have finished there.
        std::atomic<int> next{0}, open{toDevice ? std::min(n, kSlots) : 0};
        std::atomic<int> filled[kSlots];
        for (auto& f : filled) f.store(0, std::memory_order_relaxed);
        std::atomic<bool> stop{false};
        auto work = [&] {
            for (;;) {
                const int i = next.fetch_add(1, std::memory_order_relaxed);
                if (i >= n) return;
                while (open.load(std::memory_order_acquire) <= i) {
                    if (stop.load(std::memory_order_relaxed)) return;
                    std::this_thread::yield();
                }
                const Piece p = piece(copies, i);
                char* slot = slots_ + (i % kSlots) * kSlotBytes;
                if (toDevice)
                    std::memcpy(slot, p.host, p.bytes);
                else
                    std::memcpy(p.host, slot, p.bytes);
                filled[i % kSlots].fetch_add(1, std::memory_order_release);
            }
        };
        std::thread workers[kWorkers];
        int started = 0;
        try {
            for (const int want = std::min(kWorkers, cpus() - 1); started < want; ++started)
                workers[started] = std::thread(work);
        } catch (...) {  // as many as the system gives
        }
        // none, or this thread is bound to one CPU (create() may have run on another
        // thread): nobody would fill or empty the slots
        if (started == 0) return straight(copies, count, stream, toDevice);

        // done(i): the workers have finished piece i (pieces of a slot in order)
        auto done = [&](int i) {
            return filled[i % kSlots].load(std::memory_order_acquire) > i / kSlots;
        };
        hipError_t e = hipSuccess;
        int issued = 0, landed = 0;  // transfers queued, transfers complete
        while (landed < n && e == hipSuccess) {
            const bool may = issued < n && (toDevice ? done(issued) : issued < kSlots || done(issued - kSlots));
            if (may) {
                const Piece p = piece(copies, issued);
                char* slot = slots_ + (issued % kSlots) * kSlotBytes;
                e = toDevice ? hipMemcpyAsync(p.dev, slot, p.bytes, hipMemcpyHostToDevice, stream)
                             : hipMemcpyAsync(slot, p.dev, p.bytes, hipMemcpyDeviceToHost, stream);
                if (e == hipSuccess) e = hipEventRecord(done_[issued % kSlots], stream);
                ++issued;
            }
            if (landed < issued && e == hipSuccess) {
                hipError_t q = hipEventQuery(done_[landed % kSlots]);
                if (q == hipSuccess) {
                    ++landed;
                    open.store(toDevice ? std::min(n, landed + kSlots) : landed, std::memory_order_release);
                } else if (q == hipErrorNotReady) {
                    (void)hipGetLastError();
                } else {
                    e = q;
                }
            } else if (!may) {
                std::this_thread::yield();
            }
        }
        if (e != hipSuccess) stop.store(true, std::memory_order_relaxed);
        for (int i = 0; i < started; ++i) workers[i].join();
        if (e != hipSuccess) (void)hipStreamSynchronize(stream);  // no transfer uses the slots any more
        return e;
    }

    char* slots_ = nullptr;
    hipEvent_t done_[kSlots] = {};
};

}  // namespace swe
