// Copies of device arrays into ordinary host memory.
//
// hipMemcpyAsync into pageable memory goes through the runtime's own staging
// buffer, one megabyte and one host thread at a time, and the thread also takes
// the page faults of a fresh array: 10 GB/s for 2-4 GB of fields, and 115 us a call for
// 256 KiB.  Here the device copies into pinned slots at the link's rate (50 GB/s
// in 4 MiB pieces, 38 in 1 MiB) while a few threads move finished slots on
// (4 GB of fields: 41-46 GB/s with four threads and 4 MiB pieces, 24-27 with
// two, no more with eight); a small read is one wait and one memcpy.  Read of
// the four fields, ms, before / after: TGV 512^3 416 / 94, 256^3 52.6 / 12.6, channel
// 512x256x256 103 / 24, cavity 128^3 7.8 / 2.4, TGV 32^3 0.20 / 0.10, 15 ensemble members
// 27.4 / 11.6.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <thread>
#include <vector>

namespace imx {

class ReadBack {
  public:
    struct Part {
        void *dst;
        const void *src;
        size_t bytes;
    };

    ReadBack() = default;
    ReadBack(const ReadBack &) = delete;
    ReadBack &operator=(const ReadBack &) = delete;
    ~ReadBack() { release(); }

    // Copies the parts, ordered after the work queued on `st`, and returns when
    // all of them are in place.  A destination that the runtime knows (pinned,
    // managed or device memory) is copied to directly.
    hipError_t copy(const Part *parts, int n, int device, hipStream_t st)
    {
        size_t total = 0;
        bool plain = false;
        for (int k = 0; k < n; ++k) {
            total += parts[k].bytes;
            plain = plain || known(parts[k].dst);
        }
        hipError_t e = hipErrorNotReady;
        if (!plain) {
            try {
                e = total <= SMALL ? copy_small(parts, n, total, st) : copy_large(parts, n, total, device, st);
            } catch (...) {  // no memory or no thread: nothing is in flight
                e = hipErrorNotReady;
            }
        }
        if (e != hipErrorNotReady) return e;
        for (int k = 0; k < n; ++k)
            if ((e = hipMemcpyAsync(parts[k].dst, parts[k].src, parts[k].bytes, hipMemcpyDeviceToHost, st)) != hipSuccess) return e;
        return hipStreamSynchronize(st);
    }

    void release()
    {
        if (pin_) (void)hipHostFree(pin_);
        pin_ = nullptr;
        cap_ = 0;
        for (hipEvent_t &e : ev_) {
            if (e) (void)hipEventDestroy(e);
            e = nullptr;
        }
    }

  private:
    static constexpr size_t MIB = size_t(1) << 20;
    static constexpr size_t SMALL = 2 * MIB;  // below, starting threads costs what they save
    static constexpr int THREADS = 4, SLOTS = 2 * THREADS;

    static bool known(const void *p)
    {
        hipPointerAttribute_t a;
        const bool ok = hipPointerGetAttributes(&a, p) == hipSuccess;
        if (!ok) (void)hipGetLastError();
        return ok && a.type != hipMemoryTypeUnregistered;
    }

    // Pinned memory of at least `bytes`; false (and none held) if there is none.
    bool hold(size_t bytes)
    {
        if (cap_ >= bytes) return true;
        if (pin_) (void)hipHostFree(pin_);
        cap_ = 0;
        if (hipHostMalloc((void **)&pin_, bytes, 0) != hipSuccess) {
            (void)hipGetLastError();
            pin_ = nullptr;
            return false;
        }
        cap_ = bytes;
        return true;
    }

    hipError_t copy_small(const Part *parts, int n, size_t total, hipStream_t st)
    {
        if (!hold(std::max<size_t>(total, 4096))) return hipErrorNotReady;
        size_t at = 0;
        for (int k = 0; k < n; ++k) {
            const hipError_t e = hipMemcpyAsync(pin_ + at, parts[k].src, parts[k].bytes, hipMemcpyDeviceToHost, st);
            if (e != hipSuccess) {
                (void)hipStreamSynchronize(st);
                return e;
            }
            at += parts[k].bytes;
        }
        const hipError_t e = hipStreamSynchronize(st);
        if (e != hipSuccess) return e;
        at = 0;
        for (int k = 0; k < n; ++k) {
            std::memcpy(parts[k].dst, pin_ + at, parts[k].bytes);
            at += parts[k].bytes;
        }
        return hipSuccess;
    }

    hipError_t copy_large(const Part *parts, int n, size_t total, int device, hipStream_t st)
    {
        // pieces of 1 to 4 MiB, so that a read of a few MiB overlaps too
        const size_t piece = std::min(4 * MIB, std::max(MIB, (total / 32 + MIB - 1) / MIB * MIB));
        if (!hold(piece * SLOTS)) return hipErrorNotReady;
        for (hipEvent_t &e : ev_)
            if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
                (void)hipGetLastError();
                return hipErrorNotReady;
            }
        std::vector<Part> work;
        for (int k = 0; k < n; ++k)
            for (size_t o = 0; o < parts[k].bytes; o += piece)
                work.push_back({(char *)parts[k].dst + o, (const char *)parts[k].src + o, std::min(piece, parts[k].bytes - o)});
        const int pieces = (int)work.size();
        // wait for the steps here, not in every thread
        hipError_t e = hipStreamSynchronize(st);
        if (e != hipSuccess) return e;

        std::atomic<int> queued{0}, next{0}, failed{(int)hipSuccess};
        std::atomic<int> freed[SLOTS];  // pieces that have left the slot
        for (auto &f : freed) f = 0;
        auto worker = [&]() {
            (void)hipSetDevice(device);
            for (;;) {
                const int k = next.fetch_add(1);
                if (k >= pieces) return;
                while (queued.load(std::memory_order_acquire) <= k) {
                    if (failed.load() != (int)hipSuccess) return;
                    std::this_thread::yield();
                }
                const hipError_t w = hipEventSynchronize(ev_[k % SLOTS]);
                if (w != hipSuccess) {
                    failed.store((int)w);
                    return;
                }
                std::memcpy(work[k].dst, pin_ + (size_t)(k % SLOTS) * piece, work[k].bytes);
                freed[k % SLOTS].store(k / SLOTS + 1, std::memory_order_release);
            }
        };
        const int want = std::min({THREADS, pieces, std::max(1, (int)std::thread::hardware_concurrency())});
        std::vector<std::thread> threads;
        threads.reserve((size_t)want);
        try {
            for (int t = 0; t < want; ++t) threads.emplace_back(worker);
        } catch (...) {
            if (threads.empty()) return hipErrorNotReady;
        }
        for (int k = 0; k < pieces && e == hipSuccess; ++k) {
            while (freed[k % SLOTS].load(std::memory_order_acquire) < k / SLOTS && failed.load() == (int)hipSuccess)
                std::this_thread::yield();
            if (failed.load() != (int)hipSuccess) break;
            e = hipMemcpyAsync(pin_ + (size_t)(k % SLOTS) * piece, work[k].src, work[k].bytes, hipMemcpyDeviceToHost, st);
            if (e == hipSuccess) e = hipEventRecord(ev_[k % SLOTS], st);
            if (e == hipSuccess) queued.store(k + 1, std::memory_order_release);
            else failed.store((int)e);
        }
        for (auto &t : threads) t.join();
        if (failed.load() != (int)hipSuccess) {
            (void)hipStreamSynchronize(st);
            return (hipError_t)failed.load();
        }
        return hipSuccess;
    }

    char *pin_ = nullptr;  // at most SLOTS pieces of 4 MiB
    size_t cap_ = 0;
    hipEvent_t ev_[SLOTS] = {};
};

}  // namespace imx
