// Copies of device arrays into ordinary host memory.
//
// hipMemcpyAsync into pageable memory goes through the runtime's own staging
// buffer, one megabyte and one host thread at a time, and the thread also takes
// the page faults of a fresh array: 10 GB/s for 2-4 GB of fields, and 115 us a call for
// 256 KiB.  Here the device copies into pinned slots by a kernel of its own
// (aux.hip k_copy_out; hipMemcpyAsync leaves 11 us between copies) while a few threads
// move finished slots on: GB/s for 512 MB / 4 GB of fields 37 / 44 with four
// threads, 42 / 46.5 with six, no more with eight.  A small read is one launch for
// all its arrays, one wait and one memcpy: TGV 32^3 fields 95 -> 71 us and diagnostics
// 31 -> 22 against one hipMemcpyAsync each.  Read of the four fields, ms, before any of
// this / after: TGV 512^3 416 / 93, 256^3 52.6 / 12.7, channel 512x256x256 103 / 24,
// cavity 128^3 7.8 / 2.3, TGV 32^3 0.20 / 0.07, 15 ensemble members 27.4 / 11.6.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

#include "kernels.h"

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
    // managed or device memory) is copied to directly.  Reads of several threads
    // take turns: they share the slots (an uncontended lock costs some 20 ns).
    hipError_t copy(const Part *parts, int n, int device, hipStream_t st)
    {
        std::lock_guard<std::mutex> turn(m_);
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
    static constexpr int THREADS = 6, SLOTS = 2 * THREADS;

    static bool known(const void *p)
    {
        hipPointerAttribute_t a;
        const bool ok = hipPointerGetAttributes(&a, p) == hipSuccess;
        if (!ok) (void)hipGetLastError();
        return ok && a.type != hipMemoryTypeUnregistered;
    }

    // The room of `bytes` in pinned memory: whole 16-byte units.
    static size_t held(size_t bytes) { return (bytes + 15) / 16 * 16; }

    // Up to four parts into pinned memory, one launch.
    static hipError_t copy_out(const Part *parts, int n, char *pinned, hipStream_t st)
    {
        CopyOut c{};
        for (int k = 0; k < 4; ++k) {
            c.src[k] = k < n ? (const char *)parts[k].src : nullptr;
            c.bytes[k] = k < n ? parts[k].bytes : 0;
            c.at[k + 1] = c.at[k] + held(c.bytes[k]) / 16;
        }
        hipError_t e = hipHostGetDevicePointer((void **)&c.dst, pinned, 0);
        return e == hipSuccess ? launch_copy_out(c, st) : e;
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
        if (!hold(std::max<size_t>(total + 16 * (size_t)n, 4096))) return hipErrorNotReady;
        size_t at = 0;
        hipError_t e = hipSuccess;
        for (int k = 0; k < n && e == hipSuccess; k += 4) {
            const int m = std::min(4, n - k);
            e = copy_out(parts + k, m, pin_ + at, st);
            for (int i = k; i < k + m; ++i) at += held(parts[i].bytes);
        }
        const hipError_t w = hipStreamSynchronize(st);
        if (e != hipSuccess || w != hipSuccess) return e != hipSuccess ? e : w;
        at = 0;
        for (int k = 0; k < n; ++k) {
            std::memcpy(parts[k].dst, pin_ + at, parts[k].bytes);
            at += held(parts[k].bytes);
        }
        return hipSuccess;
    }

    hipError_t copy_large(const Part *parts, int n, size_t total, int device, hipStream_t st)
    {
        // pieces of 1 or 2 MiB, so that a read of a few MiB overlaps too (4 GB of
        // fields: 42 / 46 / 46 GB/s in 1 / 2 / 4 MiB pieces; the first read of a handle, which
        // allocates the slots, 256^3: 13.9 ms with 2 MiB, 16 with 4)
        const size_t piece = std::min(2 * MIB, std::max(MIB, (total / 32 + MIB - 1) / MIB * MIB));
        std::vector<Part> work;
        for (int k = 0; k < n; ++k)
            for (size_t o = 0; o < parts[k].bytes; o += piece)
                work.push_back({(char *)parts[k].dst + o, (const char *)parts[k].src + o, std::min(piece, parts[k].bytes - o)});
        const int pieces = (int)work.size(), slots = std::min(SLOTS, pieces);
        // (pinning memory takes longer than copying into it: no slot that stays empty)
        if (!hold(piece * (size_t)slots)) return hipErrorNotReady;
        for (int k = 0; k < slots; ++k)
            if (!ev_[k] && hipEventCreateWithFlags(&ev_[k], hipEventDisableTiming) != hipSuccess) {
                (void)hipGetLastError();
                return hipErrorNotReady;
            }
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
            e = copy_out(&work[k], 1, pin_ + (size_t)(k % SLOTS) * piece, st);
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

    std::mutex m_;
    char *pin_ = nullptr;  // at most SLOTS pieces of 2 MiB
    size_t cap_ = 0;
    hipEvent_t ev_[SLOTS] = {};
};

}  // namespace imx
