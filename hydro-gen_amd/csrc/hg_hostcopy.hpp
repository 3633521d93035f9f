// hg_hostcopy.hpp — copies between a caller's memory and the device; what
// follows is about pageable memory (of other memory see known()).
//
// The link moves 56 GB/s each way from pinned memory, one host thread copies
// from or to it at 28 GB/s, and the runtime's own path for pageable memory ran
// at 5 to 36 GB/s.  So a copy goes through a ring of pinned slots: while the
// link fills or drains some slots, this thread and a few helpers copy the
// pieces of the others.  A kernel fills the slots of a read (launch_copy_out, where
// the reason is), the runtime's copies empty those of a write.  Measured, us, against one copy of
// up to 16 MB and then one memcpy (reads) or the runtime's path (writes, a batch's
// reads): 64 MB to the host 2600 -> 1520, 16 MB 850 -> 398 (a batch's plane 950),
// 4 MB 232 -> 122; 64 MB to the device 2300 -> 1670.  Slots of 1 MB leave the link
// idle between copies (16 MB in 431 us), of 4 MB the helpers (4 MB in 148 us); 6
// helpers or 8 slots gain nothing over 3 and 4.
//
// A HostCopy belongs to one context or batch and is used by its one host
// thread.  The pinned slots (8 MB) and the helper threads are made when first
// needed, sleep between copies, and end with the object.  At most kCrews objects
// of a process have helpers at a time; the others copy by their own thread.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <thread>

#include "hg_kernels.hpp"

class HostCopy {
public:
    HostCopy() = default;
    HostCopy(const HostCopy&) = delete;
    HostCopy& operator=(const HostCopy&) = delete;
    ~HostCopy() {
        {
            std::lock_guard<std::mutex> lk(mu_);
            stop_ = true;
        }
        cv_.notify_all();
        for (std::thread& t : helper_)
            if (t.joinable()) t.join();
        if (counted_) crews().fetch_sub(1);
        for (int i = 0; i < kSlots; ++i) {
            if (pin_[i]) (void)hipHostFree(pin_[i]);
            if (ev_[i]) (void)hipEventDestroy(ev_[i]);
        }
    }

    // `bytes` from device `src` to `dst`, after the work on `s`; returns when
    // dst is filled.
    hipError_t to_host(const void* src, void* dst, size_t bytes, hipStream_t s) {
        if (bytes == 0) return hipSuccess;
        hipError_t e = hipSuccess;
        if (known(dst) || bytes % 16 || (e = reserve(bytes)) != hipSuccess)
            return direct(dst, src, bytes, hipMemcpyDeviceToHost, s);
        const char* from = static_cast<const char*>(src);
        const size_t chunks = (bytes + kSlot - 1) / kSlot;
        auto enqueue = [&](size_t c) {
            const size_t off = c * kSlot;
            const hipError_t r = hgk::launch_copy_out(pin_[c % kSlots], from + off, chunk_bytes(bytes, c), s);
            return r != hipSuccess ? r : hipEventRecord(ev_[c % kSlots], s);
        };
        for (size_t c = 0; c < chunks && c < kSlots && e == hipSuccess; ++c) e = enqueue(c);
        bool begun = false;
        for (size_t c = 0; c < chunks && e == hipSuccess; ++c) {
            e = hipEventSynchronize(ev_[c % kSlots]);
            if (e != hipSuccess) break;
            if (!begun) {                                     // the helpers wait for data, not for the GPU's queue
                begin(static_cast<char*>(dst), nullptr, bytes);
                begun = true;
            }
            copy_chunk(c);
            if (c + kSlots < chunks) e = enqueue(c + kSlots);
        }
        if (begun) end();
        if (e != hipSuccess) (void)hipStreamSynchronize(s);   // no copy may write the slots after this
        return e;
    }

    // `bytes` from `src` to device `dst`, in order with the work on `s`;
    // returns when the device holds them or, without `wait`, when they are on their
    // way: the caller then waits for the stream before it gives src back or copies
    // again.
    hipError_t to_device(const void* src, void* dst, size_t bytes, hipStream_t s, bool wait = true) {
        hipError_t e = hipSuccess;
        const bool first = !wrote_ && !pin_[0];
        wrote_ = true;
        if (bytes < kRingWrite || first || known(src) || (e = reserve(bytes)) != hipSuccess)
            return direct(dst, src, bytes, hipMemcpyHostToDevice, s, wait);
        const size_t chunks = (bytes + kSlot - 1) / kSlot;
        begin(nullptr, static_cast<const char*>(src), bytes);
        for (size_t c = 0; c < chunks && e == hipSuccess; ++c) {
            if (c >= kSlots) e = hipEventSynchronize(ev_[c % kSlots]);
            if (e != hipSuccess) break;
            copy_chunk(c);
            e = hipMemcpyAsync(static_cast<char*>(dst) + c * kSlot, pin_[c % kSlots], chunk_bytes(bytes, c),
                               hipMemcpyHostToDevice, s);
            if (e == hipSuccess) e = hipEventRecord(ev_[c % kSlots], s);
        }
        end();
        if (!wait) return e;
        const hipError_t w = hipStreamSynchronize(s);         // the slots are free again, whatever happened
        return e != hipSuccess ? e : w;
    }

private:
    static constexpr size_t kSlot = size_t(2) << 20;
    static constexpr size_t kSlots = 4;
    static constexpr size_t kPiece = size_t(128) << 10;       // what a thread copies at a time
    static constexpr size_t kPiecesPerSlot = kSlot / kPiece;
    static constexpr size_t kCrewMin = size_t(1) << 20;       // smaller copies are over before a helper wakes
    static constexpr int kHelpers = 3;
    // Smaller writes, and the first of a new object, take the runtime's own path:
    // the ring gains nothing on the former, and its slots and helpers cost the
    // latter more than one write gains.  us by the runtime / by the ring, for a
    // plane of one of three states of 9 planes written in turn, of a state that is
    // new, for a single plane of new data, and for the first write of a new object:
    //    1 MB    66/53      56/57      53/61      57/123
    //    2 MB   111/101    109/107     91/110     94/191
    //    4 MB   176/140    187/157    135/153    139/234
    //   16 MB   590/455    643/475    483/505    506/647
    static constexpr size_t kRingWrite = size_t(4) << 20;
    // a helper without work yields this often (some 0.1 ms, a few slots' time on
    // the link) and then sleeps: a copy may be queued behind seconds of GPU work
    static constexpr int kIdleYields = 256;
    static constexpr int kCrews = 32;                         // more copying at once than a host has links or cores for

    static std::atomic<int>& crews() {
        static std::atomic<int> n{0};
        return n;
    }

    static size_t chunk_bytes(size_t bytes, size_t c) { return std::min(kSlot, bytes - c * kSlot); }
    static size_t pieces_of(size_t bytes) { return (bytes + kPiece - 1) / kPiece; }

    // Whether the caller's memory is the runtime's: pinned, which the link reaches
    // without a second copy (16 MB in 300 us, 435 through the ring), managed, or a
    // device's, which is not the host's to copy.  The question costs 0.4 us.
    static bool known(const void* p) {
        hipPointerAttribute_t a{};
        if (hipPointerGetAttributes(&a, p) != hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
        return a.type != hipMemoryTypeUnregistered;
    }

    // The runtime's own path; also when no more can be pinned.
    static hipError_t direct(void* dst, const void* src, size_t bytes, hipMemcpyKind kind, hipStream_t s,
                             bool wait = true) {
        const hipError_t e = hipMemcpyAsync(dst, src, bytes, kind, s);
        return e != hipSuccess || !wait ? e : hipStreamSynchronize(s);
    }

    hipError_t reserve(size_t bytes) {
        for (size_t i = 0; i < kSlots && i * kSlot < bytes; ++i) {   // each piece stored only once it exists
            if (!pin_[i]) {
                void* p = nullptr;
                const hipError_t e = hipHostMalloc(&p, kSlot, hipHostMallocCoherent);
                if (e != hipSuccess) {
                    (void)hipGetLastError();                  // the caller's other path is not to find it
                    return e;
                }
                pin_[i] = static_cast<char*>(p);
            }
            if (!ev_[i]) {
                hipEvent_t v = nullptr;
                const hipError_t e = hipEventCreateWithFlags(&v, hipEventDisableTiming);
                if (e != hipSuccess) {
                    (void)hipGetLastError();
                    return e;
                }
                ev_[i] = v;
            }
        }
        return hipSuccess;
    }

    // Starts a copy of the slots' contents to `to`, or of `from` to the slots.
    void begin(char* to, const char* from, size_t bytes) {
        to_ = to;
        from_ = from;
        bytes_ = bytes;
        next_.store(0, std::memory_order_relaxed);
        limit_.store(0, std::memory_order_relaxed);
        over_.store(false, std::memory_order_relaxed);
        for (auto& d : done_) d.store(0, std::memory_order_relaxed);
        if (bytes < kCrewMin) return;
        if (!counted_) {                                      // at each copy: another object may have gone
            counted_ = crews().fetch_add(1) < kCrews;
            if (!counted_) crews().fetch_sub(1);
            try {
                if (counted_)
                    for (std::thread& t : helper_) t = std::thread([this] { help(); });
            } catch (...) {                                   // no threads to be had: fewer helpers, or none
            }
        }
        {
            std::lock_guard<std::mutex> lk(mu_);
            active_ = true;
            ++job_;
        }
        cv_.notify_all();
    }

    // Copies chunk c's pieces together with the helpers.
    void copy_chunk(size_t c) {
        const size_t first = c * kPiecesPerSlot;
        const size_t last = first + pieces_of(chunk_bytes(bytes_, c));
        limit_.store(last);
        wake();
        while (copy_piece()) {
        }
        std::atomic<size_t>& d = done_[c % kSlots];
        while (d.load(std::memory_order_acquire) != last - first) std::this_thread::yield();
        d.store(0, std::memory_order_relaxed);
    }

    // Copies the next piece that is there to be copied; false if there is none.
    bool copy_piece() {
        size_t p = next_.load(std::memory_order_relaxed);
        do {
            if (p >= limit_.load(std::memory_order_acquire)) return false;
        } while (!next_.compare_exchange_weak(p, p + 1, std::memory_order_relaxed));
        const size_t off = p * kPiece, len = std::min(kPiece, bytes_ - off);
        char* slot = pin_[off / kSlot % kSlots] + off % kSlot;
        if (to_)
            std::memcpy(to_ + off, slot, len);
        else
            std::memcpy(slot, from_ + off, len);
        done_[off / kSlot % kSlots].fetch_add(1, std::memory_order_release);
        return true;
    }

    void end() {
        if (bytes_ < kCrewMin) return;
        {
            std::lock_guard<std::mutex> lk(mu_);
            active_ = false;                                  // no helper joins any more
        }
        over_.store(true);
        wake();
        while (inside_.load(std::memory_order_acquire) != 0) std::this_thread::yield();
    }

    // Wakes the helpers that went to sleep within a copy.  (What they look at is
    // stored before parked_ is read here, and they raise parked_ before they look:
    // one of the two sees the other.)
    void wake() {
        if (parked_.load() == 0) return;
        { std::lock_guard<std::mutex> lk(mu_); }
        cv_.notify_all();
    }

    void help() {
        unsigned long long seen = 0;
        std::unique_lock<std::mutex> lk(mu_);
        for (;;) {
            cv_.wait(lk, [&] { return stop_ || (active_ && job_ != seen); });
            if (stop_) return;
            seen = job_;
            inside_.fetch_add(1, std::memory_order_relaxed);
            lk.unlock();
            for (int idle = 0; !over_.load(std::memory_order_acquire);) {
                if (copy_piece()) {
                    idle = 0;
                } else if (++idle < kIdleYields) {
                    std::this_thread::yield();
                } else {
                    idle = 0;
                    lk.lock();
                    parked_.fetch_add(1);
                    cv_.wait(lk, [&] { return over_.load() || next_.load() < limit_.load(); });
                    parked_.fetch_sub(1);
                    lk.unlock();
                }
            }
            inside_.fetch_sub(1, std::memory_order_release);
            lk.lock();
        }
    }

    bool wrote_ = false;
    char* pin_[kSlots] = {};
    hipEvent_t ev_[kSlots] = {};
    // the copy in progress
    char* to_ = nullptr;
    const char* from_ = nullptr;
    size_t bytes_ = 0;
    std::atomic<size_t> next_{0}, limit_{0}, done_[kSlots] = {};
    std::atomic<bool> over_{true};
    std::atomic<int> inside_{0}, parked_{0};
    // the helpers
    std::thread helper_[kHelpers];
    bool counted_ = false;
    std::mutex mu_;
    std::condition_variable cv_;
    bool stop_ = false, active_ = false;
    unsigned long long job_ = 0;
};
