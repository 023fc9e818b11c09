// host_copy.hpp -- copies between a caller's (pageable) arrays and device memory.
//
// hipMemcpy on pageable memory moves the data through the runtime's own staging on one thread, and the
// first touch of a fresh destination (numpy's empty/zeros) costs that same thread a page fault for every
// page: 128 MB to fresh pages 14.9 ms (9 GB/s), to touched pages 7.3, from them 4.3, where the link does
// 57 GB/s. HostCopy cuts the array into 2 MB chunks that up to four threads (the caller's among them)
// take in turn; each thread has two pinned chunks, so that the DMA of one runs while the other is copied
// by the CPU: 3.8 / 3.4 / 3.4 ms. Two threads leave fresh pages at 6.9 ms, eight change nothing (3.8);
// 1 MB chunks cost 4.7, 4 MB the same with twice the pinned memory. From 8 MB on (four chunks) it is
// ahead in each direction (16 MB: 1.9 -> 0.65, 0.9 -> 0.5, 0.6 -> 0.5 ms); 2 MB is level (0.12-0.25).
//
// The pinned chunks (16 MB) are one buffer of the process: made by the first context that copies a large
// array, shared by all that follow while one of them lives, given back with the last. The first of a process
// costs 0.6 ms, one made after it was given back 15 us (the runtime keeps freed ones), so contexts that live for
// one state gain as well: open, set, step, read and close 6.6 -> 6.0 ms at 64^3, 16.8 -> 13.6 at 96^3,
// 36.4 -> 32.8 at 128^3. The threads live within one call. A copy that finds the buffer
// in use, or cannot have it, is a plain hipMemcpy.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <memory>
#include <mutex>
#include <thread>

namespace laps {

class HostCopy {
  public:
    static constexpr size_t kChunk = size_t(2) << 20;
    static constexpr size_t kMin = 4 * kChunk;
    static constexpr int kThreads = 4;

    // n bytes from src (device) to dst (host), after what `s` holds; returns when dst is written
    hipError_t to_host(void* dst, const void* src, size_t n, int device, hipStream_t s) {
        return copy((char*)dst, (char*)const_cast<void*>(src), n, true, device, s);
    }
    // n bytes from src (host) to dst (device), after what `s` holds; returns when dst is written
    hipError_t to_device(void* dst, const void* src, size_t n, int device, hipStream_t s) {
        return copy((char*)const_cast<void*>(src), (char*)dst, n, false, device, s);
    }
    void release() {
        for (hipEvent_t& e : ev_) {
            if (e) (void)hipEventDestroy(e);
            e = nullptr;
        }
        ring_.reset();
    }

  private:
    struct Ring {
        char* p = nullptr;
        std::mutex busy;  // one copy at a time
        ~Ring() {
            if (p) (void)hipHostFree(p);
        }
    };
    // the process's buffer, made if no context holds one; null without memory for it
    static std::shared_ptr<Ring> shared_ring() {
        static std::mutex mu;
        static std::weak_ptr<Ring> last;
        std::lock_guard<std::mutex> lk(mu);
        std::shared_ptr<Ring> r = last.lock();
        if (!r) {
            r = std::make_shared<Ring>();
            if (hipHostMalloc((void**)&r->p, 2 * kThreads * kChunk, hipHostMallocPortable) != hipSuccess) {
                r->p = nullptr;
                return nullptr;
            }
            last = r;
        }
        return r;
    }
    static hipError_t plain(char* host, char* dev, size_t n, bool down, hipStream_t s) {
        hipError_t e = hipStreamSynchronize(s);
        if (e != hipSuccess) return e;
        return down ? hipMemcpy(host, dev, n, hipMemcpyDeviceToHost) : hipMemcpy(dev, host, n, hipMemcpyHostToDevice);
    }
    bool prepare() {
        if (ring_) return true;
        bool ok = true;
        try {
            ring_ = shared_ring();
        } catch (...) {
        }
        for (hipEvent_t& e : ev_) ok = ok && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
        if (!ok || !ring_) {
            release();
            (void)hipGetLastError();  // the plain copy reports its own
        }
        return ring_ != nullptr;
    }
    hipError_t copy(char* host, char* dev, size_t n, bool down, int device, hipStream_t s) {
        std::unique_lock<std::mutex> lk(mu_, std::try_to_lock);
        if (n < kMin || !lk.owns_lock() || !prepare()) return plain(host, dev, n, down, s);
        std::unique_lock<std::mutex> own(ring_->busy, std::try_to_lock);
        if (!own.owns_lock()) return plain(host, dev, n, down, s);
        char* const ring = ring_->p;
        std::atomic<size_t> next{0};
        std::atomic<int> bad{(int)hipSuccess};
        // the chunks are handed out in order; a thread's two slots and events are its own
        auto work = [&](int t) {
            const auto check = [&](hipError_t e) {
                if (e != hipSuccess) bad = (int)e;
                return e == hipSuccess;
            };
            if (!check(hipSetDevice(device))) return;
            size_t at[2], len[2] = {0, 0};  // what a slot's last transfer carries (0: nothing)
            for (int k = 0; bad == (int)hipSuccess; k ^= 1) {
                char* slot = ring + (size_t)(2 * t + k) * kChunk;
                hipEvent_t e = ev_[2 * t + k];
                const size_t o = next.fetch_add(1) * kChunk;
                const bool more = o < n;
                if (!down && !more) return;  // the caller waits for the stream
                if (more) {
                    const size_t l = std::min(kChunk, n - o);
                    if (!down) {
                        if (len[k] && !check(hipEventSynchronize(e))) return;
                        std::memcpy(slot, host + o, l);
                    }
                    if (!check(down ? hipMemcpyAsync(slot, dev + o, l, hipMemcpyDeviceToHost, s)
                                    : hipMemcpyAsync(dev + o, slot, l, hipMemcpyHostToDevice, s)) ||
                        !check(hipEventRecord(e, s)))
                        return;
                    at[k] = o;
                    len[k] = l;
                }
                if (down) {  // the other slot's chunk, while this one's is on its way
                    const int q = k ^ 1;
                    if (len[q]) {
                        if (!check(hipEventSynchronize(ev_[2 * t + q]))) return;
                        std::memcpy(host + at[q], ring + (size_t)(2 * t + q) * kChunk, len[q]);
                        len[q] = 0;
                    }
                    if (!more) return;
                }
            }
        };
        const int nt = (int)std::min<size_t>(std::min<unsigned>(kThreads, std::max(1u, std::thread::hardware_concurrency())),
                                             (n + kChunk - 1) / kChunk);
        std::thread th[kThreads];
        for (int t = 1; t < nt; ++t) {
            try {
                th[t] = std::thread(work, t);
            } catch (...) {
                break;  // no thread to be had: the others take its chunks
            }
        }
        work(0);
        for (std::thread& x : th)
            if (x.joinable()) x.join();
        const hipError_t e = hipStreamSynchronize(s);  // nothing in flight reads or writes the slots after this
        return bad != (int)hipSuccess ? (hipError_t)bad.load() : e;
    }

    std::shared_ptr<Ring> ring_;
    hipEvent_t ev_[2 * kThreads] = {};
    std::mutex mu_;  // this object's events: one copy at a time
};

}  // namespace laps
