// host_stage.h — pageable host memory to the device at the link's rate.
//
// A plain hipMemcpyAsync from pageable memory is staged by the runtime on the
// calling thread: 82 MB of expert blobs (ten of gpu_expert_ffn's) took 3.0 ms
// (27 GB/s), half of what the link carries from pinned memory. Here a few
// threads copy the blobs into a ring of pinned slots while the calling thread
// hands the filled ones to the device in order: 1.81 ms for the same call with
// slots of 8 MiB (1.95 with 4, 2.19 with 2, whatever the thread count: the
// device's share of each copy counts). One per context (a context is one host
// thread's), threads and slots released with it; the threads take no signals
// and sleep between calls and while the ring is full.
#pragma once

#include <hip/hip_runtime.h>
#include <pthread.h>
#include <signal.h>
#include <stdint.h>
#include <string.h>

#include <atomic>
#include <condition_variable>
#include <mutex>
#include <thread>
#include <vector>

class HostStage {
  public:
    static constexpr size_t kPart = 512u << 10;             // what one thread copies at a time
    static constexpr int kParts = 16;                       // parts of a slot, one device copy
    static constexpr size_t kSlot = kPart * kParts;
    static constexpr int kSlots = 4, kThreads = 6;          // one thread copies 8-10 GB/s
    static constexpr uint64_t kMaxBytes = 120u << 20;       // of one run: ten blobs of 12 MiB

    // nullptr where the threads or the pinned memory cannot be had.
    static HostStage *create() {
        if (std::thread::hardware_concurrency() < kThreads + 2) return nullptr;
        HostStage *h = nullptr;
        try {
            h = new HostStage();
            if (h->init()) return h;
        } catch (...) {   // no exception leaves the C entry points
        }
        delete h;
        return nullptr;
    }

    ~HostStage() {
        {
            std::lock_guard<std::mutex> l(m_);
            quit_ = true;
        }
        cv_.notify_all();   // (no run is under way: its caller is ours)
        for (std::thread &t : threads_) t.join();
        for (hipEvent_t e : ev_)
            if (e) (void)hipEventDestroy(e);
        if (ring_) (void)hipHostFree(ring_);
    }

    // dst[0 .. n * bytes) = the n source blobs of `bytes` bytes each, one after
    // the other, on s (n * bytes <= kMaxBytes). Returns once every source byte
    // has been read; the last device copies may still be in flight from the ring.
    hipError_t run(const void *const *src, int n, uint64_t bytes, uint8_t *dst, hipStream_t s) {
        src_ = src;
        bytes_ = bytes;
        total_ = (uint64_t)n * bytes;
        n_ = (int)((total_ + kPart - 1) / kPart);
        const int units = (n_ + kParts - 1) / kParts;
        for (int u = 0; u < units; u++) done_[u].store(0, std::memory_order_relaxed);
        next_.store(0, std::memory_order_relaxed);
        limit_.store(kSlots, std::memory_order_relaxed);
        failed_.store(false, std::memory_order_relaxed);
        hipError_t err = hipSuccess;
        // the previous run's last copies may still be on their way from the ring
        for (int k = 0; k < kSlots && err == hipSuccess; k++)
            if (used_[k]) err = hipEventSynchronize(ev_[k]);
        if (err != hipSuccess) return err;
        active_.store(kThreads, std::memory_order_relaxed);
        {
            std::lock_guard<std::mutex> l(m_);
            job_++;
        }
        cv_.notify_all();
        for (int u = 0; u < units; u++) {
            // a slot is refilled once its copy has left: kept half a ring behind
            if (u >= kSlots / 2) {
                const int old = u - kSlots / 2;
                if (err == hipSuccess) err = hipEventSynchronize(ev_[old % kSlots]);
                {
                    std::lock_guard<std::mutex> l(m_);
                    if (err != hipSuccess) failed_.store(true, std::memory_order_relaxed);   // the slot may still be read: it is not refilled
                    limit_.store(old + 1 + kSlots, std::memory_order_release);
                }
                room_.notify_all();
            }
            const uint64_t off = (uint64_t)u * kSlot, len = total_ - off < kSlot ? total_ - off : kSlot;
            const int parts = (int)((len + kPart - 1) / kPart), k = u % kSlots;
            while (done_[u].load(std::memory_order_acquire) < parts) std::this_thread::yield();
            if (err == hipSuccess) err = hipMemcpyAsync(dst + off, ring_ + k * kSlot, len, hipMemcpyHostToDevice, s);
            if (err == hipSuccess) err = hipEventRecord(ev_[k], s);
            if (err == hipSuccess) used_[k] = true;
        }
        while (active_.load(std::memory_order_acquire) > 0) std::this_thread::yield();
        return err;
    }

  private:
    HostStage() : done_(kMaxBytes / kSlot + 1) {}

    bool init() {
        if (hipHostMalloc((void **)&ring_, kSlots * kSlot, hipHostMallocDefault) != hipSuccess) {
            ring_ = nullptr;
            (void)hipGetLastError();
            return false;
        }
        for (hipEvent_t &e : ev_)
            if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) return false;
        struct NoSignals {   // a new thread inherits the mask: the program's handlers stay on its own threads
            sigset_t old;
            NoSignals() { sigset_t all; sigfillset(&all); pthread_sigmask(SIG_SETMASK, &all, &old); }
            ~NoSignals() { pthread_sigmask(SIG_SETMASK, &old, nullptr); }
        } no_signals;
        for (int t = 0; t < kThreads; t++) threads_.emplace_back([this] { work(); });
        return true;
    }

    void part(int i) {   // bytes [i * kPart, ...) of the blobs into the ring
        uint64_t off = (uint64_t)i * kPart;
        const uint64_t end = off + kPart < total_ ? off + kPart : total_;
        uint8_t *to = ring_ + off % (kSlots * kSlot);
        while (off < end) {
            const uint64_t e = off / bytes_, w = off - e * bytes_;
            const uint64_t len = end - off < bytes_ - w ? end - off : bytes_ - w;
            memcpy(to, (const uint8_t *)src_[e] + w, len);
            to += len;
            off += len;
        }
    }

    void work() {
        uint64_t seen = 0;
        for (;;) {
            {
                std::unique_lock<std::mutex> l(m_);
                cv_.wait(l, [&] { return quit_ || job_ != seen; });
                if (quit_) return;
                seen = job_;
            }
            for (;;) {
                const int i = next_.fetch_add(1, std::memory_order_relaxed), u = i / kParts;
                if (i >= n_) break;
                if (limit_.load(std::memory_order_acquire) <= u) {   // the ring is full: a device copy away
                    std::unique_lock<std::mutex> l(m_);
                    room_.wait(l, [&] { return limit_.load(std::memory_order_relaxed) > u; });
                }
                // (after a failure failed_ is set before the limit that lets a refill in)
                if (u < kSlots || !failed_.load(std::memory_order_relaxed)) part(i);
                done_[u].fetch_add(1, std::memory_order_release);
            }
            active_.fetch_sub(1, std::memory_order_release);
        }
    }

    uint8_t *ring_ = nullptr;
    hipEvent_t ev_[kSlots] = {};
    bool used_[kSlots] = {};
    std::vector<std::thread> threads_;
    std::mutex m_;
    std::condition_variable cv_, room_;   // a new run (or the end), a slot to fill
    bool quit_ = false;
    std::atomic<bool> failed_{false};
    uint64_t job_ = 0;
    const void *const *src_ = nullptr;
    uint64_t bytes_ = 0, total_ = 0;
    int n_ = 0;
    std::atomic<int> next_{0}, limit_{0}, active_{0};
    std::vector<std::atomic<int>> done_;
};
