// Large results from device memory into a caller's pageable array: a ring of
// pinned slots that the copy engine fills in order and a few threads empty.
//
// What bounds it: a plain copy into an array that was just allocated runs at
// 9 GB/s (the runtime stages it through one thread, which also takes the
// array's page faults), the link at 54 GB/s, one thread's memcpy into fresh pages
// at 12, five threads' at 40.  36 MB: 4.1 -> 1.1 ms, 65 MB: 6.7 -> 1.8 ms.
#pragma once

#include <hip/hip_runtime.h>

#include <condition_variable>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace mafm {

class HostLink {
   public:
    // A transfer below this goes by one plain copy (1 MB: 0.07 ms plainly, 0.17
    // with threads to wake; 16 MB: 1.2 against 0.55).
    static constexpr size_t MIN_BYTES = 4u << 20;
    // The ring and its threads take 0.7 to 1.4 ms to set up (5 in a process's first
    // use), what they save on some 25 MB: a context that transfers less never has
    // them (one 14 MB result of a fresh context: plainly 1.0 ms, with them 1.3).
    static constexpr size_t OPEN_BYTES = 32u << 20;

    HostLink() = default;
    HostLink(const HostLink&) = delete;
    HostLink& operator=(const HostLink&) = delete;
    ~HostLink() { close(); }

    // dst <- src (device memory) behind the work queued on st; complete on return.
    hipError_t to_host(void* dst, const void* src, size_t bytes, int device, hipStream_t st) {
        if (bytes < MIN_BYTES || !pageable(dst) || !worth(bytes) || !open(device)) {
            hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st);
            return e == hipSuccess ? hipStreamSynchronize(st) : e;
        }
        const size_t n = (bytes + SLOT - 1) / SLOT;
        auto size = [&](size_t k) { return k + 1 < n ? SLOT : bytes - SLOT * (n - 1); };
        hipError_t err = hipSuccess;
        size_t queued = 0, given = 0;
        while (given < n && err == hipSuccess) {
            // keep the engine busy: refill every slot that has been emptied
            while (queued < n && queued < given + SLOTS && err == hipSuccess && emptied(queued, queued == given)) {
                const int s = (int)(queued % SLOTS);
                err = hipMemcpyAsync(ring_ + SLOT * s, static_cast<const char*>(src) + SLOT * queued, size(queued),
                                     hipMemcpyDeviceToHost, st);
                if (err == hipSuccess) err = hipEventRecord(ev_[s], st);
                if (err == hipSuccess) ++queued;
            }
            if (err != hipSuccess) break;
            const int s = (int)(given % SLOTS);
            err = hipEventSynchronize(ev_[s]);
            if (err != hipSuccess) break;
            give({static_cast<char*>(dst) + SLOT * given, ring_ + SLOT * s, size(given)});
            ++given;
        }
        // every slot that was given out is emptied, also after an error
        std::unique_lock<std::mutex> l(m_);
        idle_.wait(l, [&] { return done_ == jobs_; });
        l.unlock();
        if (err != hipSuccess) (void)hipStreamSynchronize(st);   // no copy into the ring is left running
        return err;
    }

   private:
    static constexpr size_t SLOT = 2u << 20;
    static constexpr int SLOTS = 8, THREADS = 5;
    struct Job {
        char* dst;
        const char* src;
        size_t bytes;
    };

    char* ring_ = nullptr;
    size_t plain_ = 0;                         // bytes of the transfers so far that it might have taken
    hipEvent_t ev_[SLOTS] = {};
    int n_ev_ = 0;
    bool failed_ = false;
    std::vector<std::thread> threads_;
    std::mutex m_;
    std::condition_variable work_, idle_;
    Job job_[SLOTS];
    size_t jobs_ = 0, taken_ = 0, done_ = 0;   // numbered through the link's life
    bool slot_full_[SLOTS] = {};
    bool stop_ = false;

    // Memory the runtime knows (pinned, managed, a device's) keeps the plain copy.
    static bool pageable(const void* p) {
        hipPointerAttribute_t a{};
        if (hipPointerGetAttributes(&a, p) != hipSuccess) {
            (void)hipGetLastError();   // older runtimes report unknown memory as an error
            return true;
        }
        return a.type == hipMemoryTypeUnregistered;
    }

    bool worth(size_t bytes) {
        if (!ring_) plain_ += bytes;
        return ring_ || plain_ >= OPEN_BYTES;
    }

    bool open(int device) {
        if (ring_) return true;
        if (failed_) return false;
        failed_ = true;
        int current = device;
        (void)hipGetDevice(&current);
        (void)hipSetDevice(device);   // the events belong to the stream's device
        const bool ok = make();
        (void)hipSetDevice(current);
        if (!ok) close();
        failed_ = !ok;
        return ok;
    }

    bool make() {
        void* p = nullptr;
        if (hipHostMalloc(&p, SLOT * SLOTS, hipHostMallocDefault) != hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
        ring_ = static_cast<char*>(p);
        for (; n_ev_ < SLOTS; ++n_ev_)
            if (hipEventCreateWithFlags(&ev_[n_ev_], hipEventDisableTiming) != hipSuccess) {
                (void)hipGetLastError();
                return false;
            }
        try {
            threads_.reserve(THREADS);
            for (int t = 0; t < THREADS; ++t) threads_.emplace_back([this] { loop(); });
        } catch (...) {   // fewer threads than asked for; no exception leaves the C interface
        }
        return !threads_.empty();
    }

    void close() {
        {
            std::lock_guard<std::mutex> l(m_);
            stop_ = true;
        }
        work_.notify_all();
        for (std::thread& t : threads_) t.join();
        threads_.clear();
        for (int k = 0; k < n_ev_; ++k) (void)hipEventDestroy(ev_[k]);
        n_ev_ = 0;
        if (ring_) (void)hipHostFree(ring_);
        ring_ = nullptr;
        stop_ = false;
    }

    // What chunk k's slot held before has been copied out (wait: until it has).
    bool emptied(size_t k, bool wait) {
        const int s = (int)(k % SLOTS);
        std::unique_lock<std::mutex> l(m_);
        if (wait) idle_.wait(l, [&] { return !slot_full_[s]; });
        return !slot_full_[s];
    }

    void give(const Job& j) {
        {
            std::lock_guard<std::mutex> l(m_);
            const int s = (int)((j.src - ring_) / SLOT);
            slot_full_[s] = true;
            job_[jobs_ % SLOTS] = j;
            ++jobs_;
        }
        work_.notify_one();
    }

    void loop() {
        std::unique_lock<std::mutex> l(m_);
        for (;;) {
            work_.wait(l, [&] { return stop_ || taken_ < jobs_; });
            if (taken_ == jobs_) return;
            const Job j = job_[taken_++ % SLOTS];
            l.unlock();
            memcpy(j.dst, j.src, j.bytes);
            l.lock();
            slot_full_[(j.src - ring_) / SLOT] = false;
            ++done_;
            idle_.notify_all();
        }
    }
};

}  // namespace mafm
