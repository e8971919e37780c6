// ttsh_hostcopy.h -- device arrays to pageable host memory.
//
// A plain hipMemcpy to pageable memory stages through the runtime's own pinned
// buffer with one thread, which also takes the page faults of a destination
// that was just allocated: 8 to 11 GB/s, of the 50 to 56 GB/s that copies to
// pinned memory reach.  HostCopier keeps a ring of pinned chunks: the calling
// thread queues the copies and hands each finished chunk to worker threads,
// which store it (widened to FP64 if asked) in the destination.  Four workers
// take 56 GB/s with the page faults, one 16.  State of a 256^3 droplet (470
// MB) 58 -> 11 ms, 128^3 (59 MB) 7.2 -> 1.7 ms.  A destination that is pinned
// already has nothing to gain: 128^3 takes 1.1 ms by hipMemcpy, 1.5 through
// the ring.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace ttsh {

struct HostPiece {
    const float* src;  // device, n floats
    void* dst;         // host, n floats or doubles
    size_t n;
};

// A ring of pinned chunks.
struct Ring {
    float* p = nullptr;  // nullptr: no pinned memory to be had
    size_t n = 0;        // floats
};

// Rings shared by the copiers of a process: at most kIdle are kept while no copy
// uses them, the larger ones, and none once the last copier is gone.
class PinnedRings {
public:
    static PinnedRings& get()
    {
        static PinnedRings* const r = new PinnedRings();  // never destroyed: copiers may outlive main
        return *r;
    }
    void join()
    {
        std::lock_guard<std::mutex> lk(mu);
        ++copiers;
    }
    void leave()
    {
        std::lock_guard<std::mutex> lk(mu);
        if (--copiers > 0) return;
        for (const Ring& r : idle) (void)hipHostFree(r.p);
        idle.clear();
    }
    // A ring of at least n floats.
    Ring borrow(size_t n)
    {
        {
            std::lock_guard<std::mutex> lk(mu);
            for (size_t k = 0; k < idle.size(); ++k)
                if (idle[k].n >= n) {
                    const Ring r = idle[k];
                    idle.erase(idle.begin() + (long)k);
                    return r;
                }
        }
        void* p = nullptr;
        if (hipHostMalloc(&p, sizeof(float) * n, hipHostMallocPortable) != hipSuccess) {
            (void)hipGetLastError();
            return Ring{};
        }
        return Ring{static_cast<float*>(p), n};
    }
    void give(Ring r)
    {
        {
            std::lock_guard<std::mutex> lk(mu);
            if (idle.size() < kIdle) {
                idle.push_back(r);
                return;
            }
            for (Ring& k : idle)
                if (k.n < r.n) std::swap(k, r);
        }
        (void)hipHostFree(r.p);
    }

private:
    static constexpr size_t kIdle = 2;
    PinnedRings() { idle.reserve(kIdle); }
    std::mutex mu;
    std::vector<Ring> idle;
    int copiers = 0;
};

class HostCopier {
public:
    // Below this the threads cost more than they save.
    static constexpr size_t kMinBytes = (size_t)8 << 20;
    // States below kLargeBytes use chunks of 2 MiB, larger ones of 4 MiB.  The
    // first copy through a ring takes the page faults of its host mapping, about
    // 0.13 ms per MiB: a first read of a 96^3 state (25 MB) takes 3.0 ms, with
    // chunks of 4 MiB 4.7, with one plain copy 2.5.  Later reads take 0.79 ms
    // against 0.75 (in FP64 0.89 and 1.0).  At 128^3 (59 MB) they would take 1.62
    // against 1.47, and a plain copy takes as long as the larger ring's first.
    static constexpr size_t kLargeBytes = (size_t)32 << 20;

    HostCopier() { PinnedRings::get().join(); }
    HostCopier(const HostCopier&) = delete;
    HostCopier& operator=(const HostCopier&) = delete;
    ~HostCopier()
    {
        release();
        PinnedRings::get().leave();
    }

    // Destroys the events (the device's streams are done).
    void release()
    {
        for (auto& e : ev) {
            if (e) (void)hipEventDestroy(e);
            e = nullptr;
        }
    }

    // Takes the pieces that go through the ring out of the list, copies them on
    // stream st and returns when they are in place.  What stays is the caller's
    // to copy: FP32 for destinations that are not pageable, less than kMinBytes
    // altogether, or all if threads or pinned memory were not to be had.
    hipError_t copy(std::vector<HostPiece>& pieces, bool f64, hipStream_t st)
    {
        const auto bytes_from = [&](std::vector<HostPiece>::iterator p) {
            size_t b = 0;
            for (; p != pieces.end(); ++p) b += p->n * sizeof(float);
            return b;
        };
        // before the look at each pointer, which small copies need not pay
        if (bytes_from(pieces.begin()) < kMinBytes) return hipSuccess;
        const auto mine = std::stable_partition(pieces.begin(), pieces.end(),
                                                [&](const HostPiece& p) { return !f64 && !pageable(p.dst); });
        const size_t bytes = bytes_from(mine);
        if (bytes < kMinBytes || !events()) return hipSuccess;
        chunk_n = bytes < kLargeBytes ? kChunk / 2 : kChunk;
        struct Loan {
            Ring r;
            ~Loan()
            {
                if (r.p) PinnedRings::get().give(r);
            }
        } loan{PinnedRings::get().borrow(chunk_n * kSlots)};  // outlives the workers and every copy into it
        ring = loan.r.p;
        if (!ring) return hipSuccess;
        std::vector<HostPiece> chunk;
        for (auto p = mine; p != pieces.end(); ++p)
            for (size_t o = 0; o < p->n; o += chunk_n) {
                const size_t n = std::min(chunk_n, p->n - o);
                chunk.push_back(HostPiece{p->src + o, static_cast<char*>(p->dst) + o * (f64 ? 8 : 4), n});
            }
        head = tail = 0;
        for (bool& b : busy) b = false;
        quit = false;
        std::vector<std::thread> th;
        th.reserve(kWorkers);
        try {
            for (int k = 0; k < kWorkers; ++k) th.emplace_back([this, f64] { work(f64); });
        } catch (...) {
            if (th.empty()) return hipSuccess;  // with fewer workers it goes on
        }
        pieces.erase(mine, pieces.end());
        hipError_t e = hipSuccess;
        size_t issued = 0;
        for (size_t i = 0; i < chunk.size() && e == hipSuccess; ++i) {
            // keep every free slot's copy in flight; chunk i's slot frees up
            // when the workers have stored chunk i - kSlots
            while (issued < chunk.size() && issued < i + kSlots && e == hipSuccess) {
                const int s = (int)(issued % kSlots);
                {
                    std::unique_lock<std::mutex> lk(mu);
                    if (busy[s]) {
                        if (issued > i) break;
                        free_cv.wait(lk, [&] { return !busy[s]; });
                    }
                    busy[s] = true;
                }
                e = hipMemcpyAsync(slot(s), chunk[issued].src, chunk[issued].n * sizeof(float), hipMemcpyDeviceToHost, st);
                if (e == hipSuccess) e = hipEventRecord(ev[s], st);
                ++issued;
            }
            if (e != hipSuccess) break;
            const int s = (int)(i % kSlots);
            e = hipEventSynchronize(ev[s]);
            if (e != hipSuccess) break;
            {
                std::lock_guard<std::mutex> lk(mu);
                ready[tail++ % kSlots] = Job{s, chunk[i].dst, chunk[i].n};
            }
            ready_cv.notify_one();
        }
        {
            std::lock_guard<std::mutex> lk(mu);
            quit = true;
        }
        ready_cv.notify_all();
        for (auto& t : th) t.join();
        if (e != hipSuccess) (void)hipStreamSynchronize(st);  // no copy into the ring stays in flight
        return e;
    }

private:
    static constexpr size_t kChunk = (size_t)1 << 20;  // floats: 4 MiB
    static constexpr int kSlots = 8, kWorkers = 4;
    struct Job {
        int slot;
        void* dst;
        size_t n;
    };

    static bool pageable(const void* p)
    {
        hipPointerAttribute_t at{};
        if (hipPointerGetAttributes(&at, p) == hipSuccess) return at.type == hipMemoryTypeUnregistered;
        (void)hipGetLastError();  // memory that the runtime does not know
        return true;
    }

    float* slot(int s) const { return ring + (size_t)s * chunk_n; }

    bool events()
    {
        for (auto& e : ev)
            if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
                e = nullptr;
                (void)hipGetLastError();
                return false;
            }
        return true;
    }

    void work(bool f64)
    {
        for (;;) {
            Job j;
            {
                std::unique_lock<std::mutex> lk(mu);
                ready_cv.wait(lk, [&] { return quit || head != tail; });
                if (head == tail) return;
                j = ready[head++ % kSlots];
            }
            const float* s = slot(j.slot);
            if (f64) {
                double* d = static_cast<double*>(j.dst);
                for (size_t i = 0; i < j.n; ++i) d[i] = s[i];
            } else {
                std::memcpy(j.dst, s, j.n * sizeof(float));
            }
            {
                std::lock_guard<std::mutex> lk(mu);
                busy[j.slot] = false;
            }
            free_cv.notify_one();
        }
    }

    float* ring = nullptr;
    size_t chunk_n = kChunk;  // of the copy under way
    hipEvent_t ev[kSlots] = {};
    std::mutex mu;
    std::condition_variable ready_cv, free_cv;
    Job ready[kSlots] = {};  // a queue: each slot holds at most one chunk
    size_t head = 0, tail = 0;
    bool busy[kSlots] = {};
    bool quit = false;
};

}  // namespace ttsh
