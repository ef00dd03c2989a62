/*
 * snh_landing.h -- device-to-host copies of a state's fields into the caller's
 * pageable arrays.
 *
 * A plain copy into fresh pageable memory runs at 8-10 GB/s: the runtime moves
 * it through its own staging buffer with one thread, which also takes every
 * page fault of the caller's new array.  Here the DMA engine fills pinned
 * chunks at the link's rate while several threads carry the chunks that have
 * landed into the caller's array, faults included.  The chunks belong to the
 * process (at most LAND_CHUNKS of them, allocated when downloads are large or
 * have repeated, LAND_ALLOC, and given back with the last context); a download
 * that finds too few of them free, or no threads, takes the plain copy.
 */
#ifndef SNH_LANDING_H
#define SNH_LANDING_H

#include <sched.h>

#include <atomic>
#include <condition_variable>
#include <mutex>
#include <thread>
#include <vector>

#define LAND_CHUNK ((size_t)4 << 20)
#define LAND_SLOTS 4      /* chunks of one download */
#define LAND_CHUNKS 8     /* of the process: two downloads at a time */
#define LAND_THREADS 8
/* below this a plain copy is as fast (the threads cost 0.1 ms to start) */
#define LAND_LEAST ((size_t)8 << 20)
/* Allocating the chunks costs 1.5-2 ms, and as much again is lost to the copies
   after they are given back, which a download of less than LAND_ALLOC does not
   earn: the first of a context that is the process's only one took 2.4 ms for
   13 MB and 2.9 ms for 31 MB, against 1.1 and 2.5 with the plain copy (63 MB:
   4.2 against 6.9).  So chunks are allocated for a larger download, or when the
   smaller ones together have come to twice that. */
#define LAND_ALLOC ((size_t)40 << 20)

struct LandPool {
    std::mutex mu;
    void* chunk[LAND_CHUNKS] = {};
    bool used[LAND_CHUNKS] = {};
    int contexts = 0;
    size_t plain = 0;   /* bytes copied plainly for want of chunks */
};
static LandPool g_land;

static void land_context_made() {
    std::lock_guard<std::mutex> l(g_land.mu);
    g_land.contexts++;
}
/* the last context takes the chunks with it */
static void land_context_gone() {
    std::lock_guard<std::mutex> l(g_land.mu);
    if (--g_land.contexts > 0) return;
    g_land.plain = 0;
    for (int k = 0; k < LAND_CHUNKS; k++)
        if (g_land.chunk[k] && !g_land.used[k]) {
            (void)hipHostFree(g_land.chunk[k]);
            g_land.chunk[k] = nullptr;
        }
}

static int land_threads() {
    cpu_set_t set;
    CPU_ZERO(&set);
    int n = LAND_THREADS;
    if (sched_getaffinity(0, sizeof set, &set) == 0 && CPU_COUNT(&set) < n) n = CPU_COUNT(&set);
    return n;
}

/* bytes a to b of the n that go to dst are thread t's of T.  Parts end at page
   boundaries of the destination, so that no two threads fault one page. */
static void land_part(const char* dst, size_t n, size_t T, size_t t, size_t* a, size_t* b) {
    const size_t page = 4096, into = (uintptr_t)dst % page;
    const size_t part = ((n + into + T - 1) / T + page - 1) / page * page;   /* in pages from dst's own */
    const size_t lo = part * t, hi = part * (t + 1);
    *a = t == 0 || lo <= into ? 0 : (lo - into < n ? lo - into : n);
    *b = t + 1 == T || hi - into > n ? n : hi - into;
}

/* One download: push() the fields in stream order, finish() once.  The chunks
   are pinned for every device, since contexts of several may take turns at
   them. */
class Landing {
  public:
    Landing(hipStream_t stream, size_t total) : stream_(stream) {
        if (total >= LAND_LEAST) open(total);
    }
    ~Landing() { close(); }
    Landing(const Landing&) = delete;
    Landing& operator=(const Landing&) = delete;

    /* bytes from device memory src to dst, after what the stream holds; src
       may be overwritten by later work of the same stream */
    hipError_t push(void* dst, const void* src, size_t bytes) {
        pushed_ = true;
        if (!open_) {
            hipError_t r = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, stream_);
            return r != hipSuccess ? r : hipStreamSynchronize(stream_);
        }
        for (size_t at = 0; at < bytes; at += LAND_CHUNK) {
            const size_t n = bytes - at < LAND_CHUNK ? bytes - at : LAND_CHUNK;
            const int s = (int)(posted_ % LAND_SLOTS);
            Job& j = job_[s];
            if (posted_ >= LAND_SLOTS) {   /* the slot's last chunk has been carried off */
                std::unique_lock<std::mutex> l(mu_);
                cv_.wait(l, [&] { return j.left == 0; });
            }
            hipError_t r = hipMemcpyAsync(slot_[s], (const char*)src + at, n, hipMemcpyDeviceToHost, stream_);
            if (r == hipSuccess) r = hipEventRecord(j.landed, stream_);
            if (r != hipSuccess) return r;
            {
                std::lock_guard<std::mutex> l(mu_);
                j.dst = (char*)dst + at;
                j.bytes = n;
                j.left = (int)th_.size();
                posted_++;
            }
            cv_.notify_all();
        }
        return hipSuccess;
    }
    /* every pushed byte is in its place, and the stream's work is done also
       when there was none to push */
    hipError_t finish() {
        close();
        if (!pushed_) return hipStreamSynchronize(stream_);
        return hipError_t(error_.load());
    }

  private:
    struct Job {
        hipEvent_t landed = nullptr;
        char* dst = nullptr;
        size_t bytes = 0;
        int left = 0;      /* threads that still have to carry their part */
    };
    void open(size_t total) {
        {
            std::lock_guard<std::mutex> l(g_land.mu);
            int have = 0;
            for (int k = 0; k < LAND_CHUNKS; k++) have += g_land.chunk[k] && !g_land.used[k];
            if (have < LAND_SLOTS && total < LAND_ALLOC && (g_land.plain += total) < 2 * LAND_ALLOC) return;
            int n = 0;
            for (int k = 0; k < LAND_CHUNKS && n < LAND_SLOTS; k++) {
                if (g_land.used[k]) continue;
                if (!g_land.chunk[k] && hipHostMalloc(&g_land.chunk[k], LAND_CHUNK, hipHostMallocPortable) != hipSuccess) {
                    g_land.chunk[k] = nullptr;
                    (void)hipGetLastError();
                    break;
                }
                g_land.used[k] = true;
                slot_[n] = g_land.chunk[k];
                index_[n++] = k;
            }
            slots_ = n;
        }
        bool ok = slots_ == LAND_SLOTS;
        for (int s = 0; s < LAND_SLOTS && ok; s++)
            if (hipEventCreateWithFlags(&job_[s].landed, hipEventDisableTiming) != hipSuccess) {
                job_[s].landed = nullptr;
                (void)hipGetLastError();   /* not the next launch's error */
                ok = false;
            }
        if (ok) {
            const int T = land_threads();
            try {
                th_.reserve(T);
                std::lock_guard<std::mutex> l(mu_);   /* none starts before the number of them is known */
                for (int t = 0; t < T; t++) th_.emplace_back([this, t] { carry(t); });
            } catch (...) {
                /* as many as there are; they share the chunks all the same */
            }
            ok = !th_.empty();
        }
        open_ = ok;
    }
    void carry(int t) {
        size_t T;
        {
            std::lock_guard<std::mutex> l(mu_);
            T = th_.size();
        }
        for (size_t i = 0;; i++) {
            Job& j = job_[i % LAND_SLOTS];
            {
                std::unique_lock<std::mutex> l(mu_);
                cv_.wait(l, [&] { return posted_ > i || done_; });
                if (posted_ <= i) return;
            }
            const hipError_t r = hipEventSynchronize(j.landed);
            if (r != hipSuccess) error_ = (int)r;
            size_t a, b;
            land_part(j.dst, j.bytes, T, (size_t)t, &a, &b);
            if (r == hipSuccess && b > a) memcpy(j.dst + a, (char*)slot_[i % LAND_SLOTS] + a, b - a);
            bool last;
            {
                std::lock_guard<std::mutex> l(mu_);
                last = --j.left == 0;
            }
            if (last) cv_.notify_all();
        }
    }
    void close() {
        if (closed_) return;
        closed_ = true;
        {
            std::lock_guard<std::mutex> l(mu_);
            done_ = true;
        }
        cv_.notify_all();
        for (std::thread& t : th_) t.join();
        th_.clear();
        for (Job& j : job_)
            if (j.landed) (void)hipEventDestroy(j.landed);
        std::lock_guard<std::mutex> l(g_land.mu);
        for (int s = 0; s < slots_; s++) g_land.used[index_[s]] = false;
    }

    hipStream_t stream_;
    bool open_ = false, pushed_ = false, closed_ = false, done_ = false;
    int slots_ = 0, index_[LAND_SLOTS] = {};
    void* slot_[LAND_SLOTS] = {};
    Job job_[LAND_SLOTS];
    size_t posted_ = 0;
    std::atomic<int> error_{0};
    std::mutex mu_;
    std::condition_variable cv_;
    std::vector<std::thread> th_;
};

#endif
