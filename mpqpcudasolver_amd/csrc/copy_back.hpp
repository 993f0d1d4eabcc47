// copy_back.hpp — copies between device memory and the caller's arrays
// through pinned blocks.  Host code only; included by mpqp_hip.hip.
#pragma once
#include <hip/hip_runtime.h>
#include <pthread.h>
#include <signal.h>
#include <sys/mman.h>
#include <unistd.h>

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <memory>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#ifndef MADV_POPULATE_WRITE
#define MADV_POPULATE_WRITE 23
#endif

namespace {

struct HipError {
    std::string msg;
};

#define HIP_OK(expr)                                                                   \
    do {                                                                               \
        hipError_t e_ = (expr);                                                        \
        if (e_ != hipSuccess)                                                          \
            throw HipError{std::string(#expr) + ": " + hipGetErrorString(e_)};         \
    } while (0)

// Pinned host memory for copies to and from the caller's arrays: SLOTS blocks
// with an event each, 32 MiB in all, made by warm_up() and kept.  Making a
// block inside a call, and then the first access to each of its pages from
// the host (a page fault, 1.3 ms a block), cost the first mpqp_regions() call
// of a process 4 to 10 ms.
struct Staging {
    static constexpr size_t SLOT = (size_t)4 << 20;
    static constexpr int SLOTS = 8;
    unsigned char *p[SLOTS] = {};
    hipEvent_t ev[SLOTS] = {};
    bool ok = false;  // false: not to be had, copies go directly

    void make() {
        if (ok) return;
        unsigned char *all = nullptr;
        if (hipHostMalloc(reinterpret_cast<void **>(&all), SLOT * SLOTS) != hipSuccess) {
            (void)hipGetLastError();
            return;
        }
        int n = 0;
        while (n < SLOTS && hipEventCreateWithFlags(&ev[n], hipEventDisableTiming) == hipSuccess) ++n;
        if (n < SLOTS) {
            (void)hipGetLastError();
            while (n > 0) (void)hipEventDestroy(ev[--n]);
            (void)hipHostFree(all);
            return;
        }
        const size_t page = (size_t)sysconf(_SC_PAGESIZE);
        volatile unsigned char sink = 0;
        for (size_t i = 0; i < SLOT * SLOTS; i += page) sink = all[i];
        (void)sink;
        for (int i = 0; i < SLOTS; ++i) p[i] = all + i * SLOT;
        ok = true;
    }
};

class CopyBack;

// Threads that help CopyBack, parked between calls and joined with the
// context (at the process's end or dlclose()).
class CopyThreads {
  public:
    ~CopyThreads() {
        // (the child of a fork() has the objects without the threads: there
        // they are left as they are, a join or the destruction of the
        // condition variable would wait for ever)
        if (!k || getpid() != k->owner) return;
        {
            std::lock_guard<std::mutex> lk(k->m);
            k->quit = true;
            k->cv.notify_all();
        }
        for (std::thread &t : k->th) t.join();
        delete k;
    }
    // up to n threads (fewer if they are not to be had)
    void make(size_t n) {
        // signals are for the program's own threads
        sigset_t all, old;
        sigfillset(&all);
        pthread_sigmask(SIG_SETMASK, &all, &old);
        try {
            if (!k) k = new Kept;
            while (k->th.size() < n) k->th.emplace_back([kk = k] { kk->run(); });
        } catch (const std::exception &) {
        }
        pthread_sigmask(SIG_SETMASK, &old, nullptr);
    }
    void post(std::shared_ptr<CopyBack> c) {
        if (!k) return;
        std::lock_guard<std::mutex> lk(k->m);
        k->job = std::move(c);
        ++k->posted;
        k->cv.notify_all();
    }
    void drop() {
        if (!k) return;
        std::lock_guard<std::mutex> lk(k->m);
        k->job.reset();
    }

  private:
    struct Kept {
        std::mutex m;
        std::condition_variable cv;
        std::vector<std::thread> th;
        std::shared_ptr<CopyBack> job;
        long long posted = 0;
        bool quit = false;
        const pid_t owner = getpid();
        void run();
    };
    Kept *k = nullptr;
};

// Copies from device memory into the caller's arrays through the staging
// blocks.  A direct copy into pageable memory moves 16 GB/s into pages in use
// and far less into new ones, which it faults in one by one.  Here the device
// writes pinned blocks (54 GB/s) and the caller's thread empties them; from
// two blocks' bytes on, the parked threads help, first by making the arrays'
// pages present while the kernel still runs, then by copying pieces.
//
// A thread that loses its CPU in mid-piece holds up the call, by a scheduler's
// slice and more where the program's other threads keep the CPUs busy (those
// of a BLAS spin for tens of milliseconds after a product).  So the threads
// stop before the last half of the bytes, or the last ALONE of more: the
// caller copies those meanwhile, and waits only for a thread that is inside a
// piece or a range even then.  A thread that comes later finds the call ended
// and touches nothing.  n=60 m=120 p=12 (27.6 KB a set), ms a call on the same
// data / on each of several new problems:
//   3,000 sets, the threads stop at 50% 4.1 / 4.0 to 5.5, at 70% 3.9 / 3.9 to
//   12, never 3.5 / 3.6 to 13, at once 4.7 / 4.6 to 7.6; direct copies 9.8 /
//   10.4; pieces of 4 MiB instead of 1 at 70% the same / up to 12;
//   110,415 sets, at 50% 178 / 205, 64 MiB before the end 118 / 147; direct
//   337 / 334.
class CopyBack : public std::enable_shared_from_this<CopyBack> {
  public:
    struct Seg {
        size_t off, bytes;  // in the device buffer
        void *dst;
    };
    // total: bytes of all the copies to come
    CopyBack(Staging &s, CopyThreads &t, hipStream_t stream, size_t total)
        : S(s), T(t), st(stream), help_from(total >= 2 * Staging::SLOT), limit(total - std::min(total / 2, ALONE)) {}
    // segs (ascending) of the buffer at dev, read in stream order
    void copy(const unsigned char *dev, const std::vector<Seg> &segs) {
        if (!S.ok) {
            for (const Seg &s : segs) HIP_OK(hipMemcpyAsync(s.dst, dev + s.off, s.bytes, hipMemcpyDeviceToHost, st));
            return;
        }
        if (help_from) call_threads(segs);
        size_t i = 0;
        while (i < segs.size()) {
            // a run of adjacent segments
            size_t j = i, end = segs[i].off + segs[i].bytes;
            while (j + 1 < segs.size() && segs[j + 1].off == end) end += segs[++j].bytes;
            for (size_t a = segs[i].off; a < end; a += Staging::SLOT)
                issue(dev, a, std::min(Staging::SLOT, end - a), segs, i, j);
            i = j + 1;
        }
    }
    // every copy is in its array
    void finish() {
        if (!S.ok) {
            HIP_OK(hipStreamSynchronize(st));
            return;
        }
        {
            std::unique_lock<std::mutex> lk(m);
            while (step(lk)) {}
            cv.wait(lk, [this] { return drained == issued; });
        }
        stop();
        if (err != hipSuccess) throw HipError{std::string("copy to the host failed: ") + hipGetErrorString(err)};
    }
    // nothing is handed out any more, and no thread is at the arrays
    void stop() {
        {
            std::unique_lock<std::mutex> lk(m);
            ended = true;
            cv.notify_all();
            cv.wait(lk, [this] { return out == 0; });
        }
        if (posted) T.drop();
        posted = false;
    }
    // a thread's part in the call
    void help() {
        std::unique_lock<std::mutex> lk(m);
        for (;;) {
            cv.wait(lk, [this] { return ended || given >= limit || next_range < ranges.size() || taken < ready; });
            if (ended || given >= limit) return;
            if (next_range < ranges.size()) {
                const Range r = ranges[next_range++];
                ++out;
                lk.unlock();
                // (it fails on memory of other kinds, and on kernels before 5.14: the copies fault then)
                (void)madvise(r.p, r.bytes, MADV_POPULATE_WRITE);
                lk.lock();
                --out;
                if (ended) cv.notify_all();
            } else {
                one_piece(lk);
            }
        }
    }

  private:
    static constexpr size_t PIECE = (size_t)1 << 20, RANGE = (size_t)2 << 20;  // RANGE: a huge page
    static constexpr size_t ALONE = (size_t)64 << 20;
    struct Part {
        size_t src, bytes;
        unsigned char *dst;
    };
    struct Range {
        void *p;
        size_t bytes;
    };
    struct Block {
        std::vector<Part> parts;
        size_t next = 0, at = 0;  // first part not handed out, its bytes that are
        size_t left = 0;          // bytes not in their array yet
    };
    Staging &S;
    CopyThreads &T;
    hipStream_t st;
    const bool help_from;
    const size_t limit;
    std::mutex m;
    std::condition_variable cv;
    Block blk[Staging::SLOTS];
    std::vector<Range> ranges;
    size_t next_range = 0, given = 0;
    // blocks: copies queued, arrived, wholly handed out, wholly emptied
    long long issued = 0, ready = 0, taken = 0, drained = 0;
    int out = 0;  // pieces and ranges in work
    bool ended = false, posted = false;
    hipError_t err = hipSuccess;

    void call_threads(const std::vector<Seg> &segs) {
        const size_t page = (size_t)sysconf(_SC_PAGESIZE);
        {
            std::lock_guard<std::mutex> lk(m);
            for (const Seg &s : segs) {
                // whole pages of the array, cut at huge pages
                const size_t d = reinterpret_cast<size_t>(s.dst);
                size_t lo = (d + page - 1) / page * page;
                const size_t hi = (d + s.bytes) / page * page;
                while (lo < hi) {
                    const size_t e = std::min(hi, lo / RANGE * RANGE + RANGE);
                    ranges.push_back({reinterpret_cast<void *>(lo), e - lo});
                    lo = e;
                }
            }
            cv.notify_all();
        }
        if (!posted) {
            posted = true;
            T.post(shared_from_this());
        }
    }
    void issue(const unsigned char *dev, size_t a, size_t bytes, const std::vector<Seg> &segs, size_t i, size_t j) {
        const int b = (int)(issued % Staging::SLOTS);
        {
            std::unique_lock<std::mutex> lk(m);
            while (blk[b].left)
                if (!step(lk)) cv.wait(lk, [&] { return blk[b].left == 0; });
        }
        std::vector<Part> ps;
        for (size_t k = i; k <= j; ++k) {
            const size_t lo = std::max(a, segs[k].off), hi = std::min(a + bytes, segs[k].off + segs[k].bytes);
            if (lo < hi)
                ps.push_back(Part{lo - a, hi - lo, static_cast<unsigned char *>(segs[k].dst) + (lo - segs[k].off)});
        }
        HIP_OK(hipMemcpyAsync(S.p[b], dev + a, bytes, hipMemcpyDeviceToHost, st));
        HIP_OK(hipEventRecord(S.ev[b], st));
        std::lock_guard<std::mutex> lk(m);
        blk[b].parts.swap(ps);
        blk[b].next = blk[b].at = 0;
        blk[b].left = bytes;
        ++issued;
    }
    // The caller's thread, which alone calls HIP: notes a block that has
    // arrived, else copies a piece, else waits for the next block.  False:
    // nothing is left to do but to wait for the other threads.
    bool step(std::unique_lock<std::mutex> &lk) {
        if (ready < issued && arrive(lk, false)) return true;
        if (taken < ready) {
            one_piece(lk);
            return true;
        }
        return ready < issued && arrive(lk, true);
    }
    bool arrive(std::unique_lock<std::mutex> &lk, bool wait) {
        hipEvent_t e = S.ev[ready % Staging::SLOTS];
        lk.unlock();
        const hipError_t r = wait ? hipEventSynchronize(e) : hipEventQuery(e);
        if (r == hipErrorNotReady) (void)hipGetLastError();
        lk.lock();
        if (r == hipErrorNotReady) return false;
        if (r != hipSuccess) err = r;
        ++ready;
        cv.notify_all();
        return true;
    }
    // Copies the next piece of the oldest block that has arrived.
    void one_piece(std::unique_lock<std::mutex> &lk) {
        const int b = (int)(taken % Staging::SLOTS);
        Block &k = blk[b];
        const Part q = k.parts[k.next];
        const size_t at = k.at, n = std::min(PIECE, q.bytes - at);
        k.at += n;
        if (k.at == q.bytes) {
            k.at = 0;
            if (++k.next == k.parts.size()) ++taken;
        }
        given += n;
        ++out;
        const bool good = err == hipSuccess;
        lk.unlock();
        if (good) std::memcpy(q.dst + at, S.p[b] + q.src + at, n);
        lk.lock();
        --out;
        k.left -= n;
        if (k.left == 0) ++drained;
        if (k.left == 0 || ended) cv.notify_all();
    }
};

void CopyThreads::Kept::run() {
    long long seen = 0;
    std::unique_lock<std::mutex> lk(m);
    for (;;) {
        cv.wait(lk, [&] { return quit || posted != seen; });
        if (quit) return;
        seen = posted;
        const std::shared_ptr<CopyBack> c = job;
        lk.unlock();
        if (c) c->help();
        lk.lock();
    }
}

}  // namespace
