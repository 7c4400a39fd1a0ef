// Host-side helpers shared by the converters and the plan builder: a loop over
// [0, n) cut into chunks that worker threads take one after the other.
#pragma once
#include <pthread.h>
#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstddef>
#include <cstdlib>
#include <new>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace hspmm_host {

inline unsigned worker_count(size_t work_items, size_t min_per_worker)
{
    unsigned hw = std::thread::hardware_concurrency();
    if (hw == 0) hw = 1;
    if (hw > 16) hw = 16;
    size_t by_work = work_items / (min_per_worker ? min_per_worker : 1);
    if (by_work < 1) by_work = 1;
    return unsigned(std::min<size_t>(hw, by_work));
}

// The threads behind the loops below.  Starting and joining fifteen threads takes 0.35 ms where waking fifteen that wait
// takes 0.04, and a conversion with its plan runs seven such loops.  At most 15 threads per process, shared by all callers;
// a thread ends when it has had nothing to do for a second.  The caller of run() is a worker itself and needs none of them
// to get its work done, so callers on several threads and calls inside calls cannot wait for one another.
class WorkerPool {
public:
    static WorkerPool &get()
    {
        // (never destroyed: a waiting thread may outlive the static objects of the process)
        static WorkerPool *pool = make();
        return *pool;
    }
    // work(ctx, i) on the calling thread (i = 0) and on up to n - 1 others; returns when all that began have ended.
    void run(unsigned n, void (*work)(void *, unsigned), void *ctx)
    {
        Job job{work, ctx, n - 1u, 0u, 0u, nullptr};
        State &s = *state_;
        {
            std::lock_guard<std::mutex> lk(s.mutex);
            job.next = s.jobs;
            s.jobs = &job;
            try {
                for (; s.threads - s.busy < job.wanted && s.threads < kMost; ++s.threads) std::thread(serve, &s).detach();
            } catch (...) {}                              // (no more threads: those there are share the work)
        }
        s.work.notify_all();
        work(ctx, 0u);
        std::unique_lock<std::mutex> lk(s.mutex);
        for (Job **at = &s.jobs; *at; at = &(*at)->next)
            if (*at == &job) { *at = job.next; break; }
        s.done.wait(lk, [&] { return job.running == 0u; });
    }

private:
    static constexpr unsigned kMost = 15;
    struct Job {
        void (*work)(void *, unsigned);
        void *ctx;
        unsigned wanted, joined, running;                 // helpers asked for, that came, that have not ended
        Job *next;
    };
    struct State {
        std::mutex mutex;
        std::condition_variable work, done;
        Job *jobs = nullptr;
        unsigned threads = 0, busy = 0;
    };
    State *state_ = new State;

    static WorkerPool *make()
    {
        WorkerPool *pool = new WorkerPool;
        // a forked child has none of the threads, and what they held stays locked: it starts anew
        pthread_atfork(nullptr, nullptr, [] { get().state_ = new State; });
        return pool;
    }
    static void serve(State *s)
    {
        std::unique_lock<std::mutex> lk(s->mutex);
        for (;;) {
            Job *job = s->jobs;
            while (job && job->joined == job->wanted) job = job->next;
            if (job) {
                const unsigned i = ++job->joined;
                ++job->running;
                ++s->busy;
                lk.unlock();
                job->work(job->ctx, i);
                lk.lock();
                --s->busy;
                if (--job->running == 0u) s->done.notify_all();
            } else if (s->work.wait_for(lk, std::chrono::seconds(1)) == std::cv_status::timeout) {
                for (job = s->jobs; job && job->joined == job->wanted; job = job->next) {}
                if (!job) { --s->threads; return; }
            }
        }
    }
};

// fn(i) for i = 0 .. n - 1, each on a thread of its own where there are enough; an exception of one of them (out of memory) is
// rethrown on the calling thread once all are done.
template <class F>
void parallel_workers(unsigned n, F &&fn)
{
    if (n <= 1u) { fn(0u); return; }
    std::mutex mutex;
    std::exception_ptr error;
    auto work = [&](unsigned i) {
        try { fn(i); }
        catch (...) { std::lock_guard<std::mutex> lk(mutex); if (!error) error = std::current_exception(); }
    };
    WorkerPool::get().run(n, [](void *ctx, unsigned i) { (*static_cast<decltype(work) *>(ctx))(i); }, &work);
    if (error) std::rethrow_exception(error);
}

// fn(begin, end) on chunks of `chunk` items that the workers take off a shared counter until none is left.
template <class F>
void parallel_chunks(size_t n, size_t chunk, F &&fn, unsigned workers = 0)
{
    if (chunk < 1) chunk = 1;
    const unsigned nw = workers ? workers : worker_count(n, chunk);
    if (nw <= 1) { if (n) fn(size_t(0), n); return; }
    std::atomic<size_t> next{0};
    parallel_workers(nw, [&](unsigned) {
        try {
            for (size_t b = next.fetch_add(chunk); b < n; b = next.fetch_add(chunk)) fn(b, std::min(n, b + chunk));
        } catch (...) {
            next.store(n);                            // the others stop at their next chunk
            throw;
        }
    });
}

// The same with chunks of about equal weight, cut where `before` - the weight of the items in front of item i, for i = 0 .. n -
// says: the windows of a power-law graph, whose first hundredth holds a tenth of all entries and would keep one worker
// busy long after the others have ended.  Items without weight cost something too: an item weighs one more than it says.
template <class W, class F>
void parallel_weighted(size_t n, size_t min_per_worker, W &&before, F &&fn)
{
    auto weight = [&](size_t i) { return size_t(before(i)) + i; };
    const size_t total = n ? weight(n) : 0u;
    const unsigned nw = worker_count(total, min_per_worker);
    if (nw <= 1) { if (n) fn(size_t(0), n); return; }
    const size_t pieces = size_t(nw) * 8u;
    auto cut = [&](size_t piece) {                    // the first item with that much in front of it
        const size_t want = total / pieces * piece + total % pieces * piece / pieces;
        size_t lo = 0, hi = n;
        while (lo < hi) {
            const size_t mid = lo + (hi - lo) / 2;
            if (weight(mid) < want) lo = mid + 1; else hi = mid;
        }
        return lo;
    };
    // (pieces taken one after the other lie an eighth of a worker's share apart: side by side, the workers would wait for
    // one another wherever a fresh page of the output - 2 MB - has to be cleared first)
    parallel_chunks(pieces, 1, [&](size_t taken, size_t end) {
        for (; taken < end; ++taken) {
            const size_t piece = taken % nw * 8u + taken / nw, b = cut(piece), e = cut(piece + 1u);
            if (b < e) fn(b, e);
        }
    }, nw);
}

// A loop over [0, n) for as many workers as have min_per_worker items each: eight chunks per worker, none
// shorter than min_per_worker.
template <class F>
void parallel_blocks(size_t n, size_t min_per_worker, F &&fn)
{
    const unsigned nw = worker_count(n, min_per_worker);
    if (nw <= 1) { fn(size_t(0), n); return; }
    const size_t pieces = size_t(nw) * 8u;
    parallel_chunks(n, std::max<size_t>(min_per_worker, (n + pieces - 1) / pieces), fn, nw);
}

// n elements that read as zero, without the single-threaded pass a std::vector spends on clearing them
// (a fifth of a second for the arrays of a large plan): the memory comes from calloc, whose fresh pages are
// zero already, and is first touched by whichever worker fills it.  Trivial element types only.
template <class T>
class ZeroedBuffer {
    T *p_ = nullptr;
    size_t n_ = 0;
public:
    ZeroedBuffer() = default;
    explicit ZeroedBuffer(size_t n) : p_(static_cast<T *>(std::calloc(n ? n : 1, sizeof(T)))), n_(n)
    {
        if (!p_) throw std::bad_alloc();
    }
    ZeroedBuffer(const ZeroedBuffer &) = delete;
    ZeroedBuffer &operator=(const ZeroedBuffer &) = delete;
    ZeroedBuffer(ZeroedBuffer &&o) noexcept : p_(o.p_), n_(o.n_) { o.p_ = nullptr; o.n_ = 0; }
    ZeroedBuffer &operator=(ZeroedBuffer &&o) noexcept
    {
        if (this != &o) { std::free(p_); p_ = o.p_; n_ = o.n_; o.p_ = nullptr; o.n_ = 0; }
        return *this;
    }
    ~ZeroedBuffer() { std::free(p_); }
    T *data() { return p_; }
    const T *data() const { return p_; }
    size_t size() const { return n_; }
    T &operator[](size_t i) { return p_[i]; }
    const T &operator[](size_t i) const { return p_[i]; }
    void swap(ZeroedBuffer &o) noexcept { std::swap(p_, o.p_); std::swap(n_, o.n_); }
};

}  // namespace hspmm_host
