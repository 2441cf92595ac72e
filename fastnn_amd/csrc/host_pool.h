// Worker threads of the library's host side (weight packers, staging copies): started on first use, kept, shared by
// every caller of the process.
#pragma once
#include <cstdint>

#include <atomic>

// CPUs this process may run on, at most 16
int fnn_host_threads();

// Tasks 0 .. tasks-1 handed to the workers between begin() and end(); the caller takes tasks too with run_one() (false:
// none left to take) and must call end(), which runs what is left and waits for tasks still running elsewhere.  Jobs of
// several threads share the workers; in a forked child (whose workers are gone) the caller runs every task itself.
// `fn` must not throw.
struct FnnJob {
    void (*fn)(void *, int64_t);
    void *arg;
    int64_t tasks;
    std::atomic<int64_t> next{0};
    int helpers = 0, helpers_max = 0;   // workers inside the job, under the pool's mutex
    bool queued = false;
    FnnJob(int64_t n, void (*f)(void *, int64_t), void *a) : fn(f), arg(a), tasks(n) {}
    void begin(int threads);
    bool run_one()
    {
        const int64_t i = next.fetch_add(1, std::memory_order_relaxed);
        if (i >= tasks) return false;
        fn(arg, i);
        return true;
    }
    void end();
};

// f(i) for every i in [0, tasks) on up to `threads` threads, the caller among them; returns when all are done.
template <class F>
void fnn_parallel(int64_t tasks, int threads, F &&f)
{
    FnnJob job(tasks, [](void *arg, int64_t i) { (*static_cast<F *>(arg))(i); }, (void *)&f);
    job.begin(threads);
    job.end();
}
