#include "host_pool.h"

#include <atomic>
#include <condition_variable>
#include <list>
#include <mutex>
#include <thread>

#include <pthread.h>
#include <sched.h>

namespace {

struct Job {
    void (*fn)(void *, int64_t);
    void *arg;
    int64_t tasks;
    std::atomic<int64_t> next{0};
    int helpers = 0;       // workers inside run(), under Pool::mu
    int helpers_max = 0;
    void run()
    {
        for (int64_t i; (i = next.fetch_add(1, std::memory_order_relaxed)) < tasks;) fn(arg, i);
    }
};

struct Pool {
    std::mutex mu;
    std::condition_variable work, left;
    std::list<Job *> jobs;
    int workers = 0;

    void serve()
    {
        std::unique_lock<std::mutex> lock(mu);
        for (;;) {
            Job *job = nullptr;
            for (Job *j : jobs)
                if (j->helpers < j->helpers_max && j->next.load(std::memory_order_relaxed) < j->tasks) { job = j; break; }
            if (!job) { work.wait(lock); continue; }
            job->helpers++;
            lock.unlock();
            job->run();
            lock.lock();
            if (--job->helpers == 0) left.notify_all();
        }
    }
};

// Never destroyed: detached workers may still wait in it while the process ends.
Pool *g_pool = new Pool();

// A forked child has no workers and may find the mutex held by one that is gone: it starts a pool of its own.
const int g_at_fork = pthread_atfork(nullptr, nullptr, [] { g_pool = new Pool(); });

}  // namespace

int fnn_host_threads()
{
    static const int n = [] {
        cpu_set_t set;
        int c = sched_getaffinity(0, sizeof set, &set) == 0 ? CPU_COUNT(&set) : (int)std::thread::hardware_concurrency();
        return c < 1 ? 1 : (c > 16 ? 16 : c);
    }();
    return n;
}

void fnn_parallel_raw(int64_t tasks, int threads, void (*fn)(void *, int64_t), void *arg)
{
    Pool &p = *g_pool;
    Job job;
    job.fn = fn; job.arg = arg; job.tasks = tasks;
    const int64_t want = tasks - 1;
    int helpers = threads - 1 < want ? threads - 1 : (int)want;
    if (helpers <= 0) { job.run(); return; }
    job.helpers_max = helpers;
    std::list<Job *>::iterator at;
    {
        std::lock_guard<std::mutex> lock(p.mu);
        const int most = fnn_host_threads() - 1;
        try {
            while (p.workers < helpers && p.workers < most) {
                std::thread([&p] { p.serve(); }).detach();
                p.workers++;
            }
        } catch (...) {   // (no more threads to be had: those that run, and the caller, do the work)
        }
        at = p.jobs.insert(p.jobs.end(), &job);
    }
    if (helpers >= 4) p.work.notify_all();
    else for (int i = 0; i < helpers; i++) p.work.notify_one();
    job.run();
    std::unique_lock<std::mutex> lock(p.mu);
    p.jobs.erase(at);
    p.left.wait(lock, [&] { return job.helpers == 0; });
}
