#include "host_pool.h"

#include <atomic>
#include <condition_variable>
#include <list>
#include <mutex>
#include <thread>

#include <pthread.h>
#include <sched.h>

namespace {

struct Pool {
    std::mutex mu;
    std::condition_variable work, left;
    std::list<FnnJob *> jobs;
    int workers = 0;

    void serve()
    {
        std::unique_lock<std::mutex> lock(mu);
        for (;;) {
            FnnJob *job = nullptr;
            for (FnnJob *j : jobs)
                if (j->helpers < j->helpers_max && j->next.load(std::memory_order_relaxed) < j->tasks) { job = j; break; }
            if (!job) { work.wait(lock); continue; }
            job->helpers++;
            lock.unlock();
            while (job->run_one()) {}
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

void FnnJob::begin(int threads)
{
    Pool &p = *g_pool;
    helpers_max = (int)(threads - 1 < tasks - 1 ? threads - 1 : tasks - 1);
    if (helpers_max <= 0) return;
    {
        std::lock_guard<std::mutex> lock(p.mu);
        const int most = fnn_host_threads() - 1;
        try {
            while (p.workers < helpers_max && p.workers < most) {
                std::thread([&p] { p.serve(); }).detach();
                p.workers++;
            }
        } catch (...) {   // (no more threads to be had: those that run, and the caller, do the work)
        }
        p.jobs.push_back(this);
        queued = true;
    }
    if (helpers_max >= 4) p.work.notify_all();
    else for (int i = 0; i < helpers_max; i++) p.work.notify_one();
}

void FnnJob::end()
{
    while (run_one()) {}
    if (!queued) return;
    Pool &p = *g_pool;
    std::unique_lock<std::mutex> lock(p.mu);
    p.jobs.remove(this);
    p.left.wait(lock, [&] { return helpers == 0; });
}
