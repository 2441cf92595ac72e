// Worker threads of the library's host side (weight packers, staging copies): started on first use, kept, shared by
// every caller of the process.
#pragma once
#include <cstdint>

// Runs fn(arg, i) for every i in [0, tasks) on up to `threads` threads, the caller among them, and returns when all are
// done.  Safe from several threads at once (their jobs share the workers) and in a forked child (whose workers are gone:
// the caller runs every task itself).  `fn` must not throw.
void fnn_parallel_raw(int64_t tasks, int threads, void (*fn)(void *arg, int64_t task), void *arg);

// CPUs this process may run on, at most 16
int fnn_host_threads();

template <class F>
void fnn_parallel(int64_t tasks, int threads, F &&f)
{
    fnn_parallel_raw(tasks, threads, [](void *arg, int64_t i) { (*static_cast<F *>(arg))(i); }, (void *)&f);
}
