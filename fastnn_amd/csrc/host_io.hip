#include "host_io.h"

#include <immintrin.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstring>
#include <map>
#include <mutex>

#include "host_pool.h"

namespace {

constexpr size_t kPinnedLive = 1u << 30, kPinnedKept = 256u << 20;
// A kernel's stores leave for pinned memory at the link's rate too, and it needs no hand-over to the copy engine and back: 1.6 MB out 52 -> 40 us,
// 3.3 MB 83 -> 72, 8 MB 170 -> 161; from 13 MB on the engine is ahead (260 against 264).  (Its loads from there are slower.)
constexpr size_t kKernelOut = 8u << 20;
constexpr size_t kBlock = 512u << 10;              // of a large input: one task of the copying threads
constexpr size_t kLargeStaging = 256u << 20;       // larger inputs are left to the runtime
constexpr int kCopyThreads = 8;                    // (one thread copies 31 GB/s from memory, the engine moves 57)
constexpr auto kSpin = std::chrono::microseconds(200);

// T = the widest access that source, destination and size allow
template <class T>
__global__ __launch_bounds__(256) void copy_kernel(const T *__restrict__ src, T *__restrict__ dst, size_t n)
{
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) dst[i] = src[i];
}

// Everything before this kernel in the stream is done when it starts; writes to pinned memory are not cached on the device.
__global__ void signal_kernel(uint32_t *flag, uint32_t value)
{
    __hip_atomic_store(flag, value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

template <class T>
hipError_t launch_copy(hipStream_t s, void *dst, const void *src, size_t bytes)
{
    const size_t n = bytes / sizeof(T);
    copy_kernel<T><<<(unsigned)((n + 255) / 256), 256, 0, s>>>((const T *)src, (T *)dst, n);
    return hipGetLastError();
}

hipError_t device_copy(hipStream_t s, void *dst, const void *src, size_t bytes)
{
    const uintptr_t low = reinterpret_cast<uintptr_t>(dst) | reinterpret_cast<uintptr_t>(src) | bytes;
    if (!(low & 15)) return launch_copy<uint4>(s, dst, src, bytes);
    if (!(low & 3)) return launch_copy<uint32_t>(s, dst, src, bytes);
    return launch_copy<uint8_t>(s, dst, src, bytes);
}

struct PinnedPool {
    std::mutex mu;
    std::map<uintptr_t, size_t> blocks;            // every block, by address
    std::multimap<size_t, void *> unused;
    size_t live = 0, kept = 0;
};
PinnedPool &pinned() { static PinnedPool *p = new PinnedPool(); return *p; }   // (never destroyed: arrays may outlive it)

}  // namespace

void *fnn_pinned_alloc(size_t bytes)
{
    size_t cap = 64u << 10;                        // 64 KB, then four sizes per power of two
    while (cap < bytes) cap <<= 1;
    for (size_t c = cap / 2 + cap / 8; c < cap && cap > (64u << 10); c += cap / 8)
        if (c >= bytes) { cap = c; break; }
    PinnedPool &p = pinned();
    {
        std::lock_guard<std::mutex> lock(p.mu);
        auto it = p.unused.lower_bound(cap);
        if (it != p.unused.end() && it->first <= 2 * cap) {
            void *b = it->second;
            p.kept -= it->first;
            p.unused.erase(it);
            return b;
        }
        if (p.live + cap > kPinnedLive) return nullptr;
        p.live += cap;
    }
    void *b = nullptr;
    const bool ok = hipHostMalloc(&b, cap, hipHostMallocCoherent) == hipSuccess;
    if (!ok) (void)hipGetLastError();
    std::lock_guard<std::mutex> lock(p.mu);
    if (!ok) { p.live -= cap; return nullptr; }
    p.blocks[reinterpret_cast<uintptr_t>(b)] = cap;
    return b;
}

void fnn_pinned_free(void *ptr)
{
    if (!ptr) return;
    PinnedPool &p = pinned();
    {
        std::lock_guard<std::mutex> lock(p.mu);
        auto it = p.blocks.find(reinterpret_cast<uintptr_t>(ptr));
        if (it == p.blocks.end()) return;
        if (p.kept + it->second <= kPinnedKept) {
            p.kept += it->second;
            p.unused.emplace(it->second, ptr);
            return;
        }
        p.live -= it->second;
        p.blocks.erase(it);
    }
    (void)hipHostFree(ptr);
}

bool fnn_is_pinned(const void *ptr, size_t bytes)
{
    const uintptr_t a = reinterpret_cast<uintptr_t>(ptr);
    PinnedPool &p = pinned();
    std::lock_guard<std::mutex> lock(p.mu);
    auto it = p.blocks.upper_bound(a);
    if (it == p.blocks.begin()) return false;
    --it;
    return a + bytes <= it->first + it->second;
}

void FnnHostIo::destroy()
{
    if (small) (void)hipHostFree(small);
    for (void *b : borrowed) fnn_pinned_free(b);
    borrowed.clear();
    if (flag) (void)hipHostFree(flag);
    small = nullptr;
    flag = nullptr;
    for (hipStream_t *t : {&ahead, &behind})
        if (*t) {
            (void)hipStreamSynchronize(*t);
            (void)hipStreamDestroy(*t);
            *t = nullptr;
        }
    for (hipEvent_t *e : {&ev_fork, &ev_in[0], &ev_in[1], &ev_part[0], &ev_part[1], &ev_out})
        if (*e) {
            (void)hipEventDestroy(*e);
            *e = nullptr;
        }
}

hipError_t FnnHostIo::begin_parts(hipStream_t s)
{
    hipError_t e;
    for (hipStream_t *t : {&ahead, &behind})
        if (!*t && (e = hipStreamCreateWithFlags(t, hipStreamNonBlocking)) != hipSuccess) return e;
    for (hipEvent_t *v : {&ev_fork, &ev_in[0], &ev_in[1], &ev_part[0], &ev_part[1], &ev_out})
        if (!*v && (e = hipEventCreateWithFlags(v, hipEventDisableTiming)) != hipSuccess) return e;
    if ((e = hipEventRecord(ev_fork, s)) != hipSuccess) return e;
    return hipStreamWaitEvent(ahead, ev_fork, 0);
}

hipError_t FnnHostIo::in_part(hipStream_t s, int part, void *dst, const void *src, size_t bytes)
{
    hipError_t e;
    if (bytes <= kSmallTransfer) return hipErrorInvalidValue;   // (those share staging memory that a wait on s hands out anew)
    if ((e = in(ahead, dst, src, bytes, true)) != hipSuccess || (e = hipEventRecord(ev_in[part], ahead)) != hipSuccess) return e;
    return hipStreamWaitEvent(s, ev_in[part], 0);
}

hipError_t FnnHostIo::mark_part(hipStream_t s, int part) { return hipEventRecord(ev_part[part], s); }

hipError_t FnnHostIo::out_part(int part, void *dst, const void *src, size_t bytes)
{
    const hipError_t e = hipStreamWaitEvent(behind, ev_part[part], 0);
    touched = out_behind = true;
    return e != hipSuccess ? e : hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, behind);
}

hipError_t FnnHostIo::take_small(hipStream_t s, size_t bytes, size_t align_like, unsigned char **p)
{
    hipError_t e;
    if (!small && (e = hipHostMalloc((void **)&small, kSmallTransfer + 256, hipHostMallocCoherent)) != hipSuccess) return e;
    size_t at = (small_used + 63) / 64 * 64 + align_like % 16;
    if (at + bytes > kSmallTransfer + 256) {       // full: what was handed out is free once the stream has passed it
        if ((e = wait(s)) != hipSuccess) return e;
        at = align_like % 16;
    }
    small_used = at + bytes;
    *p = small + at;
    return hipSuccess;
}

hipError_t FnnHostIo::in2(hipStream_t s, void *dst, const void *src0, size_t bytes0, size_t at1, const void *src1, size_t bytes1, bool held)
{
    if (!bytes1 || at1 + bytes1 > kSmallTransfer) {
        const hipError_t e = in(s, dst, src0, bytes0, held);
        return e != hipSuccess || !bytes1 ? e : in(s, (unsigned char *)dst + at1, src1, bytes1, held);
    }
    unsigned char *p;
    const hipError_t e = take_small(s, at1 + bytes1, reinterpret_cast<uintptr_t>(dst), &p);
    if (e != hipSuccess) return e;
    std::memcpy(p, src0, bytes0);
    std::memcpy(p + at1, src1, bytes1);
    return device_copy(s, dst, p, at1 + bytes1);
}

hipError_t FnnHostIo::in(hipStream_t s, void *dst, const void *src, size_t bytes, bool held)
{
    if (!bytes) return hipSuccess;
    if ((held || bytes > kSmallTransfer) && fnn_is_pinned(src, bytes)) {   // a result array of an earlier call: no staging
        touched = true;
        const hipError_t e = bytes <= kSmallTransfer ? device_copy(s, dst, src, bytes) : hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s);
        return e != hipSuccess || held ? e : hipStreamSynchronize(s);
    }
    if (bytes > kSmallTransfer) return in_large(s, (unsigned char *)dst, (const unsigned char *)src, bytes);
    unsigned char *p;
    const hipError_t e = take_small(s, bytes, reinterpret_cast<uintptr_t>(dst), &p);
    if (e != hipSuccess) return e;
    std::memcpy(p, src, bytes);
    return device_copy(s, dst, p, bytes);
}

hipError_t FnnHostIo::in_large(hipStream_t s, unsigned char *dst, const unsigned char *src, size_t bytes)
{
    unsigned char *stage = nullptr;
    if (bytes <= kLargeStaging) {
        borrowed.reserve(borrowed.size() + 1);
        stage = (unsigned char *)fnn_pinned_alloc(bytes);
    }
    if (!stage) {
        const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s);
        return e != hipSuccess ? e : hipStreamSynchronize(s);
    }
    borrowed.push_back(stage);
    const int64_t blocks = (int64_t)((bytes + kBlock - 1) / kBlock);
    struct Copy {
        unsigned char *to;
        const unsigned char *from;
        size_t bytes;
        std::vector<std::atomic<uint8_t>> done;
    } copy{stage, src, bytes, std::vector<std::atomic<uint8_t>>((size_t)blocks)};
    FnnJob job(blocks, [](void *arg, int64_t i) {
        Copy &c = *static_cast<Copy *>(arg);
        const size_t at = (size_t)i * kBlock;
        std::memcpy(c.to + at, c.from + at, std::min(kBlock, c.bytes - at));
        c.done[(size_t)i].store(1, std::memory_order_release);
    }, &copy);
    job.begin(std::min(fnn_host_threads(), kCopyThreads));
    // Every transfer costs the engine 9 us beside its bytes (78 MB in blocks of 1 MB: 2.1 ms, of 8 MB: 1.48 ms), so they
    // grow: 8 MB, then as much as the one before took time for the threads to stage.
    hipError_t e = hipSuccess;
    int64_t ready = 0;
    for (size_t sent = 0, want = 8u << 20; sent < bytes && e == hipSuccess;) {
        while (ready < blocks && copy.done[(size_t)ready].load(std::memory_order_acquire)) ready++;
        const size_t have = ready == blocks ? bytes : (size_t)ready * kBlock;
        if (have - sent >= std::min(want, bytes - sent)) {
            e = hipMemcpyAsync(dst + sent, stage + sent, have - sent, hipMemcpyHostToDevice, s);
            sent = have;
            want = 16u << 20;
        } else if (!job.run_one()) {
            _mm_pause();
        }
    }
    job.end();
    return e;
}

hipError_t FnnHostIo::out(hipStream_t s, void *dst, const void *src, size_t bytes)
{
    if (!bytes) return hipSuccess;
    const bool wide = !((reinterpret_cast<uintptr_t>(dst) | reinterpret_cast<uintptr_t>(src) | bytes) & 15);
    if (bytes <= (wide ? kKernelOut : kSmallTransfer) && fnn_is_pinned(dst, bytes)) {
        touched = true;
        return device_copy(s, dst, src, bytes);
    }
    if (bytes > kSmallTransfer) {
        touched = true;
        return hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s);
    }
    unsigned char *p;
    const hipError_t e = take_small(s, bytes, reinterpret_cast<uintptr_t>(src), &p);
    if (e != hipSuccess) return e;
    pending.push_back({dst, p, bytes});
    return device_copy(s, p, src, bytes);
}

void *FnnHostIo::result_slot(void *dst, size_t bytes)
{
    unsigned char *p;
    const size_t at = (small_used + 63) / 64 * 64;
    if (!small || at + bytes > kSmallTransfer + 256) return nullptr;
    small_used = at + bytes;
    p = small + at;
    pending.push_back({dst, p, bytes});
    return p;
}

hipError_t FnnHostIo::wait(hipStream_t s)
{
    hipError_t e = hipSuccess;
    bool seen = false;
    if (!flag) {
        if ((e = hipHostMalloc((void **)&flag, 64, hipHostMallocCoherent)) != hipSuccess) return e;
        *flag = 0;
    }
    if (out_behind) {   // (`ahead` is joined already: s waits for every input)
        if ((e = hipEventRecord(ev_out, behind)) == hipSuccess) e = hipStreamWaitEvent(s, ev_out, 0);
        if (e != hipSuccess) (void)hipStreamSynchronize(behind);
        out_behind = false;
    }
    // A word that the stream's last kernel writes reaches the host 3.7 us before hipStreamSynchronize returns; after
    // kSpin of polling the runtime's wait takes over (it is also the one that reports a failed kernel).
    signal_kernel<<<1, 1, 0, s>>>(flag, ++epoch);
    if (hipError_t launched = hipGetLastError(); e == hipSuccess) e = launched;
    if (e == hipSuccess) {
        const auto until = std::chrono::steady_clock::now() + kSpin;
        for (int i = 1; !(seen = __atomic_load_n(flag, __ATOMIC_ACQUIRE) == epoch); i++) {
            _mm_pause();
            if (i % 64 == 0 && std::chrono::steady_clock::now() > until) break;
        }
    }
    if (!seen) {
        const hipError_t w = hipStreamSynchronize(s);
        if (e == hipSuccess) e = w;
    }
    if (e == hipSuccess)
        for (const Pending &p : pending) std::memcpy(p.dst, p.src, p.bytes);
    pending.clear();
    for (void *b : borrowed) fnn_pinned_free(b);
    borrowed.clear();
    small_used = 0;
    touched = false;
    return e;
}

void FnnHostIo::abandon(hipStream_t s)
{
    if (ahead) {
        (void)hipStreamSynchronize(ahead);
        (void)hipStreamSynchronize(s);   // (`behind` waits for marks on it)
        if (behind) (void)hipStreamSynchronize(behind);
        out_behind = false;
    }
    if (touched) (void)hipStreamSynchronize(s);
    touched = false;
    pending.clear();   // (what it staged stays taken until the next wait)
}
