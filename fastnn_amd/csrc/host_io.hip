#include "host_io.h"

#include <immintrin.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstring>
#include <map>
#include <mutex>
#include <thread>

#include "host_pool.h"
#include "range_io.h"

namespace {

constexpr size_t kPinnedLive = 1u << 30, kPinnedKept = 256u << 20;
// A kernel's stores leave for pinned memory at the link's rate too, and it needs no hand-over to the copy engine and back: 1.6 MB out 52 -> 40 us,
// 3.3 MB 83 -> 72, 8 MB 170 -> 161; from 13 MB on the engine is ahead (260 against 264).  (Its loads from there are slower.)
constexpr size_t kKernelOut = 8u << 20;
constexpr size_t kBlock = 128u << 10;              // of a large input: one task of the copying threads
constexpr size_t kFirstSent = 512u << 10;
constexpr size_t kLargeStaging = 256u << 20;       // larger inputs are left to the runtime
constexpr int kCopyThreads = 8;                    // (one thread copies 31 GB/s from memory, the engine moves 57)
constexpr auto kSpin = std::chrono::microseconds(200);
// Results of up to kWatched bytes are polled themselves (1 x 1024 x 1024 14.3 -> 13.2 us, 4 x 1024 x 1024 16.0 -> 15.0, the same at 64 KB): their staging memory is filled with a word that no arithmetic makes (a not-a-number with a
// payload; one that a caller passes in and gets out again costs kSpin), and what differs from it has been written.  It spares the launch of
// signal_kernel behind the last one of the call, which with its distance from it is 3 us.
constexpr size_t kWatched = 40u << 10;
// For a mark the host polls this long without a pause (a detector's pass on 16 images of 640 x 640 reaches its first in 1.6 ms), from there on between pauses of a
// sixteenth of the time that it has waited, at most 1 ms: what a result then leaves late is small beside the pass.
constexpr auto kMarkSpin = std::chrono::milliseconds(4), kMarkPause = std::chrono::milliseconds(1);
constexpr uint32_t kUnwritten = 0xffd3b5c9u;

// T = the widest access that source, destination and size allow
template <class T>
__global__ __launch_bounds__(256) void copy_kernel(const T *__restrict__ src, T *__restrict__ dst, size_t n)
{
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) dst[i] = src[i];
}

// Everything before this kernel in the stream is done when it starts; writes to pinned memory are not cached on the device.
// As a mark it lets another stream's copy begin, with no wait between the two but the host's look at the word.  That holds because a
// kernel sees what those before it in its stream wrote on any XCD: where each XCD has an L2 of its own, the end of a kernel puts its lines
// into memory.  The release at system scope hands all that this kernel could see to whoever has seen the word, and the copy is enqueued after that.  A
// runtime that ended kernels without their release would break this, and the kernel behind as well.
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

// One look at a watched result: what is there by now, in pieces of 64 bytes from *at on, goes to dst; true: all of it.  (A word at a time it was slower than
// the signal it spares from 16 KB on.)
bool take_written(const FnnHostIo::Pending &p, size_t *at)
{
    const unsigned char *src = static_cast<const unsigned char *>(p.src);
    unsigned char *dst = static_cast<unsigned char *>(p.dst);
    const __m128i unwritten = _mm_set1_epi32((int)kUnwritten);
    size_t i = *at;
    for (; i + 64 <= p.bytes; i += 64) {
        __m128i v[4];
        for (int j = 0; j < 4; j++) v[j] = _mm_loadu_si128(reinterpret_cast<const __m128i *>(src + i) + j);
        const __m128i missing = _mm_or_si128(_mm_or_si128(_mm_cmpeq_epi32(v[0], unwritten), _mm_cmpeq_epi32(v[1], unwritten)),
                                             _mm_or_si128(_mm_cmpeq_epi32(v[2], unwritten), _mm_cmpeq_epi32(v[3], unwritten)));
        if (_mm_movemask_epi8(missing)) break;
        for (int j = 0; j < 4; j++) _mm_storeu_si128(reinterpret_cast<__m128i *>(dst + i) + j, v[j]);
    }
    if (i + 64 > p.bytes)
        for (; i < p.bytes; i += 4) {
            const uint32_t w = __atomic_load_n(reinterpret_cast<const uint32_t *>(src + i), __ATOMIC_RELAXED);
            if (w == kUnwritten) break;
            std::memcpy(dst + i, &w, 4);
        }
    std::atomic_signal_fence(std::memory_order_seq_cst);   // (the next look reads again)
    *at = i;
    return i == p.bytes;
}

// Into staging memory that only the engine reads: past the caches, which spares the lines' way into them and back.
void stream_copy(unsigned char *to, const unsigned char *from, size_t bytes)
{
    if ((reinterpret_cast<uintptr_t>(to) & 15) == 0) {
        for (; bytes >= 64; bytes -= 64, to += 64, from += 64) {
            __m128i v[4];
            for (int i = 0; i < 4; i++) v[i] = _mm_loadu_si128(reinterpret_cast<const __m128i *>(from) + i);
            for (int i = 0; i < 4; i++) _mm_stream_si128(reinterpret_cast<__m128i *>(to) + i, v[i]);
        }
        _mm_sfence();
    }
    std::memcpy(to, from, bytes);
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
    if (marks) (void)hipHostFree(marks);
    marks = nullptr;
    for (hipStream_t *t : {&ahead, &behind})
        if (*t) {
            (void)hipStreamSynchronize(*t);
            (void)hipStreamDestroy(*t);
            *t = nullptr;
        }
    for (hipEvent_t *e : {&ev_fork, &ev_in[0], &ev_in[1]})
        if (*e) {
            (void)hipEventDestroy(*e);
            *e = nullptr;
        }
}

hipError_t FnnHostIo::make_streams()
{
    hipError_t e;
    for (hipStream_t *t : {&ahead, &behind})
        if (!*t && (e = hipStreamCreateWithFlags(t, hipStreamNonBlocking)) != hipSuccess) return e;
    for (hipEvent_t *v : {&ev_fork, &ev_in[0], &ev_in[1]})
        if (!*v && (e = hipEventCreateWithFlags(v, hipEventDisableTiming)) != hipSuccess) return e;
    return hipSuccess;
}

bool FnnHostIo::marks_ready()
{
    if (marks) return true;
    if (make_streams() != hipSuccess || hipHostMalloc((void **)&marks, FNN_MARKS * 64, hipHostMallocCoherent) != hipSuccess) {
        (void)hipGetLastError();
        marks = nullptr;
    }
    return marks != nullptr;
}

void FnnHostIo::clear_mark(int i) { if (marks) __atomic_store_n(marks + i * 16, 0u, __ATOMIC_RELEASE); }

hipError_t FnnHostIo::mark(hipStream_t s, int i)
{
    if (!marks) return hipSuccess;   // (a plan cut on another context: nobody here waits for the mark)
    signal_kernel<<<1, 1, 0, s>>>(marks + i * 16, 1u);
    return hipGetLastError();
}

hipError_t FnnHostIo::send(hipStream_t s, int i, void *dst, const void *src, size_t bytes)
{
    const auto from = std::chrono::steady_clock::now();
    for (int n = 1; __atomic_load_n(marks + i * 16, __ATOMIC_ACQUIRE) == 0; n++) {
        _mm_pause();
        if (n % 64) continue;
        const auto waited = std::chrono::steady_clock::now() - from;
        if (waited < kMarkSpin) continue;
        const hipError_t e = hipStreamQuery(s);   // (the stream's end is as good, and its failure ends the wait)
        if (e == hipSuccess) break;
        if (e != hipErrorNotReady) return e;
        (void)hipGetLastError();
        std::this_thread::sleep_for(std::min<std::chrono::steady_clock::duration>(waited / 16, kMarkPause));
        n = 63;   // (one look, then the clock again)
    }
    touched = out_behind = true;
    return hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, behind);
}

hipError_t FnnHostIo::begin_parts(hipStream_t s)
{
    hipError_t e = make_streams();
    if (e != hipSuccess) return e;
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
    results_last = false;
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
    results_last = false;
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
        stream_copy(c.to + at, c.from + at, std::min(kBlock, c.bytes - at));
        c.done[(size_t)i].store(1, std::memory_order_release);
    }, &copy);
    job.begin(std::min(fnn_host_threads(), kCopyThreads));
    // Every transfer costs the engine 9 us beside its bytes (78 MB in blocks of 1 MB: 2.1 ms, of 8 MB: 1.48 ms), so they
    // grow: the first begins soon, each later one is as much as those before it took time for the threads to stage.
    hipError_t e = hipSuccess;
    int64_t ready = 0;
    for (size_t sent = 0, want = kFirstSent; sent < bytes && e == hipSuccess;) {
        while (ready < blocks && copy.done[(size_t)ready].load(std::memory_order_acquire)) ready++;
        const size_t have = ready == blocks ? bytes : (size_t)ready * kBlock;
        if (have - sent >= std::min(want, bytes - sent)) {
            e = hipMemcpyAsync(dst + sent, stage + sent, have - sent, hipMemcpyHostToDevice, s);
            sent = have;
            want = std::min<size_t>(want * 3, 16u << 20);
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
    if (!((reinterpret_cast<uintptr_t>(p) | reinterpret_cast<uintptr_t>(src) | bytes) & 3)) watch(p, bytes, dst);   // (else the copy is of bytes)
    else pending.push_back({dst, p, bytes, false});
    return device_copy(s, p, src, bytes);
}

void FnnHostIo::watch(void *p, size_t bytes, void *dst)
{
    const bool watched = bytes <= kWatched;
    if (watched) std::fill_n(static_cast<uint32_t *>(p), bytes / 4, kUnwritten);
    pending.push_back({dst, p, bytes, watched});
    results_last = true;
}

bool FnnHostIo::results_tell() const
{
    size_t bytes = 0;
    for (const Pending &p : pending) {
        if (!p.watched) return false;
        bytes += p.bytes;
    }
    return bytes && bytes <= kWatched && results_last && !touched && !out_behind;
}

void *FnnHostIo::result_slot(void *dst, size_t bytes)
{
    unsigned char *p;
    const size_t at = (small_used + 63) / 64 * 64;
    if (!small || at + bytes > kSmallTransfer + 256) return nullptr;
    small_used = at + bytes;
    p = small + at;
    watch(p, bytes, dst);
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
    const auto spin = [](auto &&done) {
        const auto until = std::chrono::steady_clock::now() + kSpin;
        for (int i = 1; !done(); i++) {
            _mm_pause();
            if (i % 64 == 0 && std::chrono::steady_clock::now() > until) return false;
        }
        return true;
    };
    // What the stream's last kernel writes reaches the host 3.7 us before hipStreamSynchronize returns; after kSpin of polling
    // the runtime's wait takes over (it is also the one that reports a failed kernel).
    if (e == hipSuccess && results_tell()) {
        size_t result = 0, at = 0;
        seen = spin([&] {
            while (result < pending.size() && take_written(pending[result], &at)) result++, at = 0;
            return result == pending.size();
        });
        if (seen) pending.clear();   // (taken)
    } else {
        signal_kernel<<<1, 1, 0, s>>>(flag, ++epoch);
        if (hipError_t launched = hipGetLastError(); e == hipSuccess) e = launched;
        if (e == hipSuccess) seen = spin([&] { return __atomic_load_n(flag, __ATOMIC_ACQUIRE) == epoch; });
    }
    if (!seen) {
        const hipError_t w = hipStreamSynchronize(s);
        if (e == hipSuccess) e = w;
    }
    if (out_behind) {   // (`ahead` is joined already: s waits for every input)
        const hipError_t w = hipStreamSynchronize(behind);
        if (e == hipSuccess) e = w;
        out_behind = false;
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
        (void)hipStreamSynchronize(s);
        if (behind) (void)hipStreamSynchronize(behind);
        out_behind = false;
    }
    if (touched) (void)hipStreamSynchronize(s);
    touched = false;
    pending.clear();   // (what it staged stays taken until the next wait)
}
