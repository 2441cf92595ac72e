// Transfers between host arrays and device memory on a context's stream, through pinned memory.
//
// A pageable hipMemcpyAsync costs 10 us whatever its size and moves 29 GB/s in, 18 GB/s out; pinned memory moves 57 GB/s
// either way.  Up to kSmallTransfer bytes a copy kernel in the stream reads (writes) the pinned staging memory: it costs
// one dependent launch, 3.5 us, where a transfer by the copy engine between kernels of the stream costs two hand-overs
// between queues (64 KB in, a kernel, 64 KB out: 18 against 30 us).  From there on the copy engine's rate is the better
// one (5 MB in: 99 against 132 us; results that go to pinned memory stay with the kernel up to 8 MB); the blocks of a large input are copied into staging memory by several threads while the
// engine moves those before them.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <vector>

constexpr size_t kSmallTransfer = 1u << 20;

struct FnnHostIo {
    unsigned char *small = nullptr;     // kSmallTransfer bytes of pinned memory handed out from the start between two waits
    size_t small_used = 0;
    std::vector<void *> borrowed;       // staging blocks of large inputs, given back by wait()
    uint32_t *flag = nullptr;           // a word of pinned memory that a kernel of the stream writes last
    uint32_t epoch = 0;
    struct Pending { void *dst; const void *src; size_t bytes; };
    std::vector<Pending> pending;       // results in staging memory, copied out when the stream has reached them

    bool touched = false;               // transfers from or to the caller's own (pinned) memory may be under way

    // A call that works in parts: the transfers of one part pass beside the kernels of another, inputs on `ahead`, outputs on `behind`
    // (made on first use, at the default priority).  The stream `s` waits for a part's input, `behind` for its mark.
    static constexpr int kParts = 2;
    hipStream_t ahead = nullptr, behind = nullptr;
    hipEvent_t ev_fork = nullptr, ev_in[kParts] = {}, ev_part[kParts] = {}, ev_out = nullptr;
    bool out_behind = false;            // `behind` has transfers that no wait has joined yet
    hipError_t begin_parts(hipStream_t s);                                                   // behind everything enqueued on s so far
    hipError_t in_part(hipStream_t s, int part, void *dst, const void *src, size_t bytes);   // more than kSmallTransfer; src held
    hipError_t mark_part(hipStream_t s, int part);                                           // the part's kernels are enqueued
    hipError_t out_part(int part, void *dst, const void *src, size_t bytes);

    void destroy();
    // enqueues host -> device; the transfer is done when the stream gets there.  held: the caller leaves `src` alone until the
    // wait that ends its call (also one that fails: abandon); else it may be reused on return
    hipError_t in(hipStream_t s, void *dst, const void *src, size_t bytes, bool held);
    // two inputs into one allocation, the second at offset at1 >= bytes0 (small ones: in one launch)
    hipError_t in2(hipStream_t s, void *dst, const void *src0, size_t bytes0, size_t at1, const void *src1, size_t bytes1, bool held);
    // enqueues device -> host; `dst` holds the result after wait()
    hipError_t out(hipStream_t s, void *dst, const void *src, size_t bytes);
    // staging memory that kernels of the stream may write results to and that wait() copies to `dst`; null: too large
    void *result_slot(void *dst, size_t bytes);
    // waits until the stream has done everything enqueued and finishes the outputs
    hipError_t wait(hipStream_t s);
    // instead of wait() where a call fails half way: its results go nowhere, and nothing touches the caller's memory any more
    void abandon(hipStream_t s);

private:
    hipError_t take_small(hipStream_t s, size_t bytes, size_t align_like, unsigned char **p);
    hipError_t in_large(hipStream_t s, unsigned char *dst, const unsigned char *src, size_t bytes);
};

// Pinned blocks for result arrays, shared by the process.  At most kPinnedLive bytes exist and kPinnedKept of them are kept
// unused; null when there is no room (the caller takes ordinary memory).
void *fnn_pinned_alloc(size_t bytes);
void fnn_pinned_free(void *p);
bool fnn_is_pinned(const void *p, size_t bytes);
