// Host-side weight packers of libfastnn_hip: the quantisers fastnn's compiler pass
// applies to constant MatMul / Conv weights before a backend sees them
// (src/compiler/passes/quantization.rs:170-260, 281-495).  Results are bit-identical to
// fastnn's: strict binary32 arithmetic in the reference's evaluation order (this file is
// compiled with FMA contraction off); only order-independent work is spread over threads.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <memory>
#include <new>
#include <vector>

#include "../../include/fastnn_hip.h"
#include "host_pool.h"
#include "quantize_simd.h"

namespace {

constexpr size_t kMargin = 16;  // SIMD_MARGIN words after the last row (src/packed_tensor.rs:980-982)
constexpr int64_t kPanel = 32;  // channels a packing task takes at a time

inline int lanes_of(int dt)
{
    switch (dt) {
    case FNN_DT_I8: case FNN_DT_U8: case FNN_DT_F8: case FNN_DT_F8R: return 4;
    case FNN_DT_I4: case FNN_DT_U4: case FNN_DT_F4: case FNN_DT_I4CB: return 8;
    default: return 0;
    }
}

const FnnQuantKernels &kernels()
{
    static const FnnQuantKernels &k = __builtin_cpu_supports("avx512f") && __builtin_cpu_supports("avx512bw") && __builtin_cpu_supports("avx512dq") && __builtin_cpu_supports("avx512vl")
                                          ? fnn_quant_avx512
                                          : (__builtin_cpu_supports("avx2") ? fnn_quant_avx2 : fnn_quant_base);
    return k;
}

int threads_for(int64_t elements) { return elements < (1 << 16) ? 1 : fnn_host_threads(); }

// A task's working copy of a panel (inner x 32 floats), kept by its thread up to 4 MB so that no call pays for fresh pages.
struct PanelBuffer {
    std::unique_ptr<float[]> own;
    size_t cap = 0;
    float *get(size_t n)
    {
        if (n > cap) { own.reset(); own.reset(new float[n]); cap = n; }
        return own.get();
    }
    void done() { if (cap > (1u << 20)) { own.reset(); cap = 0; } }
};
thread_local PanelBuffer t_panel;

// Per-channel packing of an [inner, rows] matrix (kn: channels along the fast axis, as a graph holds a MatMul weight: a
// panel is read where it lies) or of its transpose (each panel is turned first).  src/packed_tensor.rs:661-742, 852-1049.
// A [4096, 11008] matrix to 4-bit words on 16 EPYC threads: 251 ms as a serial transpose followed by scalar packing,
// 1.2 ms in this form (169 GB/s of floats read, the host memory's rate).
bool quant_per_channel(int dtype, const float *w, int64_t rows, int64_t inner, bool kn, uint32_t *words, float *scales, float *zeros)
{
    const FnnQuantKernels &kern = kernels();
    const int items = lanes_of(dtype);
    const int64_t kp = (inner + items - 1) / items;
    std::atomic<bool> ok{true};
    fnn_parallel((rows + kPanel - 1) / kPanel, threads_for(rows * inner), [&](int64_t p) {
        const int64_t r0 = p * kPanel;
        const int have = (int)std::min(kPanel, rows - r0);
        const float *src = w + r0;
        int64_t ld = rows;
        if (!kn || have < kPanel) {
            float *buf;
            try { buf = t_panel.get((size_t)inner * kPanel); } catch (const std::bad_alloc &) { ok = false; return; }
            if (kn) {
                for (int64_t k = 0; k < inner; k++) {
                    std::memcpy(buf + k * kPanel, w + k * rows + r0, (size_t)have * 4);
                    std::memset(buf + k * kPanel + have, 0, (size_t)(kPanel - have) * 4);
                }
            } else {
                kern.panel_from_rows(w + r0 * inner, inner, have, buf);
            }
            src = buf;
            ld = kPanel;
        }
        kern.quant_panel(dtype, src, ld, inner, have, words + r0 * kp, kp, scales + r0, zeros + r0);
        t_panel.done();
    });
    return ok;
}

// ---- codebook

constexpr int64_t kChunk = 1 << 14;   // values of one task of the flat passes

// The values at 16 positions of the stable ascending order of `vals` (-0.0 and +0.0 are equal there and keep the order
// they came in).  Histogram of the upper 16 bits of the order-preserving integer image, then a selection inside the
// buckets that hold the positions: what a full sort gives at these positions (1 M values: 75 ms sorted, 2 ms here).
void order_statistics(const std::vector<float> &vals, const size_t *at, float *out)
{
    const int64_t n = (int64_t)vals.size();
    auto key = [](float f) -> uint32_t {
        uint32_t u;
        std::memcpy(&u, &f, 4);
        if ((u << 1) == 0) u = 0;
        return u & 0x80000000u ? ~u : u | 0x80000000u;
    };
    const int threads = threads_for(n);
    std::vector<std::vector<uint32_t>> part((size_t)threads, std::vector<uint32_t>(1 << 16, 0));
    const int64_t per = (n + threads - 1) / threads;
    fnn_parallel(threads, threads, [&](int64_t t) {
        for (int64_t i = t * per; i < std::min(n, (t + 1) * per); i++) part[(size_t)t][key(vals[(size_t)i]) >> 16]++;
    });
    std::vector<uint64_t> before((1 << 16) + 1, 0);
    for (size_t b = 0; b < 1 << 16; b++) {
        uint64_t c = 0;
        for (auto &p : part) c += p[b];
        before[b + 1] = before[b] + c;
    }
    uint32_t bucket[16];
    for (int j = 0; j < 16; j++)
        bucket[j] = (uint32_t)(std::upper_bound(before.begin(), before.end(), (uint64_t)at[j]) - before.begin() - 1);
    std::vector<std::vector<uint32_t>> found(16);
    std::vector<uint8_t> slot(1 << 16, 255);
    for (int j = 0; j < 16; j++) if (slot[bucket[j]] == 255) slot[bucket[j]] = (uint8_t)j;
    for (int j = 0; j < 16; j++) if (slot[bucket[j]] == j) found[(size_t)j].reserve(before[bucket[j] + 1] - before[bucket[j]]);
    for (float v : vals) {
        const uint32_t k = key(v);
        if (const uint8_t s = slot[k >> 16]; s != 255) found[s].push_back(k);
    }
    for (int j = 0; j < 16; j++) {
        std::vector<uint32_t> &f = found[slot[bucket[j]]];
        const size_t pos = at[j] - before[bucket[j]];
        std::nth_element(f.begin(), f.begin() + (ptrdiff_t)pos, f.end());
        const uint32_t k = f[pos], u = k & 0x80000000u ? k & 0x7fffffffu : ~k;
        std::memcpy(&out[j], &u, 4);
        if (out[j] == 0.0f) {   // which of the zeros, in the order they came
            size_t below = 0, nth = 0;
            for (float v : vals) below += v < 0.0f;
            for (float v : vals)
                if (v == 0.0f && nth++ == at[j] - below) { out[j] = v; break; }
        }
    }
}

// kmeans_16 (src/packed_tensor.rs:18-75).  The assignment is independent per value; the f32 sum of a cluster must follow
// data order: the chunks are grouped by cluster side by side, then one task per cluster adds its runs chunk after chunk
// (bound by the latency of n / 16 dependent additions).
bool kmeans16(const std::vector<float> &vals, int iters, float *c)
{
    const FnnQuantKernels &kern = kernels();
    const size_t n = vals.size();
    std::fill(c, c + 16, 0.0f);
    if (n == 0) return true;
    if (n == 1) { std::fill(c, c + 16, vals[0]); return true; }
    for (float v : vals) if (std::isnan(v)) return false;  // the reference panics on NaN
    {
        size_t at[16];
        for (int i = 0; i < 16; i++) {
            const float pct = ((float)i + 0.5f) / 16.0f;
            at[i] = std::min((size_t)(pct * (float)n), n - 1);
        }
        order_statistics(vals, at, c);
    }
    const int threads = threads_for((int64_t)n);
    const int64_t chunks = ((int64_t)n + kChunk - 1) / kChunk;
    std::vector<uint8_t> assign(n);
    std::vector<float> grouped(n);
    std::vector<int32_t> start((size_t)chunks * 17);
    for (int it = 0; it < iters; it++) {
        float cc[16];
        std::memcpy(cc, c, sizeof(cc));
        fnn_parallel(chunks, threads, [&](int64_t t) {
            const int64_t i0 = t * kChunk;
            kern.group16(vals.data() + i0, std::min(kChunk, (int64_t)n - i0), cc, assign.data() + i0, grouped.data() + i0, &start[(size_t)t * 17]);
        });
        fnn_parallel(16, threads, [&](int64_t k) {
            float sum = 0.0f;
            size_t count = 0;
            for (int64_t t = 0; t < chunks; t++) {
                const int32_t s0 = start[(size_t)(t * 17 + k)], s1 = start[(size_t)(t * 17 + k + 1)];
                const float *g = grouped.data() + t * kChunk;
                for (int32_t i = s0; i < s1; i++) sum += g[i];
                count += (size_t)(s1 - s0);
            }
            if (count > 0) c[k] = sum / (float)count;
        });
    }
    std::stable_sort(c, c + 16, [](float a, float b) { return a < b; });
    return true;
}

// from_f32_per_block_codebook (src/packed_tensor.rs:1209-1313)
int quant_codebook(const float *w, int64_t rows, int64_t inner, int64_t qb, uint32_t *words, float *bscales, float *cb)
{
    const FnnQuantKernels &kern = kernels();
    const int64_t bpr = (inner + qb - 1) / qb, kp = (inner + 7) / 8;
    const int threads = threads_for(rows * inner);
    std::vector<float> norm((size_t)(rows * inner));
    fnn_parallel(rows, threads, [&](int64_t r) {
        for (int64_t b = 0; b < bpr; b++) {
            const int64_t base = r * inner + b * qb, end = std::min(base + qb, (r + 1) * inner);
            float mx = 0.0f;
            for (int64_t i = base; i < end; i++) mx = std::fmax(mx, std::fabs(w[i]));
            bscales[r * bpr + b] = mx;
            if (mx > 0.0f) {
                const float inv = 1.0f / mx;
                for (int64_t i = base; i < end; i++) norm[(size_t)i] = w[i] * inv;
            } else {
                for (int64_t i = base; i < end; i++) norm[(size_t)i] = 0.0f;
            }
        }
    });
    // block order of the reference's normalised list == element order (blocks tile each row)
    if (!kmeans16(norm, 30, cb)) return FNN_ERR_COMPILATION;
    std::vector<uint8_t> index((size_t)(rows * inner));
    fnn_parallel(rows, threads, [&](int64_t r) {
        for (int64_t b = 0; b < bpr; b++) {
            const float s = bscales[r * bpr + b];
            const float inv = s > 0.0f ? 1.0f / s : 0.0f;
            const int64_t base = r * inner + b * qb, end = std::min(base + qb, (r + 1) * inner);
            for (int64_t i = base; i < end; i++) norm[(size_t)i] = w[i] * inv;
        }
        kern.nearest16(norm.data() + r * inner, inner, cb, index.data() + r * inner);
        for (int64_t b = 0; b < bpr; b++) {
            const int64_t base = r * inner + b * qb, end = std::min(base + qb, (r + 1) * inner);
            for (int64_t eb = 0; eb < end - base; eb += 8) {
                uint32_t word = 0;
                for (int i = 0; i < 8; i++) {
                    const int64_t e = base + eb + i;
                    if (e < end) word |= (uint32_t)index[(size_t)e] << (4 * i);
                }
                words[r * kp + (b * qb + eb) / 8] = word;  // a straddling word keeps the later block's value
            }
        }
    });
    return FNN_OK;
}

int quantize(int dtype, const float *w, int64_t rows, int64_t inner, bool kn, int qblock, uint32_t *words, float *scales,
             float *zeros, float *codebook16)
{
    const int items = lanes_of(dtype);
    if (!items || !w || !words || !scales || rows <= 0 || inner <= 0) return FNN_ERR_COMPILATION;
    if (dtype != FNN_DT_I4CB) {
        if (!zeros) return FNN_ERR_COMPILATION;
        std::memset(words + rows * ((inner + items - 1) / items), 0, kMargin * sizeof(uint32_t));
        return quant_per_channel(dtype, w, rows, inner, kn, words, scales, zeros) ? FNN_OK : FNN_ERR_MEMORY;
    }
    if (qblock <= 0 || !codebook16) return FNN_ERR_COMPILATION;
    try {
        std::memset(words, 0, fnn_packed_words(dtype, rows, inner) * sizeof(uint32_t));   // (short blocks leave words out)
        if (!kn) return quant_codebook(w, rows, inner, qblock, words, scales, codebook16);
        std::unique_ptr<float[]> t(new float[(size_t)(rows * inner)]);
        fnn_transpose_kn_to_nk(w, inner, rows, t.get());
        return quant_codebook(t.get(), rows, inner, qblock, words, scales, codebook16);
    } catch (const std::bad_alloc &) {
        return FNN_ERR_MEMORY;
    }
}

}  // namespace

extern "C" {

size_t fnn_packed_words(int dtype, int64_t rows, int64_t inner)
{
    const int items = lanes_of(dtype);
    if (!items || rows < 0 || inner < 0) return 0;
    return (size_t)(rows * ((inner + items - 1) / items)) + kMargin;
}

void fnn_transpose_kn_to_nk(const float *w_kn, int64_t k, int64_t n, float *w_nk)
{
    constexpr int64_t T = 32;
    fnn_parallel((n + T - 1) / T, threads_for(k * n), [&](int64_t t) {
        const int64_t n0 = t * T, n1 = std::min(n, n0 + T);
        for (int64_t k0 = 0; k0 < k; k0 += T)
            for (int64_t nn = n0; nn < n1; nn++)
                for (int64_t kk = k0; kk < std::min(k, k0 + T); kk++) w_nk[nn * k + kk] = w_kn[kk * n + nn];
    });
}

int fnn_quantize_weights(int dtype, const float *w, int64_t rows, int64_t inner, int qblock,
                         uint32_t *words, float *scales, float *zeros, float *codebook16)
{
    return quantize(dtype, w, rows, inner, false, qblock, words, scales, zeros, codebook16);
}

int fnn_quantize_weights_kn(int dtype, const float *w_kn, int64_t k, int64_t n, int qblock,
                            uint32_t *words, float *scales, float *zeros, float *codebook16)
{
    return quantize(dtype, w_kn, n, k, true, qblock, words, scales, zeros, codebook16);
}

}  // extern "C"
