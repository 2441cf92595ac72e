// Body of quantize_simd_*.cpp.  Only compiler vector extensions and local functions here: nothing from a header may be
// emitted in a unit compiled for a newer instruction set than the rest of the library.
//
// Each lane does what the scalar packer of the reference does for one channel, in the same order and in binary32
// (FMA contraction is off), so words, scales and zeros are bit-identical to it.  What bounds it: the two passes over the
// floats (16 threads read 180 MB of a 4096 x 11008 weight at the host's memory rate, the second pass comes from the
// core's own cache: a panel of 32 channels is 0.5 MB), about 20 vector instructions per 32 values beside them.
#include "quantize_simd.h"

#include "../../include/fastnn_hip.h"

namespace {

constexpr int L = 16;                                   // lanes of one vector
typedef float vf __attribute__((vector_size(64)));
typedef int32_t vi __attribute__((vector_size(64)));
typedef uint32_t vu __attribute__((vector_size(64)));

inline vf splat(float x) { return vf{} + x; }
inline vf load(const float *p) { vf v; __builtin_memcpy(&v, p, sizeof v); return v; }
inline vf vabs(vf x) { return (vf)((vi)x & 0x7fffffff); }
inline vf vmin(vf m, vf x) { return x < m ? x : m; }     // (a NaN x leaves m, as fmin does)
inline vf vmax(vf m, vf x) { return x > m ? x : m; }
// round half away from zero for |x| < 2^22: x + 0.49999997 (the largest float below one half) truncated
inline vi round_away(vf x)
{
    const vf half = (vf)((vi)splat(0.49999997f) | ((vi)x & (int32_t)0x80000000));
    return __builtin_convertvector(x + half, vi);
}

// ---- lane encoders: the code of each value, in the low bits
template <int LO, int HI, int BITS>
struct EncInt {   // clamp (NaN stays), round, `as iN` (NaN becomes 0)
    static constexpr int kBits = BITS;
    static inline vu enc(vf x)
    {
        const vi nan = x != x;
        x = x < splat((float)LO) ? splat((float)LO) : (x > splat((float)HI) ? splat((float)HI) : x);
        x = (vf)((vi)x & ~nan);
        return (vu)round_away(x) & ((1u << BITS) - 1u);
    }
};

// E4M3 / E5M2 with the mantissa rounded half away from zero: rounding the bit pattern at the mantissa's last kept bit is
// the same, and its carry is the reference's step to the next exponent
template <int MBITS, int BIAS, int EMAX, bool INF>
struct EncMini {
    static constexpr int kBits = 8;
    static inline vu enc(vf x, float max_val, float sub_limit, float sub_mul, uint32_t max_code)
    {
        const vu sign = ((vu)x >> 24) & 0x80u;
        const vi nan = x != x;
        const vf a0 = vabs(x);
        const vf a = a0 > splat(max_val) ? splat(max_val) : a0;
        const vu r = (vu)a + (1u << (22 - MBITS));
        vu norm = (r >> (23 - MBITS)) - ((127u - BIAS) << MBITS);
        norm = (vi)norm >= (vi)(vu{} + (uint32_t)(EMAX << MBITS)) ? vu{} + max_code : norm;
        vf small = a * splat(sub_mul);
        small = small > splat(255.0f) ? splat(255.0f) : small;
        vi m = round_away((vf)((vi)small & ~nan));
        m = m > (1 << MBITS) ? vi{} + (1 << MBITS) : m;
        vu code = a < splat(sub_limit) ? (vu)m : norm;
        if (INF) code = a0 > splat(3.40282347e+38f) ? vu{} + 0x7Cu : code;
        code |= sign;
        return nan ? vu{} + 0x7Fu : code;
    }
};
struct EncF8 {
    static constexpr int kBits = 8;
    static inline vu enc(vf x) { return EncMini<3, 7, 15, false>::enc(x, 240.0f, 0.015625f, 512.0f, 0x7Bu); }
};
struct EncF8R {
    static constexpr int kBits = 8;
    static inline vu enc(vf x) { return EncMini<2, 15, 31, true>::enc(x, 57344.0f, 1.0f / 16384.0f, 16384.0f, 0x7Cu); }
};

struct EncF4 {   // nearest of the eight magnitudes, the lower one where two are as near
    static constexpr int kBits = 4;
    static inline vu enc(vf x)
    {
        const float mag[8] = {0.0f, 0.5f, 1.0f, 1.5f, 2.0f, 3.0f, 4.0f, 6.0f};
        const vf a = vabs(x);
        vf best_d = a;
        vu best{};
        for (uint32_t i = 1; i < 8; i++) {
            const vf d = vabs(a - splat(mag[i]));
            const vi nearer = d < best_d;
            best_d = nearer ? d : best_d;
            best = nearer ? vu{} + i : best;
        }
        const vu sign = ((vu)x >> 28) & 8u;
        return best | (best != 0u ? sign : vu{});   // (NaN: no distance is smaller than NaN, the code is 0)
    }
};

struct AsymInt {};   // scale = (range + 2 range / umax) / umax, zero in the middle
struct AsymF4 {};    // zero = mean, scale = largest deviation / 4
struct Sym {};       // scale = max|x| / max_val

template <class Enc, class Form>
void panel(const float *src, int64_t ld, int64_t inner, int rows, uint32_t *words, int64_t kp, float *scales, float *zeros, float max_val)
{
    constexpr int items = 32 / Enc::kBits;
    constexpr bool kSym = __is_same(Form, Sym), kF4 = __is_same(Form, AsymF4);
    vf mn0 = splat(3.40282347e+38f), mn1 = mn0, mx0 = splat(kSym ? 0.0f : -3.40282347e+38f), mx1 = mx0, sum0{}, sum1{};
    for (int64_t k = 0; k < inner; k++) {
        __builtin_prefetch(src + (k + 24) * ld);           // (a [K, N] matrix: every step is on another page)
        __builtin_prefetch(src + (k + 24) * ld + L);
        const vf a = load(src + k * ld), b = load(src + k * ld + L);
        if (kSym) {
            mx0 = vmax(mx0, vabs(a)); mx1 = vmax(mx1, vabs(b));
        } else {
            mn0 = vmin(mn0, a); mn1 = vmin(mn1, b);
            mx0 = vmax(mx0, a); mx1 = vmax(mx1, b);
            if (kF4) { sum0 += a; sum1 += b; }
        }
    }
    float mn[32], mx[32], sum[32], sub[32], mul[32];
    __builtin_memcpy(mn, &mn0, 64); __builtin_memcpy(mn + L, &mn1, 64);
    __builtin_memcpy(mx, &mx0, 64); __builtin_memcpy(mx + L, &mx1, 64);
    __builtin_memcpy(sum, &sum0, 64); __builtin_memcpy(sum + L, &sum1, 64);
    const float umax = (float)((1u << Enc::kBits) - 1u), sbias = (float)(1u << (Enc::kBits - 1));
    for (int l = 0; l < 32; l++) {
        float scale, zero = 0.0f;
        if (kSym) {
            scale = mx[l] == 0.0f ? 1.0f : mx[l] / max_val;
            mul[l] = scale != 1.0f ? 1.0f / scale : 1.0f;
        } else {
            const float range = mx[l] - mn[l];
            if (range == 0.0f) {
                scale = 1.0f;
            } else if (kF4) {
                const float mean = sum[l] / (float)inner;
                const float d0 = __builtin_fabsf(mean - mn[l]), d1 = __builtin_fabsf(mx[l] - mean);
                const float dev = d0 != d0 ? d1 : (d1 > d0 ? d1 : d0);
                scale = (dev == 0.0f ? 1e-10f : dev) / 4.0f;
                zero = mean;
            } else {
                const float init = range / umax, lo = mn[l] - init, hi = mx[l] + init;
                scale = (hi - lo) / umax;
                zero = lo + sbias * scale;
            }
            mul[l] = scale != 0.0f ? 1.0f / scale : 0.0f;
        }
        sub[l] = zero;
        if (l < rows) { scales[l] = scale; zeros[l] = zero; }
    }
    const vf s0 = load(sub), s1 = load(sub + L), m0 = load(mul), m1 = load(mul + L);
    auto word = [&](int64_t w, uint32_t *to, int have) {   // `have` of the word's lanes hold values, the others encode 0.0
        vu lo{}, hi{};
        for (int i = 0; i < items; i++) {
            vf a{}, b{};
            if (i < have) {
                a = load(src + (w * items + i) * ld); b = load(src + (w * items + i) * ld + L);
                if (!kSym) { a = a - s0; b = b - s1; }
                a = a * m0; b = b * m1;
            }
            lo |= Enc::enc(a) << (Enc::kBits * i);
            hi |= Enc::enc(b) << (Enc::kBits * i);
        }
        __builtin_memcpy(to, &lo, 64);
        __builtin_memcpy(to + L, &hi, 64);
    };
    // sixteen words of all rows, then turned: a row's sixteen words are one 64-byte store
    uint32_t buf[16][32];
    for (int64_t w0 = 0; w0 < kp; w0 += 16) {
        const int nw = kp - w0 < 16 ? (int)(kp - w0) : 16;
        for (int i = 0; i < nw; i++) {
            const int64_t left = inner - (w0 + i) * items;
            if (left >= items) word(w0 + i, buf[i], items);
            else word(w0 + i, buf[i], (int)left);
        }
        for (int l = 0; l < rows; l++) {
            uint32_t *to = words + l * kp + w0;
            if (nw == 16) {
                uint32_t line[16];
                for (int i = 0; i < 16; i++) line[i] = buf[i][l];
                __builtin_memcpy(to, line, 64);
            } else {
                for (int i = 0; i < nw; i++) to[i] = buf[i][l];
            }
        }
    }
}

void quant_panel(int dtype, const float *src, int64_t ld, int64_t inner, int rows, uint32_t *words, int64_t kp, float *scales, float *zeros)
{
    switch (dtype) {
    case FNN_DT_I8: panel<EncInt<-128, 127, 8>, AsymInt>(src, ld, inner, rows, words, kp, scales, zeros, 0.0f); break;
    case FNN_DT_I4: panel<EncInt<-8, 7, 4>, AsymInt>(src, ld, inner, rows, words, kp, scales, zeros, 0.0f); break;
    case FNN_DT_U8: panel<EncInt<0, 255, 8>, AsymInt>(src, ld, inner, rows, words, kp, scales, zeros, 0.0f); break;
    case FNN_DT_U4: panel<EncInt<0, 15, 4>, AsymInt>(src, ld, inner, rows, words, kp, scales, zeros, 0.0f); break;
    case FNN_DT_F4: panel<EncF4, AsymF4>(src, ld, inner, rows, words, kp, scales, zeros, 0.0f); break;
    case FNN_DT_F8: panel<EncF8, Sym>(src, ld, inner, rows, words, kp, scales, zeros, 240.0f); break;
    case FNN_DT_F8R: panel<EncF8R, Sym>(src, ld, inner, rows, words, kp, scales, zeros, 57344.0f); break;
    default: break;
    }
}

void panel_from_rows(const float *src, int64_t inner, int rows, float *dst)
{
    for (int64_t k0 = 0; k0 < inner; k0 += 16) {
        const int nk = inner - k0 < 16 ? (int)(inner - k0) : 16;
        float t[16][32];
        for (int l = 0; l < 32; l++)
            for (int k = 0; k < nk; k++) t[k][l] = l < rows ? src[l * inner + k0 + k] : 0.0f;
        __builtin_memcpy(dst + k0 * 32, t, (size_t)nk * 128);
    }
}

void nearest16(const float *v, int64_t n, const float *table, uint8_t *index)
{
    int64_t i = 0;
    for (; i + L <= n; i += L) {
        const vf x = load(v + i);
        vf best_d = vabs(x - splat(table[0]));
        vi best{};
        for (int e = 1; e < 16; e++) {
            const vf d = vabs(x - splat(table[e]));
            const vi nearer = d < best_d;
            best_d = nearer ? d : best_d;
            best = nearer ? vi{} + e : best;
        }
        typedef uint8_t vb __attribute__((vector_size(16)));
        const vb b = __builtin_convertvector(best, vb);
        __builtin_memcpy(index + i, &b, 16);
    }
    for (; i < n; i++) {
        float best_d = __builtin_fabsf(v[i] - table[0]);
        uint8_t best = 0;
        for (uint8_t e = 1; e < 16; e++) {
            const float d = __builtin_fabsf(v[i] - table[e]);
            if (d < best_d) { best_d = d; best = e; }
        }
        index[i] = best;
    }
}

// Counting sort of a chunk by nearest entry, stable: `grouped` holds the values of entry 0, then of entry 1, ...; entry e's
// start at start[e].
void group16(const float *v, int64_t n, const float *table, uint8_t *index, float *grouped, int32_t *start)
{
    nearest16(v, n, table, index);
    int32_t at[16] = {0};
    for (int64_t i = 0; i < n; i++) at[index[i]]++;
    int32_t sum = 0;
    for (int e = 0; e < 16; e++) { start[e] = sum; sum += at[e]; at[e] = start[e]; }
    start[16] = sum;
    for (int64_t i = 0; i < n; i++) grouped[at[index[i]]++] = v[i];
}

}  // namespace

const FnnQuantKernels FNN_QUANT_TABLE = {quant_panel, nearest16, panel_from_rows, group16};
