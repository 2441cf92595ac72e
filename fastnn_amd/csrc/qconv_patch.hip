// Quantised Conv2d (I8 or I4 weights, f32 NCHW activations) from an int8 patch in LDS: conv2d_packed_i8x4 /
// conv2d_packed_i4x8 (src/backend/cpu/packed_conv.rs:125-283,444-841) in one launch.
//
// A workgroup of four waves owns a rectangle of output pixels of ONE image.  Phase 1: it loads the input patch under that
// rectangle (all channels, halo included), quantises every value once with the image's scale and leaves it in LDS, channels
// innermost: [chunk of 16 channels][patch pixel][16 bytes].  Phase 2: a tap of the kernel is then a fixed LDS offset, and the
// 16 bytes that a lane (pixel lane & 31, k half lane >> 5) reads there are the A operand of v_mfma_i32_32x32x32_i8 as they
// are, for k in the order (chunk of 16 channels, kernel row, kernel column, channel).  The weights are kept in that order, one KB per
// block of 32 channels and step (conv_words_kernel, built with the row sums on a weight's first call).  The waves share pixel blocks,
// channel blocks and, where there is little work, the K range; K parts meet in LDS and then share the epilogue.
//
// Where patch and weights of all channels do not fit LDS, or leave room for one small rectangle only, the channels come in segments: both
// phases for one segment after the other, the sums stay in registers, and the next segment's weights arrive in a second
// buffer during phase 2.  Against the operand kernel + GEMM pair, which has to run such layers else (and a kernel that fetched im2col taps at
// any K): 8 x 320 x 160 x 160 -> 24 channels 5x5 1427 (721) -> 214 us with the range scan, 512 x 80 x 80 -> 32 3x3 47.6 (45.5) -> 27.2, 16 x
// 512 x 40 x 40 -> 64 3x3 101 (101) -> 61.
//
// Under many output channels every workgroup of a few blocks quantises the same pixels again.  There a wave works on several blocks, one after
// the other on the one patch, and fetches their weights itself, four steps ahead (from L2; no wave shares them, so LDS would only cost
// room): no barrier behind the patch's.  Against the pair (and a kernel with pixels in LDS and im2col taps): 16 x 512 x 28 x 28 -> 1024 1x1
// 71 (55) -> 39 us, 512 x 320 x 320 -> 192 1x1 176 (124) -> 98, 256 x 208 x 208 -> 384 3x3 179 (166) -> 144.
//
// What bounded the kernels that fetched im2col taps was vector instructions and their chain: a 3 x 3 layer fetched and quantised every
// input value nine times, about 11 instructions a tap; here it is about 1.4 times (18 x 10 pixels under 16 x 8) and the tap arithmetic
// is gone.  One image: 64 -> 64 channels 3x3 at 40 x 40 10.5 -> 6.6 us (before: operand kernel + GEMM), 128 -> 128 3x3 at 20 x 20 12.0 -> 7.2,
// 512 -> 256 1x1 at 20 x 20 10.4 -> 7.0, 16 -> 32 3x3 stride 2 at 320 x 320 9.6 -> 7.8; what is left of these is the floor of a dependent launch
// (2.3) and a chain of memory, LDS and barrier latencies.  Sixteen images: 16 -> 16 3x3 at 160 x 160 34 -> 23.5 us, 3 -> 16 3x3 stride 2 at
// 640 x 640 63 -> 52 (184 MB), 64 -> 64 1x1 at 80 x 80 17.1 -> 16.1 (52 MB: 3.2 TB/s; loads in flight).  Two blocks of 32 channels a wave (one A
// operand for two products) measured slower at every size: 130 registers, three waves a SIMD, against 107 and four.
#include "mfma.h"
#include "range_io.h"

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

namespace {

struct PatchArgs {
    // of one group of the convolution
    const float *x;           // its first channel in image 0
    const int8_t *cw;         // weights in operand order: [block of 32 channels][step][64 lanes][16 bytes]
    const float *scales, *zeros, *bias;
    const int32_t *qsum;
    const float *actq, *pairs;   // ready-made scales, or npairs partial ranges per image
    float *y, *sum_out, *range_out;
    const float *residual;
    int32_t *acc_out;
    int64_t x_image, y_image;    // values of an image (all groups)
    int npairs, pair_stride, actq_stride, range_zero, range_stride;
    int cg, ocg, act, wbits, vec4;
    float kk;
    int hh, ww, ho, wo;       // geometry of a plane (1x1 without padding or stride: one row of all pixels)
    int kw, stride, pad, dil;
    int twl, th;              // rectangle: 1 << twl wide, th high
    int tiles, per, parts;    // rectangles of an image, of a workgroup, workgroups of an image
    int pw, pp, pgroups;      // patch width, pixels, groups of 64 pixels
    int split;                // patches of up to 32 pixels: the two halves of a wave take a chunk each
    int nch;                  // chunks of 16 channels (up to 4 channels: one chunk = 4 pixels of 4 channels)
    int nsteps, nkc;          // K steps of two chunks of K, chunks of K
    int lnw, lwch, lwks;      // log2 of the waves, of those over channels, over K
    int w_at, tab_at, red_at; // LDS offsets behind the patch
    FastDiv dpw, dpg, dparts, dtx, dper, dkw;   // (dper: taps, or chunks per kernel row of up to 4 channels)
    // segments of the channels that follow each other in LDS, chunks and steps of a whole one (last: the other forms do not load them)
    int segs, cs, nss;
    FastDiv dnss;
    int sets;   // blocks of output channels of a wave
};

// 64 lanes' 16 bytes each from memory into LDS, without registers: lane i's land at lds + 16 i.  The compiler does not see these loads.
__device__ __forceinline__ void load_kb(const void *gptr, unsigned lds_wave_base)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds_wave_base), "v"(gptr) : "memory");
}

__device__ __forceinline__ float row16_min(float v)
{
    v = fminf(v, dpp_f32<0xB1>(v));
    v = fminf(v, dpp_f32<0x4E>(v));
    v = fminf(v, dpp_f32<0x141>(v));
    return fminf(v, dpp_f32<0x140>(v));
}
__device__ __forceinline__ float row16_max(float v)
{
    v = fmaxf(v, dpp_f32<0xB1>(v));
    v = fmaxf(v, dpp_f32<0x4E>(v));
    v = fmaxf(v, dpp_f32<0x141>(v));
    return fmaxf(v, dpp_f32<0x140>(v));
}

constexpr uint32_t NOWHERE = 0x80000000u;   // a buffer offset past every slab (slabs are below 2 GiB)
constexpr int MAX_WAVES = 8;
constexpr int MAX_LDS = 152 * 1024;   // beside the static part

// C4: up to four channels in a group.  KS: the K range is shared by 1 << lwks waves.  SEGMENTS: the channels come in segments.  SETS: a wave
// works on several blocks of output channels, one after the other, and fetches their weights itself.
enum Form { WHOLE, SEGMENTS, SETS };
template <bool KS, bool C4, Form FORM>
__global__ void __launch_bounds__(64 * MAX_WAVES, 4) conv_patch_kernel(PatchArgs p)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    __shared__ float s_mm[2][MAX_WAVES], s_rng[MAX_WAVES][2];
    __shared__ __attribute__((aligned(16))) int s_qs[MAX_WAVES][32];
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 31, hf = lane >> 5;
    const int nw = 1 << p.lnw, lwks = KS ? p.lwks : 0, wks = 1 << lwks, wch = 1 << p.lwch;
    const int kw_ = wv & (wks - 1), cw_ = (wv >> lwks) & (wch - 1), px_ = wv >> (lwks + p.lwch);   // this wave's share of K, channels, pixels

    const int nn = __builtin_amdgcn_readfirstlane((int)p.dparts.div(blockIdx.x)), part = (int)blockIdx.x - nn * p.parts;
    const int t0 = part * p.per, t1 = min(t0 + p.per, p.tiles);
    const int chstep = p.hh * p.ww * 4;
    const __amdgpu_buffer_rsrc_t xbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p.x + nn * p.x_image), 0, p.cg * chstep, 0x00020000);

    // ---- loads of phase 1: a unit is 64 patch pixels of one chunk (or 32 of two); a channel's plane is a scalar offset, so
    // that only the pixel costs address arithmetic, once for 16 loads
    constexpr bool SEG = FORM == SEGMENTS, MANY = FORM == SETS;
    const int segs = SEG ? p.segs : 1, nss = SEG ? p.nss : p.nsteps;
    auto chunks_of = [&](int sg) { return SEG ? min(p.cs, p.nch - sg * p.cs) : p.nch; };
    auto units_of = [&](int sg) { return C4 ? p.pgroups : (p.split ? (chunks_of(sg) + 1) >> 1 : p.pgroups * chunks_of(sg)); };
    auto unit_at = [&](int u, int &chunk, int &pix) {   // (chunk: of the segment; uniform but for split patches)
        if (!C4 && p.split) {
            chunk = 2 * u + hf;
            pix = lr;
        } else {
            chunk = C4 ? 0 : __builtin_amdgcn_readfirstlane((int)p.dpg.div((uint32_t)u));
            pix = (u - chunk * p.pgroups) * 64 + lane;
        }
    };
    auto fetch = [&](int u, int t, int sg, float(&v)[16]) {
        const int ty = __builtin_amdgcn_readfirstlane((int)p.dtx.div((uint32_t)t)), tx = t - ty * (int)p.dtx.d;
        const int iy0 = ty * p.th * p.stride - p.pad, ix0 = (tx << p.twl) * p.stride - p.pad;
        int chunk, pix;
        unit_at(u, chunk, pix);
        const int py = (int)p.dpw.div((uint32_t)pix), iy = iy0 + py, ix = ix0 + pix - py * p.pw;
        bool ok = pix < p.pp && (unsigned)iy < (unsigned)p.hh && (unsigned)ix < (unsigned)p.ww;
        uint32_t vo = (uint32_t)(iy * p.ww + ix) * 4u;
        int chunk0 = 0, wide = 16;   // (uniform) the unit's first chunk, channels from there on that it may touch
        if (!C4) {
            chunk0 = p.split ? 2 * u : __builtin_amdgcn_readfirstlane(chunk);
            if (p.split) {
                ok = ok && chunk < chunks_of(sg);
                vo += hf ? (uint32_t)(16 * chstep) : 0u;
                wide = 32;
            }
        }
        if constexpr (SEG) {
            chunk0 += sg * p.cs;
            chunk += sg * p.cs;
        }
        vo = ok ? vo : NOWHERE;   // outside the image: zero by the range check
        int so = chunk0 * 16 * chstep;
        if (!C4 && chunk0 * 16 + wide <= p.cg) {
#pragma unroll
            for (int c = 0; c < 16; c++, so += chstep) v[c] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xbuf, vo, so, 0));
        } else {
            const int left = p.cg - chunk * 16, left0 = p.cg - chunk0 * 16;
#pragma unroll
            for (int c = 0; c < (C4 ? 4 : 16); c++, so += chstep)
                v[c] = c < left0 ? __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xbuf, c < left ? vo : NOWHERE, so, 0)) : 0.0f;
        }
    };
    float v0[16], v1[16];
    if (wv < units_of(0)) fetch(wv, t0, 0, v0);

    // ---- this lane's channel: a wave works on one block of 32
    const bool share = !KS && !MANY && p.ocg <= 16;   // (uniform) up to 16 channels: the lanes of channels 16 .. 31 take half of
    int blk = (int)blockIdx.y * wch * (MANY ? p.sets : 1) + cw_, n, qw;   // the pixels of the lane 16 below in the epilogue
    float sw, zw, bi;
    auto channel = [&]() {
        n = blk * 32 + (share ? (lr & 15) : lr);
        const int ch = n < p.ocg ? n : 0;
        sw = p.scales[ch]; zw = p.zeros[ch]; bi = p.bias ? p.bias[ch] : 0.0f;
        qw = p.qsum[ch];
    };
    channel();

    // ---- LDS offset of every chunk of K of a segment, relative to a pixel's first tap; bits 24 up: how many of its four words
    // count (of the segments', the last step of the last one may hold half a step)
    uint32_t *tab = reinterpret_cast<uint32_t *>(lds + p.tab_at);   // [2 halves][nss]
    for (int kc = tid; kc < 2 * nss; kc += nw * 64) {
        uint32_t e = 0;
        if (SEG || kc < p.nkc) {   // (a segment is whole steps)
            const int q = (int)p.dper.div((uint32_t)kc), r = kc - q * (int)p.dper.d;
            if (C4) {
                e = (uint32_t)((q * p.pw + r * 4) * p.dil * 4) | ((uint32_t)min(4, p.kw - r * 4) << 24);
            } else {
                const int i = (int)p.dkw.div((uint32_t)r), j = r - i * p.kw;
                e = (uint32_t)((q * p.pp + (i * p.pw + j) * p.dil) * 16) | (4u << 24);
            }
        }
        tab[(kc & 1) * nss + (kc >> 1)] = e;
    }

    // ---- the workgroup's weights on their way into LDS, where every rectangle and every wave finds them: all of them once, or a segment's
    // into one of two buffers while the segment before it is multiplied
    const int wbytes = (nss << p.lwch) * 1024;
    auto weights = [&](int sg, int buf) {
        const unsigned base = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(__attribute__((address_space(3))) unsigned char *)lds + p.w_at + buf * wbytes);
        const char *src = reinterpret_cast<const char *>(p.cw) + ((int64_t)blockIdx.y * (p.nsteps << p.lwch) + sg * nss) * 1024 + lane * 16;
        const int kbs = min(wch, ((p.ocg + 31) >> 5) - (int)blockIdx.y * wch) * nss;   // (of blocks that exist: what the others multiply is not stored)
        for (int i = wv; i < kbs; i += nw) {
            int from = i;
            if constexpr (SEG) {   // (a block's segments follow each other)
                const int blk = __builtin_amdgcn_readfirstlane((int)p.dnss.div((uint32_t)i)), s = i - blk * nss;
                if (sg * nss + s >= p.nsteps) continue;
                from = blk * p.nsteps + s;
            }
            load_kb(src + (int64_t)from * 1024, base + i * 1024);
        }
    };

    // ---- activation scale of the image: from partial ranges, or ready-made
    float sa, za, inv;
    if constexpr (!MANY) weights(0, 0);
    if (p.npairs > 0) {
        float mn = p.range_zero ? 0.0f : INFINITY, mx = p.range_zero ? 0.0f : -INFINITY;
        conv_fold_partial_ranges(p.pairs + (int64_t)nn * p.pair_stride * 2, p.npairs, tid, nw * 64, mn, mx);
        mn = wave_min(mn);
        mx = wave_max(mx);
        if (lane == 0) { s_mm[0][wv] = mn; s_mm[1][wv] = mx; }
        __syncthreads();
        // (every wave by itself: one lane a wave's pair)
        mn = row16_min(s_mm[0][lane & (nw - 1)]);
        mx = row16_max(s_mm[1][lane & (nw - 1)]);
        const float range = mx - mn;
        if (p.wbits == 4) {
            sa = (range > 0.0f) ? range / 15.0f : 1.0f;
            za = mn + 8.0f * sa;
        } else {
            sa = (range > 0.0f) ? range / 255.0f : 1.0f;
            za = (range > 0.0f) ? mn + 128.0f * sa : 0.0f;
        }
        inv = (sa != 0.0f) ? 1.0f / sa : 0.0f;
    } else {
        const float *q = p.actq + (int64_t)nn * p.actq_stride;
        sa = q[0]; za = q[1]; inv = q[2];
    }
    float wt;
    int bq;
    auto channel_terms = [&]() {
        wt = sw * (float)qw;
        bq = p.bias ? conv_bias_q(bi, sa, sw) : 0;
    };
    channel_terms();

    const int qlo = p.wbits == 4 ? -8 : -128, qhi = p.wbits == 4 ? 7 : 127;
    auto quantise = [&](int u, int sg, const float(&v)[16]) {
        int chunk, pix;
        unit_at(u, chunk, pix);
        uint32_t w[4];
#pragma unroll
        for (int i = 0; i < (C4 ? 1 : 4); i++) {
            int q[4];
#pragma unroll
            for (int t = 0; t < 4; t++) {
                // round half away from zero, then clamp: trunc(x + copysign(0.49999997, x)) equals roundf(x) after the
                // clamp for every float (the conversion truncates, saturates and maps NaN to 0)
                const float x = (v[i * 4 + t] - za) * inv;
                q[t] = max(qlo, min((int)(x + __builtin_copysignf(0.49999997f, x)), qhi));
            }
            w[i] = __builtin_amdgcn_perm((uint32_t)q[1], (uint32_t)q[0], 0x0c0c0400u) | __builtin_amdgcn_perm((uint32_t)q[3], (uint32_t)q[2], 0x04000c0cu);
        }
        if (C4 || (p.cg & 15)) {   // bytes of channels that do not exist are zero
            const int left = p.cg - ((SEG ? sg * p.cs : 0) + chunk) * 16;
#pragma unroll
            for (int i = 0; i < (C4 ? 1 : 4); i++)
                if (left < i * 4 + 4) w[i] = left <= i * 4 ? 0u : w[i] & (0xffffffffu >> (8 * (i * 4 + 4 - left)));
        }
        if (pix >= p.pp || (!C4 && p.split && chunk >= chunks_of(sg))) return;
        if (C4) reinterpret_cast<uint32_t *>(lds)[pix] = w[0];
        else reinterpret_cast<u32x4 *>(lds)[chunk * p.pp + pix] = u32x4{w[0], w[1], w[2], w[3]};
    };

    const int np = p.ho * p.wo, tw1 = (1 << p.twl) - 1;
    const int pl = px_ * 32 + lr;
    const unsigned char *a_lds = lds + ((pl >> p.twl) * p.pw + (pl & tw1)) * p.stride * (C4 ? 4 : 16);
    const unsigned char *w_lds = lds + p.w_at + cw_ * nss * 1024 + lane * 16;
    const int tail = (p.nkc & 1) && hf ? 0 : 0x01010101;   // (an odd number of chunks of K: the last step's second half is no chunk)
    int *red = reinterpret_cast<int *>(lds + p.red_at);
    float mn = INFINITY, mx = -INFINITY;

    int oy0, ox0;   // the rectangle's first pixel
    auto rectangle = [&](int t) {
        const int ty = __builtin_amdgcn_readfirstlane((int)p.dtx.div((uint32_t)t));
        oy0 = ty * p.th;
        ox0 = (t - ty * (int)p.dtx.d) << p.twl;
    };
    // pixels 8 ig + 4 hf + (0 .. 3) of the block: scale times the sum of their codes, place in a plane (false: outside)
    auto pixels = [&](int ig, float(&rs)[4], int &at, int &ow) {
        const int pq = ig * 8 + hf * 4, pt = px_ * 32 + pq, oh = oy0 + (pt >> p.twl);
        ow = ox0 + (pt & tw1);
        at = oh * p.wo + ow;
        i32x4 q4 = *reinterpret_cast<const i32x4 *>(&s_qs[wv - kw_][pq]);
        if constexpr (KS)
            for (int k2 = 1; k2 < wks; k2++) {
                const i32x4 o4 = *reinterpret_cast<const i32x4 *>(&s_qs[wv - kw_ + k2][pq]);
#pragma unroll
                for (int j = 0; j < 4; j++) q4[j] += o4[j];
            }
#pragma unroll
        for (int j = 0; j < 4; j++) rs[j] = sa * (float)q4[j];
        return oh < p.ho && ow < p.wo;
    };
    auto finish = [&](const i32x4 &a4, const float(&rs)[4], int at, int ow) {
        if (n >= p.ocg) return;
        float v[4];
        int av[4];
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = conv_affine(a4[j], sa, za, rs[j], sw, zw, wt, bq, p.kk, &av[j]);
        conv_act4(v, p.act);
        const int64_t o = nn * p.y_image + (uint32_t)(n * np + at);
        // a residual: the Add behind this convolution; v becomes the sums, whose ranges travel on instead of y's
        if (p.vec4) {
            *reinterpret_cast<float4 *>(p.y + o) = make_float4(v[0], v[1], v[2], v[3]);
            if (p.acc_out) *reinterpret_cast<int4 *>(p.acc_out + o) = make_int4(av[0], av[1], av[2], av[3]);
            if (p.residual) {
                const float4 r4 = *reinterpret_cast<const float4 *>(p.residual + o);
                v[0] = v[0] + r4.x; v[1] = v[1] + r4.y; v[2] = v[2] + r4.z; v[3] = v[3] + r4.w;
                *reinterpret_cast<float4 *>(p.sum_out + o) = make_float4(v[0], v[1], v[2], v[3]);
            }
            mn = fminf(fminf(mn, fminf(v[0], v[1])), fminf(v[2], v[3]));
            mx = fmaxf(fmaxf(mx, fmaxf(v[0], v[1])), fmaxf(v[2], v[3]));
        } else {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                if (ow + j >= p.wo) continue;
                p.y[o + j] = v[j];
                if (p.acc_out) p.acc_out[o + j] = av[j];
                if (p.residual) {
                    v[j] = v[j] + p.residual[o + j];
                    p.sum_out[o + j] = v[j];
                }
                mn = fminf(mn, v[j]);
                mx = fmaxf(mx, v[j]);
            }
        }
    };

    if constexpr (MANY) {
        const int all = (p.ocg + 31) >> 5, units = units_of(0);
        const char *w0 = reinterpret_cast<const char *>(p.cw) + lane * 16;
        auto weights_of = [&](int b, int s, i32x4(&w)[4]) {
#pragma unroll
            for (int i = 0; i < 4; i++) w[i] = *reinterpret_cast<const i32x4 *>(w0 + ((int64_t)b * p.nsteps + min(s + i, p.nsteps - 1)) * 1024);
        };
        i32x4 w[4], wn[4];
        if (blk < all) weights_of(blk, 0, w);
        for (int u = wv; u < units; u += 2 * nw) {
            if (u + nw < units) fetch(u + nw, t0, 0, v1);
            quantise(u, 0, v0);
            if (u + nw < units) {
                if (u + 2 * nw < units) fetch(u + 2 * nw, t0, 0, v0);
                quantise(u + nw, 0, v1);
            }
        }
        rectangle(t0);
        __syncthreads();
        // from here on a wave is on its own
        int qs = 0;
        for (int set = 0; set < p.sets && blk < all; set++, blk += wch) {
            i32x16 acc;
#pragma unroll
            for (int i = 0; i < 16; i++) acc[i] = 0;
            if (set > 0) channel();
            for (int s = 0; s < p.nsteps; s += 4) {
                const bool more = s + 4 < p.nsteps;   // (uniform)
                weights_of(more || blk + wch >= all ? blk : blk + wch, more ? s + 4 : 0, wn);
                uint32_t e[4];
                i32x4 af[4];
#pragma unroll
                for (int i = 0; i < 4; i++) e[i] = tab[hf * nss + min(s + i, p.nsteps - 1)];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const unsigned char *at = a_lds + (e[i] & 0xffffffu);
                    if constexpr (C4) {
#pragma unroll
                        for (int q = 0; q < 4; q++) af[i][q] = *reinterpret_cast<const int *>(at + q * p.dil * 4);
                    } else {
                        af[i] = *reinterpret_cast<const i32x4 *>(at);
                    }
                }
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    if (s + i >= p.nsteps) break;   // (uniform)
                    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[i], w[i], acc, 0, 0, 0);
                }
                if (set == 0) {
#pragma unroll
                    for (int i = 0; i < 4; i++)
#pragma unroll
                        for (int q = 0; q < 4; q++) {
                            const bool counts = s + i < p.nsteps && (C4 ? q < (int)(e[i] >> 24) : (e[i] >> 24) != 0);
                            qs = __builtin_amdgcn_sdot4(af[i][q], counts ? 0x01010101 : 0, qs, false);
                        }
                }
#pragma unroll
                for (int i = 0; i < 4; i++) w[i] = wn[i];
            }
            if (set == 0) {
                qs += __shfl_xor(qs, 32, 64);
                if (hf == 0) s_qs[wv][lr] = qs;
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            } else {
                channel_terms();
            }
            float rs[4];
            int at, ow;
#pragma unroll
            for (int t4 = 0; t4 < 4; t4++)
                if (pixels(t4, rs, at, ow)) finish(i32x4{acc[t4 * 4], acc[t4 * 4 + 1], acc[t4 * 4 + 2], acc[t4 * 4 + 3]}, rs, at, ow);
            if (p.range_out) {   // one pair per wave and block
                mn = wave_min(mn);
                mx = wave_max(mx);
                if (lane == 0) {
                    const int wpx = nw >> p.lwch;
                    float *dst = p.range_out + ((int64_t)nn * p.range_stride + (int64_t)blk * p.parts * wpx + part * wpx + px_) * 2;
                    dst[0] = mn;
                    dst[1] = mx;
                }
                mn = INFINITY;
                mx = -INFINITY;
            }
        }
        return;
    }

    int wbuf = 0;   // (segments) the buffer of this segment's weights
    i32x16 acc;
    int qs = 0, sg = 0;
    for (int t = t0; t < t1;) {
        // ---- phase 1
        const int units = units_of(sg);
        for (int u = wv; u < units; u += 2 * nw) {
            if (u + nw < units) fetch(u + nw, t, sg, v1);
            quantise(u, sg, v0);
            if (u + nw < units) {
                if (u + 2 * nw < units) fetch(u + 2 * nw, t, sg, v0);
                quantise(u + nw, sg, v1);
            }
        }
        if (SEG || t == t0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the weights are there
        __syncthreads();
        const int sn = SEG && sg + 1 < segs ? sg + 1 : 0, tn = sn ? t : t + 1;   // the next patch
        if (tn < t1) {
            if (wv < units_of(sn)) fetch(wv, tn, sn, v0);   // its first loads pass under phase 2
            if constexpr (SEG) weights(sn, wbuf ^ 1);
        }

        // ---- phase 2
        if (!SEG || sg == 0) {
#pragma unroll
            for (int i = 0; i < 16; i++) acc[i] = 0;
            qs = 0;
        }
        const int first = SEG ? sg * nss : 0, steps = SEG ? min(nss, p.nsteps - first) : nss;
        const int s0 = (steps * kw_) >> lwks, s1 = blk * 32 < p.ocg ? (steps * (kw_ + 1)) >> lwks : s0;   // (uniform; no block: nothing to multiply)
        const unsigned char *w_at = w_lds + (SEG ? wbuf * wbytes : 0);
        for (int s = s0; s < s1; s += 4) {
            uint32_t e[4];
            i32x4 af[4];
#pragma unroll
            for (int i = 0; i < 4; i++) e[i] = tab[hf * nss + min(s + i, s1 - 1)];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const unsigned char *at = a_lds + (e[i] & 0xffffffu);
                if constexpr (C4) {
#pragma unroll
                    for (int q = 0; q < 4; q++) af[i][q] = *reinterpret_cast<const int *>(at + q * p.dil * 4);
                } else {
                    af[i] = *reinterpret_cast<const i32x4 *>(at);
                }
            }
#pragma unroll
            for (int i = 0; i < 4; i++) {
                if (s + i >= s1) break;   // (wave-uniform)
                acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[i], *reinterpret_cast<const i32x4 *>(w_at + (s + i) * 1024), acc, 0, 0, 0);
                if constexpr (C4) {
#pragma unroll
                    for (int q = 0; q < 4; q++) qs = __builtin_amdgcn_sdot4(af[i][q], q < (int)(e[i] >> 24) ? 0x01010101 : 0, qs, false);
                } else {
                    const int ones = SEG ? (first + s + i == p.nsteps - 1 ? tail : 0x01010101) : ((e[i] >> 24) ? 0x01010101 : 0);
#pragma unroll
                    for (int q = 0; q < 4; q++) qs = __builtin_amdgcn_sdot4(af[i][q], ones, qs, false);
                }
            }
        }
        if constexpr (SEG) {
            wbuf ^= 1;
            if (sn) {   // (uniform) more of this rectangle's channels
                sg = sn;
                __syncthreads();   // this segment is read before the next one is written
                continue;
            }
            sg = 0;
        }
        // ---- the K parts meet (exact integers: any order), and every wave that held one finishes its share of the pixels
        qs += __shfl_xor(qs, 32, 64);   // the two k halves of a pixel
        if (hf == 0) s_qs[wv][lr] = qs;
        if constexpr (KS) {
#pragma unroll
            for (int ig = 0; ig < 4; ig++)
                *reinterpret_cast<i32x4 *>(red + ((wv * 4 + ig) * 64 + lane) * 4) = i32x4{acc[ig * 4], acc[ig * 4 + 1], acc[ig * 4 + 2], acc[ig * 4 + 3]};
            __syncthreads();
        } else {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            if (share) {
                // rows of 16 lanes: (k half 0, channels 0-15), (0, 16-31), (1, 0-15), (1, 16-31).  Registers 8 .. 15 (pixel
                // groups 2 and 3) of the even rows move into registers 0 .. 7 of the odd rows above them
#pragma unroll
                for (int i = 0; i < 8; i++) acc[i] = (int)__builtin_amdgcn_permlane16_swap((uint32_t)acc[i], (uint32_t)acc[i + 8], false, false)[0];
            }
        }
        rectangle(t);
        float rs[4];
        int at, ow;
        if constexpr (KS) {
            for (int ig = (4 * kw_) >> lwks; ig < (4 * (kw_ + 1)) >> lwks; ig++) {   // (eight parts: every other wave has one)
                const int *src = red + (((wv - kw_) * 4 + ig) * 64 + lane) * 4;
                i32x4 a4 = *reinterpret_cast<const i32x4 *>(src);
                for (int k2 = 1; k2 < wks; k2++) {
                    const i32x4 o4 = *reinterpret_cast<const i32x4 *>(src + k2 * (4 * 64 * 4));
#pragma unroll
                    for (int j = 0; j < 4; j++) a4[j] += o4[j];
                }
                if (pixels(ig, rs, at, ow)) finish(a4, rs, at, ow);
            }
        } else {
#pragma unroll
            for (int t4 = 0; t4 < 4; t4++) {
                if (share && t4 >= 2) break;
                if (pixels(share ? t4 + 2 * (lr >> 4) : t4, rs, at, ow))
                    finish(i32x4{acc[t4 * 4], acc[t4 * 4 + 1], acc[t4 * 4 + 2], acc[t4 * 4 + 3]}, rs, at, ow);
            }
        }
        if (++t < t1) __syncthreads();   // this patch is read before the next one is written
    }

    if (p.range_out) {
        // one pair per workgroup and block of 32 channels, [image][block][workgroup]: a convolution that reads whole blocks takes
        // their pairs
        mn = wave_min(mn);
        mx = wave_max(mx);
        if (lane == 0) { s_rng[wv][0] = mn; s_rng[wv][1] = mx; }
        __syncthreads();
        const int b32 = (int)blockIdx.y * wch + tid;
        if (tid < wch && b32 * 32 < p.ocg) {
            mn = INFINITY;
            mx = -INFINITY;
            for (int w2 = 0; w2 < nw; w2++)
                if (((w2 >> lwks) & (wch - 1)) == tid) { mn = fminf(mn, s_rng[w2][0]); mx = fmaxf(mx, s_rng[w2][1]); }
            float *dst = p.range_out + ((int64_t)nn * p.range_stride + (int64_t)b32 * p.parts + part) * 2;
            dst[0] = mn;
            dst[1] = mx;
        }
    }
}

// Weight rows in the order of the kernel above, one workgroup per channel (channels past the group's last: zeros), and the
// sum of a row's integers.
__global__ void __launch_bounds__(64) conv_words_kernel(const uint32_t *words, int64_t kp, int bits, int ocg, int cg, int kh, int kw, int ncb, int nsteps,
                                                        int nch, int kwc, int8_t *cw, int32_t *qsum)
{
    const int lane = threadIdx.x, nb = ncb * 32, g = blockIdx.x / nb, n = blockIdx.x % nb;
    const uint32_t *row = words + ((int64_t)g * ocg + n) * kp;
    const bool c4 = kwc > 0;
    int sum = 0;
    for (int kc = lane; kc < 2 * nsteps; kc += 64) {
        u32x4 o = {0, 0, 0, 0};
        const int per = c4 ? kwc : kh * kw, q = kc / per, r = kc - q * per;   // (kernel row, four columns) or (sixteen channels, tap)
        if (n < ocg && q < (c4 ? kh : nch)) {
#pragma unroll
            for (int b = 0; b < 16; b++) {
                const int c = c4 ? b & 3 : q * 16 + b, j = c4 ? r * 4 + (b >> 2) : r % kw, i = c4 ? q : r / kw;
                if (c >= cg || j >= kw) continue;
                const int k = (c * kh + i) * kw + j;
                const int q = bits == 4 ? ((int)(row[k >> 3] << (28 - 4 * (k & 7)))) >> 28 : (int)(int8_t)(row[k >> 2] >> (8 * (k & 3)));
                o[b >> 2] |= (uint32_t)(q & 255) << (8 * (b & 3));
                sum += q;
            }
        }
        reinterpret_cast<u32x4 *>(cw)[((int64_t)(g * ncb + n / 32) * nsteps + (kc >> 1)) * 64 + (kc & 1) * 32 + (n & 31)] = o;
    }
    sum = wave_sum_i32(sum);
    if (lane == 0 && n < ocg) qsum[g * ocg + n] = sum;
}

struct Geometry { int nch, kwc, nkc, nsteps, ncb; };   // ncb: blocks of 32 channels kept

Geometry geometry(int64_t cg, int64_t ocg, int kh, int kw)
{
    Geometry q;
    const bool c4 = cg <= 4;
    q.nch = (int)((cg + 15) / 16);
    q.kwc = c4 ? (kw + 3) / 4 : 0;
    q.nkc = c4 ? kh * q.kwc : kh * kw * q.nch;
    q.nsteps = (q.nkc + 1) / 2;
    q.ncb = (int)((ocg + 31) / 32);
    return q;
}

typedef FnnPatchShape Shape;

// The rectangle of 32 * wpx pixels with the fewest patch values to load and outputs to finish; false: does not fit the LDS.
bool place(const QConvArgs &p, const Geometry &q, Shape &s)
{
    const bool flat = p.kh == 1 && p.kw == 1 && p.pad == 0 && p.stride == 1;
    const int64_t cg = p.c / p.groups, ocg = p.oc / p.groups, np = p.ho * p.wo;
    const int64_t ho = flat ? 1 : p.ho, wo = flat ? np : p.wo;
    double best = 0;
    bool found = false;
    for (int twl = 2; twl <= 9; twl++) {
        const int tw = 1 << twl, th = 32 * s.wpx / tw;
        if (th < 1 || (flat && th != 1)) continue;
        const int64_t pw = (int64_t)(tw - 1) * p.stride + (int64_t)(p.kw - 1) * p.dil + 1, ph = (int64_t)(th - 1) * p.stride + (int64_t)(p.kh - 1) * p.dil + 1;
        if (pw * ph > 1 << 16) continue;
        const int64_t pp = pw * ph, tx = (wo + tw - 1) / tw, tiles = tx * ((ho + th - 1) / th);
        const int64_t patch = cg <= 4 ? (pp * 4 + 4 * 4 * p.dil + 15) / 16 * 16 : pp * s.cs * 16;
        const int64_t bytes = patch + (s.sets ? 0 : (int64_t)s.wch * s.nss * 1024 * (s.segs > 1 ? 2 : 1)) + (s.nss * 8 + 15) / 16 * 16 + (s.wks > 1 ? 4096 * s.nw : 0);
        if (bytes > MAX_LDS) continue;
        // vector instructions: 8 a patch value, 18 an output; narrow rectangles use less of a cache line
        const double cost = (double)tiles * ((double)((pp + 63) / 64 * 64) * (cg <= 4 ? cg : q.nch * 16) * 8 + 32.0 * s.wpx * ((ocg + 31) / 32 * 32) * 18) * (1 + 0.4 / tw);
        if (found && cost >= best) continue;
        best = cost; found = true;
        s.twl = twl; s.th = th; s.pw = (int)pw; s.pp = (int)pp; s.tiles_x = (int)tx; s.tiles = (int)tiles; s.lds = (size_t)bytes;
    }
    return found;
}

// Microseconds expected of a shape, and of the operand kernel + GEMM pair (qgemm_i8.hip); both with a range scan's launch, without its bytes.  Fitted
// by least squares to 678 layers (YOLOv8n's at 224 to 640 pixels a side and batches of 1 to 16, ResNet's at 1, 8 and 32, VGG's, U-Net's, heads, and
// 400 drawn ones: 3 to 2048 channels in and out, kernels of 1 to 7, dilated, grouped, odd widths) in every shape that fits, 38 700 timings.  A
// rectangle is a chain of latencies or what its waves issue, whichever is longer.  On 150 layers that the fit had not seen the choice is
// 1.5 % off the best one on average (5 % of them more than 9 %).
float patch_us(const QConvArgs &p, const Geometry &q, const Shape &s)
{
    const int64_t cg = p.c / p.groups, ocg = p.oc / p.groups;
    const bool c4 = cg <= 4, split = !c4 && s.pp <= 32 && s.cs > 1, flat = p.kh == 1 && p.kw == 1 && p.pad == 0 && p.stride == 1;
    const int groups = (s.pp + 63) / 64, rest = s.segs - 1;
    auto units_of = [&](int chunks) { return (float)(((split ? (chunks + 1) / 2 : groups * chunks) + s.nw - 1) / s.nw); };
    auto fours_of = [&](int steps) { return (float)(((steps + s.wks - 1) / s.wks + 3) / 4); };
    const int sets = s.sets ? s.sets : 1, blocks = s.wch * sets * s.gy;
    const float units = c4 ? 0.25f * units_of(1) : rest * units_of(s.cs) + units_of(q.nch - rest * s.cs);
    const float fours = (float)sets * (rest * fours_of(s.nss) + fours_of(q.nsteps - rest * s.nss)), busy = (float)(blocks < q.ncb ? blocks : q.ncb) / (float)blocks;
    const float steps = (float)((q.nsteps + s.wks - 1) / s.wks * sets) * busy;
    const float items = s.wks == 1 ? (ocg <= 16 && !s.sets ? 2.f : 4.f * sets) : (s.wks < 4 ? 4.f / s.wks : 1.f);
    const int64_t wgs = p.b * ((s.tiles + s.per - 1) / s.per) * s.gy, per_cu = (wgs + 255) / 256;
    int64_t resident = 160 * 1024 / (int64_t)(s.lds + 1300) < 16 / s.nw ? 160 * 1024 / (int64_t)(s.lds + 1300) : 16 / s.nw;
    if (resident < 1) resident = 1;
    const float seq = (float)((per_cu + resident - 1) / resident) * s.per, waves = (float)(per_cu * s.per * s.nw);
    // (a row of the patch begins and ends inside a line; pieces: rows that 64 of its pixels lie in)
    const float pieces = 64.f / (float)s.pw, row_mb = (float)(p.b * s.tiles * s.gy) * (float)(s.pp / s.pw) * (float)cg * 64e-6f;
    const float chain = seq * (((c4 ? 0.825f : 0.573f) + 0.0177f * (pieces < 16.f ? pieces : 16.f)) * units + (s.sets ? 0.319f : (c4 ? 0.485f : 0.39f)) * fours +
                               0.317f * items + (s.wks > 1 ? 0.5f : 0.f) + 0.412f * rest + (s.sets ? 0.458f : 0.f));
    const float issue = waves * (0.019f + ((c4 ? 0.0222f : 0.0541f) + 0.00169f * pieces) * units + (s.sets ? 0.01304f : (c4 ? 0.0118f : 0.00967f)) * steps + 0.0195f * items);
    const float c2 = chain * chain, i2 = issue * issue;
    const float out_mb = (float)(p.b * p.oc) * (float)(p.ho * p.wo) * 4e-6f, patch_mb = (float)(p.b * s.tiles * s.gy) * (float)s.pp * (float)cg * 4e-6f;
    const bool vec4 = (flat ? p.ho * p.wo : p.wo) % 4 == 0;
    const float weights = s.sets ? 0.f : 0.0108f * (float)(per_cu * s.wch * q.nsteps) * (float)(rest ? s.per : 1);
    const float each = sqrtf(sqrtf(c2 * c2 + i2 * i2)) + weights + 0.116f * (float)(per_cu * s.nw) + 0.0036f * patch_mb + 0.0946f * row_mb;
    return 3.06f + 3.88f * p.groups + p.groups * each + (vec4 ? 0.08f : 0.57f) * out_mb;
}
float pair_us(const QConvArgs &p)
{
    const int64_t np = p.ho * p.wo;
    const float rows = (float)(p.b * np), ocg = (float)(p.oc / p.groups), kk = (float)((p.c / p.groups) * p.kh * p.kw);
    const float stages = ceilf(kk / 128), wgs = ceilf(rows / 64) * ceilf(ocg / 64), rounds = ceilf(wgs / 256);
    const float in_mb = (float)(p.b * p.c) * (float)(p.h * p.w) * 4e-6f, out_mb = rows * (float)p.oc * 4e-6f;
    const float each = (0.298f + 0.203f * rounds + 0.000446f * wgs) * stages + 0.352f * rounds +
                       rows * (1.28e-6f * ocg + (0.141e-6f + (p.kh * p.kw > 1 ? 0.341e-6f : 0.f) + (p.stride > 1 ? 0.117e-6f : 0.f)) * kk);
    return 2.71f + 8.25f * p.groups + p.groups * each + (np < 64 ? 1.3f : 0.f) + (np % 4 ? 0.55f : 0.f) * out_mb + 0.075f * in_mb;
}

// false: the pair runs this convolution.  form: FNN_OPT_CONV_PATCH
bool choose(const QConvArgs &p, const Geometry &q, int option, int form, Shape &best)
{
    // waves over pixels and over channels, all of them (the rest share K)
    static const int8_t shapes[][3] = {{1, 1, 4}, {1, 1, 8}, {1, 2, 4}, {1, 2, 8}, {1, 4, 4}, {1, 4, 8}, {2, 1, 4}, {2, 1, 8}, {2, 2, 4}, {2, 4, 8}, {1, 8, 8}, {4, 1, 4}, {4, 1, 8}, {4, 2, 8}, {8, 1, 8}};
    float us = 0;
    bool found = false;
    // cs: chunks of a segment, 0: all of them in one; sets: blocks of a wave that fetches its weights itself
    auto consider = [&](int wpx, int wch, int nw, int per, int cs, int sets = 0) {
        Shape s;
        s.wpx = wpx; s.wch = wch; s.nw = nw; s.wks = nw / (wpx * wch); s.per = per;
        if (wch * (sets ? sets : 1) >= 2 * q.ncb || (sets && s.wks > 1) || (cs && (cs >= q.nch || p.c / p.groups <= 4))) return;
        s.cs = cs ? cs : q.nch;
        s.segs = (q.nch + s.cs - 1) / s.cs;
        s.nss = cs ? cs * p.kh * p.kw / 2 : q.nsteps;
        s.sets = sets;
        s.gy = (q.ncb + wch * (sets ? sets : 1) - 1) / (wch * (sets ? sets : 1));
        if (!place(p, q, s)) return;
        // several rectangles a workgroup only where that leaves work for most CUs
        for (int k = 1; k <= (per || sets ? 1 : 4); k *= 2) {
            if (!per) s.per = k;
            if (!per && k > 1 && p.b * ((s.tiles + k - 1) / k) * s.gy < 200) break;
            const float t = patch_us(p, q, s) * (sets ? 1.04f : 1.0f);   // (the margin: a shape in sets has to be ahead beyond the fit's noise)
            if (!found || t < us) { us = t; best = s; found = true; }
        }
    };
    if (form) {
        const int wpx = 1 << (form & 3), wch = 1 << ((form >> 2) & 3), nw = 4 << ((form >> 4) & 1);
        const int per = 1 << ((form >> 5) & 3), cs = (form >> 8) & 7 ? 1 << ((form >> 8) & 7) : 0, sets = (form >> 11) & 7 ? 1 << (((form >> 11) & 7) - 1) : 0;
        if (wpx * wch <= nw && !(sets && (cs || per > 1))) consider(wpx, wch, nw, per, cs, sets);
        return found;
    }
    for (const auto &c : shapes) consider(c[0], c[1], c[2], 0, 0);
    // (segments: an even number of chunks, so that a segment is whole steps of two; up to 24 KB of weights a block they gain nothing)
    for (int cs = 2; cs < q.nch && q.nsteps > 24; cs *= 2)
        for (const auto &c : shapes) consider(c[0], c[1], c[2], 0, cs);
    // (sets: the best shape of 3 % of the layers with one block of output channels, of 21 % with two, of 39 % from three on)
    for (const auto &c : shapes)
        for (int sets = 1; sets <= 8; sets *= 2) consider(c[0], c[1], c[2], 0, 0, sets);
    return found && (option != 0 || us < 1.05f * pair_us(p));   // (large layers take the pair up to 30 % longer than expected)
}

bool plan(const fnn_hip_ctx *ctx, const fnn_hip_weight *w, const QConvArgs &p, Geometry &q, Shape &s)
{
    const int option = (int)fnn_ctx_option(ctx, FNN_OPT_CONV_IMPLICIT);
    if (option == 2 || (w->dtype != FNN_DT_I8 && w->dtype != FNN_DT_I4) || p.x8 || p.payload_i4) return false;
    const int64_t cg = p.c / p.groups, ocg = p.oc / p.groups, np = p.ho * p.wo;
    // 32-bit offsets inside a slab of the input and inside an image of the output, whole tiles in 31 bits
    if (p.c * p.h * p.w >= 1ll << 29 || p.oc * np >= 1ll << 29 || p.b * np >= 1ll << 30 || p.kh > 64 || p.kw > 64 || cg * p.kh * p.kw > 1 << 20) return false;
    if (p.pad > 32767 || p.dil > 32767 || p.stride > 32767 || p.h > 1 << 24 || p.w > 1 << 24) return false;
    q = geometry(cg, ocg, p.kh, p.kw);
    return choose(p, q, option, (int)fnn_ctx_option(ctx, FNN_OPT_CONV_PATCH), s) && p.b * s.tiles < 1ll << 30;
}

template <bool KS, bool C4, Form FORM>
hipError_t launch(const PatchArgs &p, dim3 grid, size_t lds, hipStream_t s)
{
    static std::atomic<uint64_t> raised{0};
    if (lds > 48 * 1024) {
        const hipError_t e = fnn_raise_lds_limit(raised, (const void *)conv_patch_kernel<KS, C4, FORM>, MAX_LDS);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL((conv_patch_kernel<KS, C4, FORM>), grid, dim3(64u << p.lnw), lds, s, p);
    return hipGetLastError();
}

}  // namespace

// What a quantised Conv2d keeps with its weight: the rows in the kernel's order (where this call may have memory for them; false: not
// there, or in the order of another kernel geometry) and the sums of their integers.
static bool conv_words(fnn_hip_ctx *ctx, hipStream_t stream, const fnn_hip_weight *w, int groups, int64_t cg, int kh, int kw)
{
    fnn_hip_weight *wm = const_cast<fnn_hip_weight *>(w);
    if (wm->conv_words) return wm->conv_groups == groups && wm->conv_kh == kh && wm->conv_kw == kw;
    const int64_t ocg = w->rows / groups;
    const Geometry q = geometry(cg, ocg, kh, kw);
    const size_t copy = (size_t)groups * q.ncb * q.nsteps * 1024;
    if ((int64_t)groups * q.ncb * 32 > 1 << 30) return false;
    // one allocation for the copy and, behind it, the row sums
    void *mem = fnn_ctx_copy_memory(ctx, copy + (size_t)w->rows * 4 + 64);
    if (!mem) return false;
    int32_t *sums = reinterpret_cast<int32_t *>((char *)mem + copy);
    hipLaunchKernelGGL(conv_words_kernel, dim3((unsigned)(groups * q.ncb * 32)), dim3(64), 0, stream, w->words, w->kp, w->dtype == FNN_DT_I4 ? 4 : 8, (int)ocg,
                       (int)cg, kh, kw, q.ncb, q.nsteps, q.nch, q.kwc, (int8_t *)mem, sums);
    if (hipGetLastError() != hipSuccess) {
        (void)hipFree(mem);
        return false;
    }
    wm->conv_words = (int8_t *)mem;
    wm->conv_groups = groups; wm->conv_kh = kh; wm->conv_kw = kw;
    if (!wm->row_qsum) { wm->row_qsum = sums; wm->row_qsum_shared = true; }
    return true;
}

// Does the kernel take this convolution, and in which shape?  Builds the weight's copy on first use; where that cannot be had now, the
// call is left to the pair.
bool fnn_patch_conv_takes(fnn_hip_ctx *ctx, hipStream_t stream, const fnn_hip_weight *w, const QConvArgs &p, FnnPatchShape *s)
{
    Geometry q;
    return plan(ctx, w, p, q, *s) && conv_words(ctx, stream, w, p.groups, p.c / p.groups, p.kh, p.kw);
}

// p.range_out: partial ranges of y are left when the pairs fit (ctx's out_parts says so)
int fnn_patch_conv(fnn_hip_ctx *ctx, hipStream_t stream, const fnn_hip_weight *w, const QConvArgs &p, const FnnPatchShape &s)
{
    const Geometry q = geometry(p.c / p.groups, p.oc / p.groups, p.kh, p.kw);
    const int64_t cg = p.c / p.groups, ocg = p.oc / p.groups, np = p.ho * p.wo;
    const bool flat = p.kh == 1 && p.kw == 1 && p.pad == 0 && p.stride == 1, c4 = cg <= 4;
    PatchArgs a;
    a.kk = (float)(cg * p.kh * p.kw);
    a.x_image = p.c * p.h * p.w; a.y_image = p.oc * np;
    a.npairs = p.nparts > 0 ? p.nparts : 0; a.pair_stride = p.part_stride * p.groups; a.actq_stride = 4 * p.groups;
    a.range_zero = p.range_zero; a.range_stride = p.range_out_stride;
    a.cg = (int)cg; a.ocg = (int)ocg; a.act = p.act; a.wbits = p.wbits;
    a.hh = flat ? 1 : (int)p.h; a.ww = flat ? (int)np : (int)p.w;
    a.ho = flat ? 1 : (int)p.ho; a.wo = flat ? (int)np : (int)p.wo;
    a.kw = p.kw; a.stride = p.stride; a.pad = p.pad; a.dil = p.dil;
    a.twl = s.twl; a.th = s.th; a.tiles = s.tiles; a.per = s.per; a.parts = (s.tiles + s.per - 1) / s.per;
    a.pw = s.pw; a.pp = s.pp; a.pgroups = (s.pp + 63) / 64; a.split = !c4 && s.pp <= 32 && s.cs > 1;
    a.nch = q.nch; a.nsteps = q.nsteps; a.nkc = q.nkc;
    a.segs = s.segs; a.cs = s.cs; a.nss = s.nss; a.sets = s.sets;
    auto log2of = [](int v) { int l = 0; while (1 << l < v) l++; return l; };
    a.lnw = log2of(s.nw); a.lwch = log2of(s.wch); a.lwks = log2of(s.wks);
    a.w_at = c4 ? (s.pp * 4 + 4 * 4 * p.dil + 15) / 16 * 16 : s.pp * s.cs * 16;
    a.tab_at = a.w_at + (s.sets ? 0 : s.wch * s.nss * 1024 * (s.segs > 1 ? 2 : 1));
    a.red_at = a.tab_at + (s.nss * 8 + 15) / 16 * 16;
    a.dpw = fast_div((uint32_t)s.pw); a.dpg = fast_div((uint32_t)a.pgroups); a.dparts = fast_div((uint32_t)a.parts);
    a.dtx = fast_div((uint32_t)s.tiles_x); a.dper = fast_div((uint32_t)(c4 ? q.kwc : p.kh * p.kw)); a.dkw = fast_div((uint32_t)p.kw);
    a.dnss = fast_div((uint32_t)s.nss);
    const bool with_sum = p.residual && p.sum_out;
    const uintptr_t places = reinterpret_cast<uintptr_t>(p.y) | reinterpret_cast<uintptr_t>(p.acc_out) |
                             (with_sum ? reinterpret_cast<uintptr_t>(p.residual) | reinterpret_cast<uintptr_t>(p.sum_out) : 0);
    a.vec4 = a.wo % 4 == 0 && (places & 15) == 0;
    const int64_t pairs = (int64_t)a.parts * (s.sets ? s.wpx : 1), parts = q.ncb * pairs;   // of a block, of an image
    a.range_out = nullptr;
    if (p.range_out && p.groups == 1 && parts <= p.range_out_stride) {
        FnnRangeIo *rio = fnn_ctx_range_io(ctx);
        rio->out_parts = (int)parts;
        rio->out_tile_elems = 32 * (uint64_t)np;
        rio->out_tile_pairs = (int)pairs;
        a.range_out = p.range_out;
    }
    const dim3 grid((unsigned)(p.b * a.parts), (unsigned)s.gy);
    for (int g = 0; g < p.groups; g++) {
        const int64_t oc0 = g * ocg;
        a.x = p.x + g * cg * p.h * p.w;
        a.cw = w->conv_words + (int64_t)g * q.ncb * q.nsteps * 1024;
        a.scales = p.scales + oc0; a.zeros = p.zeros + oc0; a.qsum = p.row_qsum + oc0;
        a.bias = p.bias ? p.bias + oc0 : nullptr;
        a.actq = p.actq + g * 4; a.pairs = p.minmax_partial + (int64_t)g * p.part_stride * 2;
        a.y = p.y + oc0 * np;
        a.acc_out = p.acc_out ? p.acc_out + oc0 * np : nullptr;
        a.residual = with_sum ? p.residual + oc0 * np : nullptr;
        a.sum_out = with_sum ? p.sum_out + oc0 * np : nullptr;
        hipError_t e;
        if (s.sets) e = c4 ? launch<false, true, SETS>(a, grid, s.lds, stream) : launch<false, false, SETS>(a, grid, s.lds, stream);
        else if (s.segs > 1) e = s.wks > 1 ? launch<true, false, SEGMENTS>(a, grid, s.lds, stream) : launch<false, false, SEGMENTS>(a, grid, s.lds, stream);
        else if (s.wks > 1) e = c4 ? launch<true, true, WHOLE>(a, grid, s.lds, stream) : launch<true, false, WHOLE>(a, grid, s.lds, stream);
        else e = c4 ? launch<false, true, WHOLE>(a, grid, s.lds, stream) : launch<false, false, WHOLE>(a, grid, s.lds, stream);
        if (e != hipSuccess) return fnn_ctx_fail(ctx, FNN_ERR_DISPATCH, hipGetErrorString(e));
    }
    if (with_sum) fnn_ctx_residual_io(ctx)->used = 1;   // the epilogue stored y + residual as well
    return FNN_OK;
}
