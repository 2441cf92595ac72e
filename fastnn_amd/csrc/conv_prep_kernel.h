// Operand of the f16 tiles straight from a convolution's NCHW input (included by qgemm_tiled.hip, inside its namespace): the row of output
// pixel r is col[r, e] = x[b, ic, oh*s + i*d - pad, ow*s + j*d - pad] (0 outside), e = (ic*KH + i)*KW + j (src/backend/cpu/im2col.rs:32-52), and what
// is written is what act_prep_kernel writes for that row, hi and lo the same bits (its two sums meet in double here).  An f32 im2col matrix and a
// workgroup per row of it cost 4.7 of the 6.4 ms of the 45 convolutions of a 640 x 640 detector on 8 images, F8 weights: the matrix is written
// and read again, 8 times the input on the average, and a row of 27 .. 576 values is little work for 256 threads.  Here 1.2 ms (the same detector
// from host memory, us: 640 x 640 1 image 1487 -> 1078, 8 7446 -> 3838, 16 14200 -> 6390; 320 x 320 4 images 1530 -> 1130).
//
// A workgroup owns PX output pixels.  64: a lane one of them, loads coalesce along the image row, and the position of a value in the kernel
// window is the same for the wave (scalar); wave w of eight converts the eight values k = 64 b + 8 w .. of every k block b.  16: four lanes
// share a pixel and a step takes four k blocks, for images that 64 would leave on few CUs with a long chain of steps.  One pass
// for the row maxima and sums, which keeps the first KEEP steps in registers (the others are read again, from L2), then a conversion through
// LDS, a step at a time, so that whole 128-byte rows of the operand leave: 16 bytes a lane, 1 KB in a row a wave.
template <int PX, int KEEP>
__global__ void __launch_bounds__(512) conv_prep_kernel(PrepArgs p, ConvSource q)
{
    static_assert(PX == 16 || PX == 64, "whole blocks of 16 operand rows");
    constexpr int KB = 64 / PX;   // k blocks a step: lane = pixel + PX * (eight values of its wave's KB times eight)
    __shared__ uint4 tile[2][128 * 8];
    __shared__ float smx[8][PX];
    __shared__ double ssum[8][PX];
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), pix = lane % PX;
    const int grp = PX == 64 ? wv : wv * KB + lane / PX;   // of a step's 8 KB groups of eight values
    const int64_t r = (int64_t)blockIdx.x * PX + pix;
    const bool live = r < p.m;
    const unsigned nn = (unsigned)r / (unsigned)q.np, px = (unsigned)r - nn * q.np, oh = px / (unsigned)q.wo, ow = px - oh * q.wo;
    const int ih0 = (int)oh * q.stride - q.pad, iw0 = (int)ow * q.stride - q.pad, khw = q.kh * q.kw, K = (int)p.k;
    const unsigned at0 = (unsigned)(nn * (unsigned)q.c * (unsigned)q.h + (unsigned)ih0) * (unsigned)q.w + (unsigned)iw0;
    const __amdgpu_buffer_rsrc_t xbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(q.x), 0, (int)q.bytes, 0x00020000);
    const int nkb = (int)(p.kpad / 64), steps = (nkb + KB - 1) / KB;
    auto load = [&](int b, float (&v)[8]) {
        const int k0 = (b * 8 * KB + grp) * 8;
        int ic = (int)((unsigned)k0 / (unsigned)khw);
        if (PX == 64) ic = __builtin_amdgcn_readfirstlane(ic);
        const int rem = k0 - ic * khw;
        int i = (int)((unsigned)rem / (unsigned)q.kw);
        if (PX == 64) i = __builtin_amdgcn_readfirstlane(i);
        int j = rem - i * q.kw;
#pragma unroll
        for (int t = 0; t < 8; t++) {
            const bool ok = live && k0 + t < K && (unsigned)(ih0 + i * q.dil) < (unsigned)q.h && (unsigned)(iw0 + j * q.dil) < (unsigned)q.w;
            const unsigned at = at0 + ((unsigned)ic * (unsigned)q.h + (unsigned)(i * q.dil)) * (unsigned)q.w + (unsigned)(j * q.dil);
            v[t] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xbuf, ok ? at * 4u : 0x80000000u, 0, 0));   // (past the end: 0)
            if (++j == q.kw) { j = 0; if (++i == q.kh) { i = 0; ic++; } }
        }
    };
    auto over_lanes = [&](auto v, auto op) {   // of the lanes that share a pixel
#pragma unroll
        for (int d = PX; d < 64; d *= 2) v = op(v, __shfl_xor(v, d));
        return v;
    };
    auto add = [](double a, double b) { return a + b; };
    float keep[KEEP][8], mx = 0.0f;
    double sum = 0.0;
    auto gather = [&](const float (&v)[8]) {
#pragma unroll
        for (int t = 0; t < 8; t++) mx = fmaxf(mx, fabsf(v[t]));
        sum += (double)(((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7])));
    };
#pragma unroll
    for (int b = 0; b < KEEP; b++)
        if (b < steps) load(b, keep[b]);
#pragma unroll
    for (int b = 0; b < KEEP; b++)
        if (b < steps) gather(keep[b]);
    for (int b = KEEP; b < steps; b++) {
        float v[8];
        load(b, v);
        gather(v);
    }
    smx[wv][pix] = over_lanes(mx, [](float a, float b) { return fmaxf(a, b); });   // (lanes of a pixel store the same)
    ssum[wv][pix] = over_lanes(sum, add);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 8; u++) mx = fmaxf(mx, smx[u][pix]);
    int e = 0;
    if (mx > 0.0f && mx < __builtin_huge_valf()) {
        int ex;
        (void)frexpf(mx, &ex);   // mx = f * 2^ex, f in [0.5, 1)
        e = 15 - ex;             // mx * 2^e in [2^14, 2^15)
    }
    const bool own = tid < PX && (p.precise ? r < p.rows_pad / 2 : r < p.rows_pad);
    if (own) {
        sum = 0.0;
        for (int u = 0; u < 8; u++) sum += ssum[u][pix];
        p.rexp[r] = e;
        p.xsum[r] = (float)sum;
    }
    // the pixel's row of the workgroup's (precise: 16 rows of hi, their 16 of lo, ...)
    const int row = p.precise ? (pix >> 4) * 32 + (pix & 15) : pix, lg = (PX == 64 ? 6 : 4) + (p.precise ? 1 : 0), rows = 1 << lg;
    const int64_t row0 = (int64_t)blockIdx.x * rows;
    double err = 0.0;
    auto convert = [&](int b, const float (&v)[8]) {
        uint4 *buf = tile[b & 1];   // (one barrier a step: the buffer was read before the last one)
        f16x8 h, l;
        float er = 0.0f;
#pragma unroll
        for (int t = 0; t < 8; t++) {
            // operand slot t holds k = 0,4,1,5,2,6,3,7 for the nibble decoders
            const float xs = ldexpf(p.interleaved ? v[(t & 1) * 4 + (t >> 1)] : v[t], e);
            const _Float16 hh = (_Float16)xs;
            h[t] = hh;
            const float rr = xs - (float)hh;
            l[t] = (_Float16)(rr * LO_UP);
            er -= rr;
        }
        err += (double)er;
        uint4 *at = buf + (((grp >> 3) << lg) + row) * 8 + ((grp & 7) ^ (pix & 7));
        at[0] = __builtin_bit_cast(uint4, h);
        if (p.precise) at[16 * 8] = __builtin_bit_cast(uint4, l);
        __syncthreads();
        for (int c = tid; c < KB * rows * 8; c += 512) {
            const int line = c >> 3, kb = b * KB + (line >> lg), rw = line & (rows - 1);
            if (kb < nkb && row0 + rw < p.rows_pad)
                *reinterpret_cast<uint4 *>(p.ap + ((int64_t)kb * p.rows_pad + row0 + rw) * 64 + (c & 7) * 8) = buf[line * 8 + ((c & 7) ^ (rw & 7))];
        }
    };
#pragma unroll
    for (int b = 0; b < KEEP; b++)
        if (b < steps) convert(b, keep[b]);
    for (int b = KEEP; b < steps; b++) {
        float v[8];
        load(b, v);
        convert(b, v);
    }
    __syncthreads();
    ssum[wv][pix] = over_lanes(err, add);
    __syncthreads();
    if (own) {
        err = 0.0;
        for (int u = 0; u < 8; u++) err += ssum[u][pix];
        p.esum[r] = (float)err;
    }
}

template <int PX>
void launch_conv_prep_of(const PrepArgs &p, const ConvSource &q, int64_t m_pad, hipStream_t s)
{
    const dim3 grid((unsigned)((m_pad + PX - 1) / PX));
    const int64_t steps = (p.kpad + 4096 / PX - 1) / (4096 / PX);
    if (steps == 1) hipLaunchKernelGGL((conv_prep_kernel<PX, 1>), grid, dim3(512), 0, s, p, q);
    else if (steps <= 3) hipLaunchKernelGGL((conv_prep_kernel<PX, 3>), grid, dim3(512), 0, s, p, q);
    else hipLaunchKernelGGL((conv_prep_kernel<PX, 9>), grid, dim3(512), 0, s, p, q);
}

hipError_t launch_conv_prep(const PrepArgs &p, const ConvSource &q, int64_t m_pad, hipStream_t s)
{
    // 16 pixels wherever a step of four k blocks is full, up to 65536 pixels; the same detector, us, 64 / 16 everywhere to 16384 pixels / so:
    // 640 x 640 1 image 1005 / 973 / 974, 4 2148 / 2075 / 2055, 16 6070 / 6100 / 5940; 320 x 320 4 images 1053 / 1019 / 1020
    if (m_pad > 65536 || p.kpad < 256) launch_conv_prep_of<64>(p, q, m_pad, s);
    else launch_conv_prep_of<16>(p, q, m_pad, s);
    return hipGetLastError();
}
