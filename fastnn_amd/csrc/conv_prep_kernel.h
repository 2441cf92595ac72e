// Operand of the f16 tiles straight from a convolution's NCHW input (included by qgemm_tiled.hip, inside its namespace): the row of output
// pixel r is col[r, e] = x[b, ic, oh*s + i*d - pad, ow*s + j*d - pad] (0 outside), e = (ic*KH + i)*KW + j (src/backend/cpu/im2col.rs:32-52), and what
// is written is what act_prep_kernel writes for that row, hi and lo the same bits (its two sums meet in double here).  An f32 im2col matrix and a
// workgroup per row of it cost 4.7 of the 6.4 ms of the 45 convolutions of a 640 x 640 detector on 8 images, F8 weights: the matrix is written
// and read again, 8 times the input on the average, and a row of 27 .. 576 values is little work for 256 threads.  Here 1.2 ms (the same detector
// from host memory, us: 640 x 640 1 image 1487 -> 1078, 8 7446 -> 3838, 16 14200 -> 6390; 320 x 320 4 images 1530 -> 1130).
//
// A workgroup owns 64 output pixels, a lane one of them: loads coalesce along the image row, and the position of a value in the kernel window is
// the same for the wave (scalar).  Eight waves: wave w converts the eight values k = 64 b + 8 w .. of every k block b.  One pass for the row
// maxima and sums, which keeps the first KEEP blocks in registers (the others are read again, from L2), then a conversion through
// LDS, a k block at a time, so that whole 128-byte rows of the operand leave: 16 bytes a lane, 1 KB in a row a wave.
template <int KEEP>
__global__ void __launch_bounds__(512) conv_prep_kernel(PrepArgs p, ConvSource q)
{
    __shared__ uint4 tile[2][128 * 8];
    __shared__ float smx[8][64];
    __shared__ double ssum[8][64];
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t r = (int64_t)blockIdx.x * 64 + lane;
    const bool live = r < p.m;
    const unsigned nn = (unsigned)r / (unsigned)q.np, px = (unsigned)r - nn * q.np, oh = px / (unsigned)q.wo, ow = px - oh * q.wo;
    const int ih0 = (int)oh * q.stride - q.pad, iw0 = (int)ow * q.stride - q.pad, khw = q.kh * q.kw, K = (int)p.k;
    const unsigned at0 = (unsigned)(nn * (unsigned)q.c * (unsigned)q.h + (unsigned)ih0) * (unsigned)q.w + (unsigned)iw0;
    const __amdgpu_buffer_rsrc_t xbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(q.x), 0, (int)q.bytes, 0x00020000);
    const int nkb = (int)(p.kpad / 64);
    auto load = [&](int b, float (&v)[8]) {
        const int k0 = b * 64 + wv * 8;
        int ic = __builtin_amdgcn_readfirstlane((int)((unsigned)k0 / (unsigned)khw));
        const int rem = k0 - ic * khw;
        int i = __builtin_amdgcn_readfirstlane((int)((unsigned)rem / (unsigned)q.kw)), j = rem - i * q.kw;
#pragma unroll
        for (int t = 0; t < 8; t++) {
            const bool ok = live && k0 + t < K && (unsigned)(ih0 + i * q.dil) < (unsigned)q.h && (unsigned)(iw0 + j * q.dil) < (unsigned)q.w;
            const unsigned at = at0 + ((unsigned)ic * (unsigned)q.h + (unsigned)(i * q.dil)) * (unsigned)q.w + (unsigned)(j * q.dil);
            v[t] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xbuf, ok ? at * 4u : 0x80000000u, 0, 0));   // (past the end: 0)
            if (++j == q.kw) { j = 0; if (++i == q.kh) { i = 0; ic++; } }
        }
    };
    float keep[KEEP][8], mx = 0.0f;
    double sum = 0.0;
    auto gather = [&](const float (&v)[8]) {
#pragma unroll
        for (int t = 0; t < 8; t++) mx = fmaxf(mx, fabsf(v[t]));
        sum += (double)(((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7])));
    };
#pragma unroll
    for (int b = 0; b < KEEP; b++)
        if (b < nkb) load(b, keep[b]);
#pragma unroll
    for (int b = 0; b < KEEP; b++)
        if (b < nkb) gather(keep[b]);
    for (int b = KEEP; b < nkb; b++) {
        float v[8];
        load(b, v);
        gather(v);
    }
    smx[wv][lane] = mx;
    ssum[wv][lane] = sum;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 8; u++) mx = fmaxf(mx, smx[u][lane]);
    int e = 0;
    if (mx > 0.0f && mx < __builtin_huge_valf()) {
        int ex;
        (void)frexpf(mx, &ex);   // mx = f * 2^ex, f in [0.5, 1)
        e = 15 - ex;             // mx * 2^e in [2^14, 2^15)
    }
    const bool own = wv == 0 && (p.precise ? r < p.rows_pad / 2 : r < p.rows_pad);
    if (own) {
        sum = 0.0;
        for (int u = 0; u < 8; u++) sum += ssum[u][lane];
        p.rexp[r] = e;
        p.xsum[r] = (float)sum;
    }
    // the lane's row of the workgroup's 128 (precise: 16 rows of hi, their 16 of lo, ...) or 64
    const int row = p.precise ? (lane >> 4) * 32 + (lane & 15) : lane, pieces = p.precise ? 1024 : 512;
    const int64_t row0 = (int64_t)blockIdx.x * (pieces / 8);
    double err = 0.0;
    auto convert = [&](int b, const float (&v)[8]) {
        uint4 *buf = tile[b & 1];   // (one barrier a block: the buffer was read before the last one)
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
        buf[row * 8 + (wv ^ (lane & 7))] = __builtin_bit_cast(uint4, h);
        if (p.precise) buf[(row + 16) * 8 + (wv ^ (lane & 7))] = __builtin_bit_cast(uint4, l);
        __syncthreads();
        _Float16 *dst = p.ap + (b * p.rows_pad + row0) * 64;
        for (int c = tid; c < pieces; c += 512)
            if (row0 + (c >> 3) < p.rows_pad) *reinterpret_cast<uint4 *>(dst + c * 8) = buf[(c & ~7) + ((c & 7) ^ ((c >> 3) & 7))];
    };
#pragma unroll
    for (int b = 0; b < KEEP; b++)
        if (b < nkb) convert(b, keep[b]);
    for (int b = KEEP; b < nkb; b++) {
        float v[8];
        load(b, v);
        convert(b, v);
    }
    __syncthreads();
    ssum[wv][lane] = err;
    __syncthreads();
    if (own) {
        err = 0.0;
        for (int u = 0; u < 8; u++) err += ssum[u][lane];
        p.esum[r] = (float)err;
    }
}

hipError_t launch_conv_prep(const PrepArgs &p, const ConvSource &q, int64_t m_pad, hipStream_t s)
{
    const dim3 grid((unsigned)((m_pad + 63) / 64));
    const int64_t nkb = p.kpad / 64;
    if (nkb == 1) hipLaunchKernelGGL(conv_prep_kernel<1>, grid, dim3(512), 0, s, p, q);
    else if (nkb <= 3) hipLaunchKernelGGL(conv_prep_kernel<3>, grid, dim3(512), 0, s, p, q);
    else hipLaunchKernelGGL(conv_prep_kernel<9>, grid, dim3(512), 0, s, p, q);
    return hipGetLastError();
}
