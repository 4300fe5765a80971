// QLinearConv on gfx950 (reference: qlinearConvOp.Run, ops/quant.go:343-420).
//
// Four routes, all exact in int32 and requantised with the reference's
// expression (vek.RequantU8/I8, kernels/vek/quant_amd64.go:52-70):
//  * pixel GEMM: one launch writes the activations channel-innermost with
//    their padding (the zero point) and the weight with the taps outermost;
//    the int8 MFMA GEMM then reads its A rows, the output pixels, straight from
//    those activations (gemm_kernel's CONV), adds −zx′·ΣW + bias per output
//    channel, requantises with that channel's multiplier and stores the NCHW
//    planes. The reference's pointwise and im2colTiled paths (:612-673).
//  * im2col → int8 GEMM, for reductions longer than the pixel GEMM's chunk
//    table and where the column matrix is estimated to cost less (few channels
//    that pad to 16, strides that skip most pixels, more weight than columns;
//    pixel_geom in runtime.cpp): qim2col_kernel writes, per group, the byte column matrix
//    col[row = image·P + pixel][k = (c, kh, kw)] of the raw activations (taps
//    outside the image hold the zero point zx, k past the group's K zero) in
//    whole 128-byte k-tiles, the A operand of the same GEMM.
//  * depthwise: v_dot4 over a kernel row; 3 × 3 and 5 × 5 kernels of stride 1
//    or 2 by lanes that each own 4 × 4 outputs and read their rows straight
//    from memory, other forms by a wave per strip of one output plane, the
//    strip's input rows staged in LDS (the reference's depthwise path, :472-598).
//  * direct: one thread per output element sums w·(x − zx) over the taps
//    inside the image (padded taps contribute exactly 0). Used for narrow
//    groups, where a GEMM would be a sliver, and for depthwise forms the strip
//    kernel does not hold (kernel rows over 8 taps, dilated rows, strips over
//    its LDS) or that give its waves too little work (launch_qconv_depthwise).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.hpp"

#pragma clang fp contract(off)

namespace ingot {

namespace {

__device__ __forceinline__ uint8_t requant_byte(int32_t v, float mult, float zy, int u8) {
    // float32(v)·mult and + zy rounded separately, half to even, saturate
    const float t = (float)v * mult;
    const float r = rintf(t + zy);
    const int iv = u8 ? (r <= 0.f ? 0 : (r >= 255.f ? 255 : (int)r))
                      : (r <= -128.f ? -128 : (r >= 127.f ? 127 : (int)r));
    return (uint8_t)iv;
}

// 4 bytes of an image row from column c on, columns outside [0, w) holding pad:
// one load at the nearest place inside the row, moved into position (w >= 4).
struct RowWord {
    int off, up;    // where to load; bytes to move the word up (> 0) or down
    uint32_t keep;  // the bytes that lie inside
    __device__ __forceinline__ RowWord(int c, int w) {
        off = min(max(c, 0), w - 4);
        up = off - c;
        keep = up > 3 || up < -3 ? 0u : (up >= 0 ? ~0u << (8 * up) : ~0u >> (-8 * up));
    }
    __device__ __forceinline__ uint32_t place(uint32_t raw, uint32_t pad) const {
        const uint32_t v = up >= 0 ? raw << (8 * (up & 3)) : raw >> (8 * (-up & 3));
        return (v & keep) | (pad & ~keep);
    }
};

// Operands of the pixel GEMM. Workgroups below x_blocks move 64 channels × 64
// columns of one padded row: each thread loads 4 columns of 4 channels,
// transposes them with byte permutes, and the tile passes through LDS so that
// the stores are 16 channels of a pixel. The others move 16-byte chunks of the
// weight, neighbouring threads on the taps of one channel run.
struct QlayoutArgs {
    const uint8_t* x;
    uint8_t* xt;
    const int8_t* w;
    int8_t* wt;
    QconvGeom g;
    int hp, wp, cgp;       // padded rows, columns; channels of a group rounded to 16
    int ctiles, wtiles;    // 64-wide tiles over the channels of all groups (padded), over wp
    int64_t x_blocks, w_chunks;
    int64_t ldw, ldp;
    uint32_t pad;          // the zero point in every byte
    uint32_t flip;         // 0x80808080: u8 → s8
};

__global__ void __launch_bounds__(256) qconv_layout_kernel(QlayoutArgs p) {
    const QconvGeom& g = p.g;
    const int tid = threadIdx.x;
    if (blockIdx.x >= p.x_blocks) {
        const int64_t i = (blockIdx.x - p.x_blocks) * 256 + tid;
        if (i >= p.w_chunks) return;
        const int taps = g.KH * g.KW, cpc = p.cgp >> 4;
        const int64_t run = i / taps;  // (output channel, chunk of 16 input channels)
        const int tap = (int)(i - run * taps), m = (int)(run / cpc), cb = (int)(run - (int64_t)m * cpc);
        const int8_t* src = p.w + (int64_t)m * p.ldw + (int64_t)cb * 16 * taps + tap;
        int8_t v[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] = cb * 16 + e < g.Cg ? src[(int64_t)e * taps] : (int8_t)0;
        i32x4_t o;
        __builtin_memcpy(&o, v, 16);
        *(i32x4_t*)(p.wt + (int64_t)m * p.ldp + (int64_t)tap * p.cgp + cb * 16) = o;
        return;
    }
    constexpr int PITCH = 17;  // words of a pixel's 64 channels, odd
    __shared__ uint32_t tile[64 * PITCH];
    uint32_t b = blockIdx.x;
    const int ct = (int)(b % p.ctiles);
    b /= p.ctiles;
    const int wt = (int)(b % p.wtiles);
    b /= p.wtiles;
    const int ih = (int)(b % p.hp) - g.pt;  // input row (outside: padding)
    const int64_t row = b;                   // image · hp + padded row
    const int img = (int)(b / p.hp);
    const int cq = tid >> 4, pq = tid & 15;  // 4 channels, 4 columns
    const int c0 = ct * 64 + cq * 4;         // channel in the padded order: group · cgp + channel
    const int col = wt * 64 + pq * 4 - g.pl;
    uint32_t v[4];
    if (ih < 0 || ih >= g.H) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = p.pad;
    } else {
        const int grp = c0 / p.cgp, cin = c0 - grp * p.cgp;  // 4 channels never straddle groups (cgp % 16 == 0)
        const uint8_t* src = p.x + (((int64_t)img * g.C + (int64_t)grp * g.Cg + cin) * g.H + ih) * g.W;
        const int64_t plane = (int64_t)g.H * g.W;
        const int have = grp < g.G ? g.Cg - cin : 0;
        if (g.W >= 4) {
            const RowWord rw(col, g.W);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = p.pad;
                if (e < have) __builtin_memcpy(&v[e], src + e * plane + rw.off, 4);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = rw.place(v[e], p.pad);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = p.pad;
                for (int i = 0; i < 4; ++i)
                    if (e < have && col + i >= 0 && col + i < g.W)
                        v[e] = (v[e] & ~(0xFFu << (8 * i))) | ((uint32_t)src[e * plane + col + i] << (8 * i));
            }
        }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] ^= p.flip;
    // 4 channels × 4 columns → one word of 4 channels per column
    const uint32_t lo01 = __builtin_amdgcn_perm(v[1], v[0], 0x05010400), hi01 = __builtin_amdgcn_perm(v[1], v[0], 0x07030602);
    const uint32_t lo23 = __builtin_amdgcn_perm(v[3], v[2], 0x05010400), hi23 = __builtin_amdgcn_perm(v[3], v[2], 0x07030602);
    tile[(pq * 4 + 0) * PITCH + cq] = __builtin_amdgcn_perm(lo23, lo01, 0x05040100);
    tile[(pq * 4 + 1) * PITCH + cq] = __builtin_amdgcn_perm(lo23, lo01, 0x07060302);
    tile[(pq * 4 + 2) * PITCH + cq] = __builtin_amdgcn_perm(hi23, hi01, 0x05040100);
    tile[(pq * 4 + 3) * PITCH + cq] = __builtin_amdgcn_perm(hi23, hi01, 0x07060302);
    __syncthreads();
    const int px = tid >> 2, cc = tid & 3;  // one 16-byte chunk per thread
    const int64_t pitch = (int64_t)g.G * p.cgp;
    if (wt * 64 + px < p.wp && ct * 64 + cc * 16 < pitch) {
        const uint32_t* t = tile + px * PITCH + cc * 4;
        *(uint4*)(p.xt + (row * p.wp + wt * 64 + px) * pitch + ct * 64 + cc * 16) = make_uint4(t[0], t[1], t[2], t[3]);
    }
}

// One thread writes 16 consecutive k of one row (a 16-byte store); a row is
// kgl / 16 threads. blockIdx.y is the group.
__global__ void __launch_bounds__(256) qim2col_kernel(const uint8_t* __restrict__ x, QconvGeom g, int rows,
                                                      int kg, int kgl, uint8_t pad, uint8_t* __restrict__ col,
                                                      int64_t col_group) {
    const int chunks = kgl >> 4;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)rows * chunks) return;
    const int r = (int)(t / chunks);
    const int ch = (int)(t - (int64_t)r * chunks);
    const int P = g.OH * g.OW;
    const int img = r / P;
    const int pix = r - img * P;
    const int oh = pix / g.OW, ow = pix - (pix / g.OW) * g.OW;
    const int grp = blockIdx.y;
    const int64_t hw = (int64_t)g.H * g.W;
    const uint8_t* xb = x + ((int64_t)img * g.C + (int64_t)grp * g.Cg) * hw;
    const int taps = g.KH * g.KW;
    int k = ch << 4;
    int cg = k / taps;
    int rem = k - cg * taps;
    int kh = rem / g.KW;
    int kw = rem - kh * g.KW;
    const int ih0 = oh * g.sh - g.pt, iw0 = ow * g.sw - g.pl;
    uint32_t words[4] = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        uint32_t b = 0;
        if (k + i < kg) {
            const int ih = ih0 + kh * g.dh, iw = iw0 + kw * g.dw;
            b = (ih >= 0 && ih < g.H && iw >= 0 && iw < g.W) ? xb[(int64_t)cg * hw + (int64_t)ih * g.W + iw] : pad;
            if (++kw == g.KW) {
                kw = 0;
                if (++kh == g.KH) {
                    kh = 0;
                    ++cg;
                }
            }
        }
        words[i >> 2] |= b << (8 * (i & 3));
    }
    uint8_t* dst = col + (int64_t)grp * col_group + (int64_t)r * kgl + (ch << 4);
    *(uint4*)dst = make_uint4(words[0], words[1], words[2], words[3]);
}

// y[n][m][oh][ow] = requant(Σ w[m][cg][kh][kw]·(x − zx) + bias[m]); w rows are
// ldw bytes apart (the packed int8 weight). Grid-stride over all outputs.
__global__ void __launch_bounds__(256) qconv_direct_kernel(const uint8_t* __restrict__ x, int x_u8, QconvGeom g,
                                                           const int8_t* __restrict__ w, int64_t ldw,
                                                           const int32_t* __restrict__ bias,
                                                           const float* __restrict__ mult, int32_t zx, float zy,
                                                           int y_u8, uint8_t* __restrict__ y, int64_t total) {
    const int64_t hw = (int64_t)g.H * g.W;
    const int Mg = g.M / g.G;
    for (int64_t o = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; o < total; o += (int64_t)gridDim.x * blockDim.x) {
        const int ow = (int)(o % g.OW);
        int64_t t = o / g.OW;
        const int oh = (int)(t % g.OH);
        t /= g.OH;
        const int m = (int)(t % g.M);
        const int img = (int)(t / g.M);
        const int grp = m / Mg;
        const int8_t* wr = w + (int64_t)m * ldw;
        const uint8_t* xb = x + ((int64_t)img * g.C + (int64_t)grp * g.Cg) * hw;
        uint32_t acc = bias ? (uint32_t)bias[m] : 0u;
        const int ih0 = oh * g.sh - g.pt, iw0 = ow * g.sw - g.pl;
        for (int cg = 0; cg < g.Cg; ++cg) {
            const uint8_t* xc = xb + (int64_t)cg * hw;
            const int8_t* wc = wr + cg * g.KH * g.KW;
            for (int kh = 0; kh < g.KH; ++kh) {
                const int ih = ih0 + kh * g.dh;
                if (ih < 0 || ih >= g.H) continue;
                for (int kw = 0; kw < g.KW; ++kw) {
                    const int iw = iw0 + kw * g.dw;
                    if (iw < 0 || iw >= g.W) continue;
                    const uint8_t b = xc[(int64_t)ih * g.W + iw];
                    const int32_t xv = x_u8 ? (int32_t)b : (int32_t)(int8_t)b;
                    acc += (uint32_t)((xv - zx) * (int32_t)wc[kh * g.KW + kw]);
                }
            }
        }
        y[o] = requant_byte((int32_t)acc, mult[m], zy, y_u8);
    }
}

// Depthwise (one input channel per group, channel multiplier allowed): with
// the input as signed bytes xs (x, or x − 128 for u8) a sum is
// Σ w·xs − zs·Σ w (+ bias), exact in int32 (wrapping), zs = zx (− 128), and a
// padded tap holds zs, so it contributes exactly 0, as in the direct kernel.
struct QdwArgs {
    const uint8_t* x;
    const int8_t* w;
    const int32_t* bias;
    const float* mult;
    uint8_t* y;
    int64_t ldw;
    QconvGeom g;
    int mg;              // output channels per input channel
    uint32_t flip;       // 0x80808080 for u8 x, else 0
    int32_t zs;          // zero point of the signed bytes
    float zy;
    int y_u8;
    int th, strips;      // output rows of a strip, strips of a plane
    int planes;          // N·M
    int left;            // LDS column of input column 0: the left pad rounded up to a word
    int wpr;             // words of an LDS row
    int wave_words;      // LDS words per wave
    uint32_t wpr_magic, qpr_magic;  // ceil(2^32 / d): i / d = umulhi(i, magic) for i, d < 2^16
    int qpr;             // groups of 4 outputs in a row
    uint32_t ipp, ipp_magic;  // 4 × 4 output blocks of a plane
};

// The same rounding and saturation as requant_byte, without its branches: the
// rounded value is clamped as a float (a NaN becomes 0, as its conversion does).
__device__ __forceinline__ uint32_t requant_u(int32_t v, float mult, float zy, float lo, float hi) {
    const float t = (float)v * mult;
    const float r = rintf(t + zy);
    const float c = __builtin_amdgcn_fmed3f(r, lo, hi);
    return (uint32_t)(int)(r == r ? c : 0.f) & 0xFFu;
}

// 4 × 4 outputs a lane, K × K kernel, stride S both ways: every input row the
// lane needs is one 8-byte load (two for S = 2), all of them in flight before
// the first is used, shared by the output rows that read it. A load that would
// leave its image row is moved inside and shifted into place; the masks, the
// same for all rows of a lane, put the padding where it was. Blocks run on over
// planes (a 7 × 7 plane is four of them), so small planes fill waves too.
// Bound by instruction issue, about 80 per 4 outputs, and at these sizes by the
// launch: 8 images of 96 × 56 × 56, 3 × 3 (4.8 MB) took 21.0 µs in the direct
// kernel on MI355X, 8.7 µs in the strip kernel below (155 instructions per 4
// outputs) and 5.8 µs here.
template <int S, int K>
__global__ void __launch_bounds__(256) qconv_dw_block_kernel(QdwArgs p) {
    constexpr int NWD = (K + 3) / 4;         // words of a kernel row
    constexpr int NL = (3 * S + K + 7) / 8;  // 8-byte pieces of an input row that 4 outputs read
    constexpr int IR = 3 * S + K;            // input rows of 4 output rows
    const QconvGeom& g = p.g;
    const uint32_t first = blockIdx.x * 256u;
    const uint32_t p0 = first / p.ipp;
    const uint32_t local = first - p0 * p.ipp + threadIdx.x;
    const uint32_t sub = p.ipp == 1 ? local : __umulhi(local, p.ipp_magic);
    const int plane = (int)(p0 + sub);
    if (plane >= p.planes) return;
    const uint32_t blk = local - sub * p.ipp;
    const uint32_t rb = p.qpr == 1 ? blk : __umulhi(blk, p.qpr_magic);
    const int oh0 = (int)rb * 4, ow = (int)(blk - rb * p.qpr) * 4;
    int img = (int)(p0 / (uint32_t)g.M), m = (int)(p0 - (uint32_t)img * g.M + sub);
    while (m >= g.M) m -= g.M, ++img;
    const int ch = p.mg == 1 ? m : m / p.mg;
    const uint8_t* xb = p.x + ((int64_t)img * g.C + ch) * ((int64_t)g.H * g.W);
    const int8_t* wr = p.w + (int64_t)m * p.ldw;

    uint64_t raw[IR][NL], wraw[K];
    int off[NL], shift[NL];
#pragma unroll
    for (int l = 0; l < NL; ++l) {
        const int c = ow * S - g.pl + 8 * l;
        off[l] = min(max(c, 0), g.W - 8);
        shift[l] = off[l] - c;  // bytes to move the piece up (> 0) or down
    }
    const int ih0 = oh0 * S - g.pt;
#pragma unroll
    for (int i = 0; i < IR; ++i) {
        const uint8_t* row = xb + (int64_t)min(max(ih0 + i, 0), g.H - 1) * g.W;
#pragma unroll
        for (int l = 0; l < NL; ++l) __builtin_memcpy(&raw[i][l], row + off[l], 8);
    }
    // kernel rows: 8 bytes from each (inside the packed weight row, at least 256 bytes), zero past K
#pragma unroll
    for (int k = 0; k < K; ++k) __builtin_memcpy(&wraw[k], wr + k * K, 8);
    const int32_t b0 = p.bias ? p.bias[m] : 0;
    const float mu = p.mult[m];

    uint64_t keep[NL];
#pragma unroll
    for (int l = 0; l < NL; ++l)
        keep[l] = shift[l] > 7 || shift[l] < -7 ? 0ull
                  : shift[l] >= 0               ? ~0ull << (8 * shift[l])
                                                : ~0ull >> (-8 * shift[l]);
    const uint64_t pad = (uint64_t)(uint8_t)p.zs * 0x0101010101010101ull;
    const uint64_t flip = ((uint64_t)p.flip << 32) | p.flip;
    int wd[K][NWD], wsum = 0;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const uint64_t w = wraw[k] & ((1ull << (8 * K)) - 1);
#pragma unroll
        for (int d = 0; d < NWD; ++d) {
            wd[k][d] = (int)(uint32_t)(w >> (32 * d));
            wsum = __builtin_amdgcn_sdot4(wd[k][d], 0x01010101, wsum, false);
        }
    }
    int acc[4][4] = {};
#pragma unroll
    for (int i = 0; i < IR; ++i) {
        const int ih = ih0 + i;
        uint32_t x[2 * NL + 1];
        x[2 * NL] = 0;  // past the last window's taps
#pragma unroll
        for (int l = 0; l < NL; ++l) {
            uint64_t v = raw[i][l] ^ flip;
            v = shift[l] >= 0 ? v << (8 * (shift[l] & 7)) : v >> (8 * (-shift[l] & 7));
            v = ih >= 0 && ih < g.H ? (v & keep[l]) | (pad & ~keep[l]) : pad;
            x[2 * l] = (uint32_t)v;
            x[2 * l + 1] = (uint32_t)(v >> 32);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int d = 0; d < NWD; ++d) {
                const int o = ((e * S) >> 2) + d, sh = (e * S) & 3;
                const int xw = (int)(sh ? __builtin_amdgcn_alignbyte(x[o + 1], x[o], sh) : x[o]);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int k = i - r * S;
                    if (k >= 0 && k < K) acc[r][e] = __builtin_amdgcn_sdot4(xw, wd[k][d], acc[r][e], false);
                }
            }
    }
    const int32_t corr = wrap_add(wrap_mul(wsum, -p.zs), b0);
    const float lo = p.y_u8 ? 0.f : -128.f, hi = p.y_u8 ? 255.f : 127.f;
    uint8_t* yo = p.y + ((int64_t)plane * g.OH + oh0) * g.OW + ow;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        if (oh0 + r >= g.OH) break;
        uint32_t out = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) out |= requant_u(wrap_add(acc[r][e], corr), mu, p.zy, lo, hi) << (8 * e);
        if (ow + 3 < g.OW) {
            __builtin_memcpy(yo, &out, 4);
        } else {
            for (int e = 0; e < g.OW - ow; ++e) yo[e] = (uint8_t)(out >> (8 * e));
        }
        yo += g.OW;
    }
}

// Other forms: a wave owns a strip of `th` output rows of one plane. It copies
// the input rows they read into its LDS slice as signed bytes, padding written
// as zs, so that no tap needs a bound; then each lane forms 4 neighbouring
// outputs of a row, a kernel row at a time, as v_dot4 of 4·NWD bytes of input
// and the kernel row (zero past KW). SW: the column stride when 1 or 2 (the
// four windows come out of one run of words); 0: any stride, one window fetched
// per output.

template <int SW, int NWD>
__global__ void __launch_bounds__(256) qconv_dw_kernel(QdwArgs p) {
    extern __shared__ uint32_t dw_lds[];
    const QconvGeom& g = p.g;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int item = blockIdx.x * 4 + wave;
    if (item >= p.planes * p.strips) return;
    const int plane = item / p.strips, strip = item - plane * p.strips;
    const int img = plane / g.M, m = plane - img * g.M;
    uint32_t* rows = dw_lds + wave * p.wave_words;
    uint32_t* wk = rows + p.wave_words - g.KH * NWD;  // packed kernel rows, after the strip

    const int oh0 = strip * p.th, nrow = min(p.th, g.OH - oh0);
    const int ih0 = oh0 * g.sh - g.pt;
    const int irows = (nrow - 1) * g.sh + (g.KH - 1) * g.dh + 1;
    const uint8_t* xb = p.x + ((int64_t)img * g.C + m / p.mg) * ((int64_t)g.H * g.W);
    const uint32_t pad = (uint32_t)(uint8_t)p.zs * 0x01010101u;
    // The kernel rows and the strip's words: every load of a batch of U words
    // is issued before the first is used. A word that sticks out of its row is
    // read where it fits and shifted into place, one in a padded row is read
    // from the nearest row, and the mask keeps the padding.
    constexpr int U = 8;
    const int8_t* wr = p.w + (int64_t)m * p.ldw;
    const int32_t b0 = p.bias ? p.bias[m] : 0;
    const float mu = p.mult[m];
    const int words = irows * p.wpr;
    for (int i0 = lane; i0 < words; i0 += 64 * U) {
        uint32_t raw[U];
        int sh[U];  // bytes the word is shifted up (> 0) or down; 4: all padding
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = min(i0 + 64 * u, words - 1);
            const int r = (int)__umulhi((uint32_t)i, p.wpr_magic), c = (i - r * p.wpr) * 4 - p.left;
            const int ih = ih0 + r, ihc = min(max(ih, 0), g.H - 1), cc = min(max(c, 0), max(g.W - 4, 0));
            sh[u] = ih != ihc || cc - c > 3 || cc - c < -3 ? 4 : cc - c;
            const uint8_t* s = xb + (int64_t)ihc * g.W + cc;
            if (g.W >= 4) {
                __builtin_memcpy(&raw[u], s, 4);
            } else {  // rows of 1..3 bytes
                raw[u] = s[0];
                if (g.W > 1) raw[u] |= (uint32_t)s[1] << 8;
                if (g.W > 2) raw[u] |= (uint32_t)s[2] << 16;
            }
        }
        const uint32_t in_row = g.W >= 4 ? 0xFFFFFFFFu : (1u << (8 * g.W)) - 1;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int up = max(sh[u], 0) * 8, down = max(-sh[u], 0) * 8;
            const uint32_t mask = sh[u] == 4 ? 0u : (in_row << up) >> down;
            const uint32_t v = sh[u] == 4 ? 0u : ((raw[u] ^ p.flip) << up) >> down;
            if (i0 + 64 * u < words) rows[i0 + 64 * u] = (v & mask) | (pad & ~mask);
        }
    }
    for (int i = lane; i < g.KH * NWD; i += 64) {
        const int kh = i / NWD, k0 = (i - kh * NWD) * 4;
        uint32_t v = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (k0 + e < g.KW) v |= (uint32_t)(uint8_t)wr[kh * g.KW + k0 + e] << (8 * e);
        wk[i] = v;
    }
    // the slice belongs to this wave alone and its LDS operations complete in order
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

    for (int i = lane; i < nrow * p.qpr; i += 64) {
        const int orow = p.qpr == 1 ? i : (int)__umulhi((uint32_t)i, p.qpr_magic), ow = (i - orow * p.qpr) * 4;
        const int sw = SW ? SW : g.sw;
        const int byte0 = ow * sw - g.pl + p.left;
        int acc[4] = {0, 0, 0, 0}, wsum = 0;
        for (int kh = 0; kh < g.KH; ++kh) {
            const uint32_t* lr = rows + (orow * g.sh + kh * g.dh) * p.wpr;
            int wd[NWD];
#pragma unroll
            for (int d = 0; d < NWD; ++d) {
                wd[d] = (int)wk[kh * NWD + d];
                wsum = __builtin_amdgcn_sdot4(wd[d], 0x01010101, wsum, false);
            }
            if constexpr (SW != 0) {
                constexpr int NV = NWD + (3 * SW + 3) / 4;  // words from byte0 that the four windows cover
                const uint32_t* q = lr + (byte0 >> 2);
                uint32_t raw[NV + 1], v[NV];
#pragma unroll
                for (int d = 0; d <= NV; ++d) raw[d] = q[d];
#pragma unroll
                for (int d = 0; d < NV; ++d) v[d] = __builtin_amdgcn_alignbyte(raw[d + 1], raw[d], byte0 & 3);
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int d = 0; d < NWD; ++d) {
                        const int o = (e * SW) >> 2, sh = (e * SW) & 3;
                        const uint32_t xw = sh ? __builtin_amdgcn_alignbyte(v[o + d + 1], v[o + d], sh) : v[o + d];
                        acc[e] = __builtin_amdgcn_sdot4((int)xw, wd[d], acc[e], false);
                    }
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int be = min(ow + e, g.OW - 1) * sw - g.pl + p.left;
#pragma unroll
                    for (int d = 0; d < NWD; ++d) {
                        const uint32_t* q = lr + (be >> 2) + d;
                        acc[e] = __builtin_amdgcn_sdot4((int)__builtin_amdgcn_alignbyte(q[1], q[0], be & 3), wd[d], acc[e],
                                                        false);
                    }
                }
            }
        }
        const int32_t corr = wrap_add(wrap_mul(wsum, -p.zs), b0);
        uint32_t out = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            out |= (uint32_t)requant_byte(wrap_add(acc[e], corr), mu, p.zy, p.y_u8) << (8 * e);
        uint8_t* yo = p.y + ((int64_t)plane * g.OH + oh0 + orow) * g.OW + ow;
        if (ow + 3 < g.OW) {
            __builtin_memcpy(yo, &out, 4);
        } else {
            for (int e = 0; e < g.OW - ow; ++e) yo[e] = (uint8_t)(out >> (8 * e));
        }
    }
}

// LDS bytes of a workgroup (4 waves) of the depthwise kernel.
constexpr int DW_LDS = 64 * 1024;

}  // namespace

hipError_t launch_qconv_depthwise(const void* x, int x_u8, const QconvGeom& g, const int8_t* w, int64_t ldw,
                                  const int32_t* bias, const float* mult, int32_t zx, float zy, int y_u8, void* y,
                                  hipStream_t st, int against, bool* done) {
    *done = false;
    const bool any = against == 2;
    // what the kernel's windows and 16-bit index arithmetic hold; anything else is the direct kernel's
    if (g.Cg != 1 || g.KW > 8 || g.dw != 1 || g.KH > 64 || g.W >= (1 << 15) || g.OW >= (1 << 15) || g.pl >= (1 << 12) ||
        g.sw > (1 << 10) || (int64_t)g.N * g.M >= (1 << 30))
        return hipSuccess;
    QdwArgs p;
    p.x = (const uint8_t*)x, p.w = w, p.bias = bias, p.mult = mult, p.y = (uint8_t*)y, p.ldw = ldw, p.g = g;
    p.mg = g.M / g.G;
    p.flip = x_u8 ? 0x80808080u : 0u;
    p.zs = x_u8 ? zx - 128 : zx;
    p.zy = zy, p.y_u8 = y_u8;
    p.planes = g.N * g.M;
    p.left = (g.pl + 3) & ~3;
    const int nwd = g.KW <= 4 ? 1 : 2;
    p.qpr = (g.OW + 3) / 4;
    // last byte a window touches: the last group of 4 outputs' first byte, its 3 strides, the words read from there
    const int64_t span = (int64_t)(p.qpr * 4 - 1) * g.sw - g.pl + p.left + 4 * nwd + 8;
    const int64_t cols = std::max<int64_t>(p.left + g.W, span);
    if (cols >= (1 << 16)) return hipSuccess;
    p.wpr = (int)((cols + 3) / 4);
    // Strip height: 1024 outputs (four groups of 4 per lane) or the plane,
    // shorter where the rows it reads would overrun the wave's LDS.
    const auto irows = [&](int th) { return (int64_t)(th - 1) * g.sh + (int64_t)(g.KH - 1) * g.dh + 1; };
    const auto words = [&](int th) { return irows(th) * p.wpr + 4 + g.KH * nwd; };
    int th = (int)std::min<int64_t>(g.OH, std::max(1, 1024 / std::max(1, p.qpr * 4)));
    while (th > 1 && words(th) * 16 > DW_LDS) th = (th + 1) / 2;
    if (words(th) * 16 > DW_LDS || irows(th) * p.wpr >= (1 << 16) || (int64_t)th * p.qpr >= (1 << 16)) return hipSuccess;
    p.strips = (g.OH + th - 1) / th;
    p.th = th = (g.OH + p.strips - 1) / p.strips;  // strips of about one height
    p.wave_words = (int)words(th);
    const auto magic = [](int d) { return (uint32_t)((((uint64_t)1 << 32) + d - 1) / d); };  // d = 1 is not divided
    p.wpr_magic = magic(p.wpr);
    p.qpr_magic = magic(p.qpr);
    const int64_t items = (int64_t)p.planes * p.strips;
    if (items >= (1ll << 26) || p.wpr < 2) return hipSuccess;  // 64 threads an item: the grid stays below 2^32
    const dim3 grid((unsigned)((items + 3) / 4));
    const size_t lds = (size_t)p.wave_words * 16;
    // whole 8-byte row pieces, indexes the magic division holds
    p.ipp = (uint32_t)p.qpr * (uint32_t)((g.OH + 3) / 4);
    const int64_t blocks4 = (int64_t)p.planes * p.ipp;
    // (one output row at stride 2 leaves three quarters of a lane's rows unused: 32768 planes of 2 × 8, 3 × 3 4.7 µs,
    // 4.2 in the direct kernel)
    if (g.KH == g.KW && (g.KH == 3 || g.KH == 5) && g.sh == g.sw && g.sw <= 2 && g.dh == 1 && g.W >= 8 &&
        (any || g.sw == 1 || g.OH > 1) && (int64_t)p.qpr * ((g.OH + 3) / 4) + 256 < (1 << 16) && blocks4 < (1ll << 31)) {
        p.ipp_magic = magic((int)p.ipp);
        const dim3 bg((unsigned)((blocks4 + 255) / 256));
        if (g.KH == 3 && g.sw == 1) hipLaunchKernelGGL((qconv_dw_block_kernel<1, 3>), bg, dim3(256), 0, st, p);
        else if (g.KH == 3) hipLaunchKernelGGL((qconv_dw_block_kernel<2, 3>), bg, dim3(256), 0, st, p);
        else if (g.sw == 1) hipLaunchKernelGGL((qconv_dw_block_kernel<1, 5>), bg, dim3(256), 0, st, p);
        else hipLaunchKernelGGL((qconv_dw_block_kernel<2, 5>), bg, dim3(256), 0, st, p);
        *done = true;
        return hipGetLastError();
    }
    // A strip costs a wave about 0.8 ns of the chip and 5–6 µs from launch to
    // store however little it holds; the direct kernel about 6 ps + 0.44 ps a tap
    // and output, and 3 µs + 0.12 a tap. So the strip kernel takes what holds
    // enough products per strip and per call, and a stride only with the taps
    // that pay for the input it skips (MI355X, strip / direct µs: 30720 planes of
    // 7 × 7, 3 × 3 25.4 / 16.0, 5 × 5 30.5 / 25.1, 24576 of 7 × 7, 7 × 7 26.6 / 32.5;
    // 32768 of 1 × 1 26.3 / 3.5; 32 of 28 × 28, 1 × 1 6.5 / 3.1, 768 of 56 × 56 8.0 /
    // 14.0; 2 × 2 stride 2, 56 × 56 10.7 / 7.0, 4 × 4 10.8 / 11.4; 512 of 112 × 112
    // stride 3, 3 × 3 11.9 / 10.3, 7 × 7 16.5 / 31.0).
    const int64_t taps = (int64_t)g.KH * g.KW, outs = (int64_t)p.th * g.OW;
    // Few strips run at their latency, 5.4 µs + 0.8 ns each, which 3 µs + 0.12 a tap of the direct kernel exceed unless most
    // taps lie outside the image: up to 150·taps − 3000 strips, and 4096 of 25 outputs and more (672 planes of 7 × 7, 5 × 5
    // 5.4 / 6.0; 7 × 7 stride 2 on 7 × 7 6.6 / 9.2, on 4 × 4 6.6 / 7.9; 3840 of 4 × 4, 7 × 7 8.1 / 9.3, 5 × 5 7.6 / 5.9; 672
    // of 3 × 3, 7 × 7 7.6 / 6.9).
    const bool few = taps >= 24 && std::min(g.H, g.W) >= 4 && (items <= 150 * taps - 3000 || (outs >= 25 && items <= 4096));
    if (!any && ((outs * (13 + taps) < 2000 && !few) ||
                 (int64_t)p.planes * g.OH * g.OW * (13 + taps) + 284000 * taps < 6800000 ||
                 taps < 16 * (int64_t)(std::max(g.sh, g.sw) - 1)))
        return hipSuccess;
    // Channel multipliers of 16 and more have the GEMM, too: it is ahead where the strips are too few for the chip,
    // or small while each channel has enough outputs to fill its tiles (strip / GEMM µs, 7 × 7: 1 × 1 × 224 × 224 → 32
    // stride 2 11.6 / 9.7, 8 images 19.9 / 31.8; 4 × 1 × 64 × 64 → 64 9.1 / 11.1, stride 2 11.5 / 8.3; 1 × 64 × 28 × 28 →
    // 1024 10.0 / 18.3; 32 × 4 × 14 × 14 → 512 20.2 / 18.0, stride 2 19.5 / 11.6; 8 × 1 × 224 × 224 → 32 stride 4 16.6 /
    // 13.8).
    if (against == 1 && (items < 1024 || std::max(g.sh, g.sw) > 3 || (p.mg >= 64 && outs < 400))) return hipSuccess;
#define INGOT_DW(SW, NWD) hipLaunchKernelGGL((qconv_dw_kernel<SW, NWD>), grid, dim3(256), lds, st, p)
    if (nwd == 1) {
        if (g.sw == 1) INGOT_DW(1, 1);
        else if (g.sw == 2) INGOT_DW(2, 1);
        else INGOT_DW(0, 1);
    } else {
        if (g.sw == 1) INGOT_DW(1, 2);
        else if (g.sw == 2) INGOT_DW(2, 2);
        else INGOT_DW(0, 2);
    }
#undef INGOT_DW
    *done = true;
    return hipGetLastError();
}

hipError_t launch_qim2col(const void* x, const QconvGeom& g, int rows, int kg, int kgl, uint8_t pad, void* col,
                          int64_t col_group, hipStream_t st) {
    if (rows <= 0) return hipSuccess;
    const int64_t threads = (int64_t)rows * (kgl / 16);
    const int64_t blocks = (threads + 255) / 256;
    hipLaunchKernelGGL(qim2col_kernel, dim3((unsigned)blocks, (unsigned)g.G), dim3(256), 0, st, (const uint8_t*)x, g,
                       rows, kg, kgl, pad, (uint8_t*)col, col_group);
    return hipGetLastError();
}

hipError_t launch_qconv_layout(const void* x, const QconvGeom& g, int images, int hp, int wp, int cgp, uint8_t pad,
                               int x_u8, void* xt, const int8_t* w, int64_t ldw, int64_t ldp, int8_t* wt, hipStream_t st) {
    QlayoutArgs p;
    p.x = (const uint8_t*)x, p.xt = (uint8_t*)xt, p.w = w, p.wt = wt, p.g = g;
    p.hp = hp, p.wp = wp, p.cgp = cgp, p.ldw = ldw, p.ldp = ldp;
    p.ctiles = (g.G * cgp + 63) / 64;
    p.wtiles = (wp + 63) / 64;
    p.x_blocks = (int64_t)images * hp * p.wtiles * p.ctiles;
    p.w_chunks = (int64_t)g.M * g.KH * g.KW * (cgp / 16);
    p.pad = pad * 0x01010101u;
    p.flip = x_u8 ? 0x80808080u : 0u;
    const int64_t blocks = p.x_blocks + (p.w_chunks + 255) / 256;
    if (blocks >= (1 << 24)) return hipErrorInvalidValue;  // 256 threads each: the grid stays below 2^32
    hipLaunchKernelGGL(qconv_layout_kernel, dim3((unsigned)blocks), dim3(256), 0, st, p);
    return hipGetLastError();
}

hipError_t launch_qconv_direct(const void* x, int x_u8, const QconvGeom& g, const int8_t* w, int64_t ldw,
                               const int32_t* bias, const float* mult, int32_t zx, float zy, int y_u8, void* y,
                               hipStream_t st) {
    const int64_t total = (int64_t)g.N * g.M * g.OH * g.OW;
    if (total <= 0) return hipSuccess;
    const int64_t blocks = std::min<int64_t>((total + 255) / 256, 16384);
    hipLaunchKernelGGL(qconv_direct_kernel, dim3((unsigned)blocks), dim3(256), 0, st, (const uint8_t*)x, x_u8, g, w,
                       ldw, bias, mult, zx, zy, y_u8, (uint8_t*)y, total);
    return hipGetLastError();
}

}  // namespace ingot
