// Memory-bound helper kernels: weight and activation packing, DequantizeLinear,
// the standalone activation / bias pass, the f32 → bf16 cast and fills.

#include <algorithm>
#include <type_traits>

#include "kernels.hpp"

namespace ingot {

namespace {

inline unsigned grid_for(int64_t work, int per_block) {
    int64_t b = (work + per_block - 1) / per_block;
    if (b > (1 << 20)) b = 1 << 20;
    if (b < 1) b = 1;
    return (unsigned)b;
}

// One wave per row: colsum[j] = Σ_k packed[j][k] (int32 wrap-around).
__global__ void colsum_kernel(const int8_t* packed, int64_t kp, int64_t ldk, int64_t n, int32_t* colsum) {
    const int64_t j = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (j >= n) return;
    uint32_t s = 0;
    for (int64_t k = lane; k < kp; k += 64) s += (uint32_t)(int32_t)packed[j * ldk + k];
    for (int off = 32; off > 0; off >>= 1) s += (uint32_t)__shfl_xor((int)s, off);
    if (lane == 0) colsum[j] = (int32_t)s;
}

// ---- operand packs ----
// One operand matrix (a weight, or a call's activations) becomes rows of the
// destination kind, k-contiguous, zero past n rows and past k columns. The
// element types a kind is packed from: S is the source element, D the
// destination's 16-byte chunk of EPC elements.
template <int KD> struct PackOf { static constexpr int EPC = KD == KIND_F32 ? 4 : (KD == KIND_I8 ? 16 : 8); };

struct PackArgs {
    const void* src;
    int64_t ld;          // source row pitch, elements
    int64_t n, k;        // logical rows and columns of the destination
    void* dst;
    int64_t np, kp, ldk; // written rows and columns (kp a multiple of the chunk), row pitch, elements
    int64_t plane;       // KIND_BF16X2: elements from the hi plane to the lo plane
    int64_t src_item, dst_item;  // elements between batch items (blockIdx.y)
    uint32_t flip;       // KIND_I8: XOR of every source byte inside the matrix (0x80: u8 → s8)
};

// EPC consecutive elements from p, the first `have` of them inside the matrix
// (the rest are zero), as f32 (bits kept for a bf16 → bf16 copy) or bytes.
template <int KD, typename S>
struct Chunk {
    static constexpr int EPC = PackOf<KD>::EPC;
    S v[EPC];
    __device__ __forceinline__ void load(const S* p, int64_t have) {
        constexpr int BYTES = EPC * (int)sizeof(S);
        constexpr int VB = BYTES >= 16 ? 16 : BYTES;
        if (have >= EPC && (((uintptr_t)p) & (VB - 1)) == 0) {
            if constexpr (VB == 16) {
                i32x4_t t[BYTES / 16];
#pragma unroll
                for (int i = 0; i < BYTES / 16; ++i) t[i] = ((const i32x4_t*)p)[i];
                __builtin_memcpy(v, t, BYTES);
            } else {
                const uint2 t = *(const uint2*)p;
                __builtin_memcpy(v, &t, 8);
            }
        } else {
#pragma unroll
            for (int e = 0; e < EPC; ++e) v[e] = e < have ? p[e] : S(0);
        }
    }
};

__device__ __forceinline__ float pack_f32(float v) { return v; }
__device__ __forceinline__ float pack_f32(uint16_t v) { return bf16_to_f32(v); }
__device__ __forceinline__ uint16_t pack_bf16(float v) { return f32_to_bf16(v); }
__device__ __forceinline__ uint16_t pack_bf16(uint16_t v) { return v; }

// Writes one chunk (kept inside the matrix by `live` elements for the byte flip).
template <int KD, typename S>
__device__ __forceinline__ void store_chunk(const S (&v)[PackOf<KD>::EPC], int64_t live, const PackArgs& p, char* d) {
    constexpr int EPC = PackOf<KD>::EPC;
    i32x4_t out;
    if constexpr (KD == KIND_I8) {
        uint8_t b[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) b[e] = e < live ? (uint8_t)(v[e] ^ p.flip) : (uint8_t)0;
        __builtin_memcpy(&out, b, 16);
        *(i32x4_t*)d = out;
    } else if constexpr (KD == KIND_F32) {
        float f[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) f[e] = pack_f32(v[e]);
        __builtin_memcpy(&out, f, 16);
        *(i32x4_t*)d = out;
    } else {
        uint16_t h[EPC], l[EPC];
#pragma unroll
        for (int e = 0; e < EPC; ++e) {
            if constexpr (KD == KIND_BF16X2)
                split_bf16(pack_f32(v[e]), h[e], l[e]);
            else
                h[e] = pack_bf16(v[e]);
        }
        __builtin_memcpy(&out, h, 16);
        *(i32x4_t*)d = out;
        if constexpr (KD == KIND_BF16X2) {
            __builtin_memcpy(&out, l, 16);
            *(i32x4_t*)(d + p.plane * 2) = out;
        }
    }
}

template <int KD> constexpr int pack_esz() { return KD == KIND_F32 ? 4 : (KD == KIND_I8 ? 1 : 2); }

// Source rows are k-contiguous ([n][k]): a thread converts one 16-byte chunk
// of a destination row, 2^txs threads side by side on a row and 256 >> txs
// rows per workgroup, so short rows (an attention head) fill a workgroup too
// and no thread divides. Few long rows are spread over gridDim.z workgroups
// each: with one per row, the chunks of a thread follow one another at a load's
// latency (the hi/lo planes of 64 × 11008 took 10.3 µs on MI355X, 5.8 spread; of 17 ×
// 11008 7.9 and 4.9; bf16 of 128 × 11008 7.0 and 5.4).
template <int KD, typename S>
__global__ __launch_bounds__(256) void pack_rows_kernel(PackArgs p, int txs) {
    constexpr int EPC = PackOf<KD>::EPC;
    const int tx = threadIdx.x & ((1 << txs) - 1), ty = threadIdx.x >> txs;
    const int rows = 256 >> txs;
    const S* src = (const S*)p.src + (int64_t)blockIdx.y * p.src_item;
    char* dst = (char*)p.dst + (int64_t)blockIdx.y * p.dst_item * pack_esz<KD>();
    for (int64_t j = (int64_t)blockIdx.x * rows + ty; j < p.np; j += (int64_t)gridDim.x * rows) {
        const int64_t kin = j < p.n ? p.k : 0;
        for (int64_t k0 = ((int64_t)blockIdx.z << txs | tx) * EPC; k0 < p.kp; k0 += (int64_t)gridDim.z * EPC << txs) {
            Chunk<KD, S> c;
            c.load(src + j * p.ld + k0, kin - k0);
            store_chunk<KD, S>(c.v, kin - k0, p, dst + (j * p.ldk + k0) * pack_esz<KD>());
        }
    }
}

// Source rows are n-contiguous ([k][n]): tiles of 64 n × 64 k (32 k of f32)
// transposed through LDS, so that both the reads (along n) and the writes
// (16-byte chunks along k) are whole lines. Bound by its latency at the sizes of
// attention heads: one element a thread, read straight into its padded place,
// the pack took 18.2 µs for 96 items of 128 × 64 f32 (2.4 MB) on MI355X, 64 × 64
// tiles 5.7, 64 × 32 ones (twice the workgroups) 5.1; with this kernel and the
// items' own rows only, Q·Kᵀ (read in place) and P·V of 96 heads of 128 × 64 went
// from 48.0 to 19.0 µs together.
template <typename S>
constexpr int pack_tk() {
    return sizeof(S) == 4 ? 32 : 64;
}
template <int KD, typename S>
__global__ __launch_bounds__(256) void pack_cols_kernel(PackArgs p, int64_t tiles, int tiles_k) {
    constexpr int EPC = PackOf<KD>::EPC;
    constexpr int T = 64, TK = pack_tk<S>();
    // row pitch in elements: an odd number of 4-byte words
    constexpr int PITCH = TK + (sizeof(S) == 4 ? 1 : (sizeof(S) == 2 ? 2 : 4));
    __shared__ S tile[T * PITCH];
    const S* src = (const S*)p.src + (int64_t)blockIdx.y * p.src_item;
    char* dst = (char*)p.dst + (int64_t)blockIdx.y * p.dst_item * pack_esz<KD>();
    const int tid = threadIdx.x;
    for (int64_t t = blockIdx.x; t < tiles; t += gridDim.x) {
        const int64_t j0 = t / tiles_k * T, k0 = t % tiles_k * TK;
        // 4 n of one k per thread and step: 16 threads a source row, 16 rows a step
        const int n4 = (tid & 15) * 4, kr = tid >> 4;
#pragma unroll
        for (int i = 0; i < TK / 16; ++i) {
            const int kk = kr + i * 16;
            const int64_t have = k0 + kk < p.k ? p.n - (j0 + n4) : 0;
            const S* s = src + (k0 + kk) * p.ld + j0 + n4;
            S v[4];
            if (have >= 4 && (((uintptr_t)s) & (4 * sizeof(S) - 1)) == 0) {
                if constexpr (sizeof(S) == 4) {
                    const i32x4_t w = *(const i32x4_t*)s;
                    __builtin_memcpy(v, &w, 16);
                } else if constexpr (sizeof(S) == 2) {
                    const uint2 w = *(const uint2*)s;
                    __builtin_memcpy(v, &w, 8);
                } else {
                    const uint32_t w = *(const uint32_t*)s;
                    __builtin_memcpy(v, &w, 4);
                }
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = e < have ? s[e] : S(0);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) tile[(n4 + e) * PITCH + kk] = v[e];
        }
        __syncthreads();
        constexpr int CPR = TK / EPC;  // chunks of a tile row
        for (int c = tid; c < T * CPR; c += 256) {
            const int jj = c / CPR, kc = c % CPR * EPC;
            const int64_t j = j0 + jj, k = k0 + kc;
            if (j >= p.np || k >= p.kp) continue;
            S v[EPC];
#pragma unroll
            for (int e = 0; e < EPC; ++e) v[e] = tile[jj * PITCH + kc + e];
            store_chunk<KD, S>(v, j < p.n ? p.k - k : 0, p, dst + (j * p.ldk + k) * pack_esz<KD>());
        }
        __syncthreads();
    }
}

// rows: the source is [n][k], else [k][n].
template <int KD, typename S>
hipError_t launch_pack(const PackArgs& p, bool rows, int items, hipStream_t st) {
    if (p.np <= 0 || p.kp <= 0) return hipSuccess;
    if (rows) {
        int txs = 0;
        while (txs < 8 && ((int64_t)PackOf<KD>::EPC << txs) < p.kp) ++txs;
        // one step of 256 chunks a workgroup, until the chip has enough of them (eight workgroups a CU)
        const int64_t wgs = (int64_t)grid_for(p.np, 256 >> txs) * items, steps = (p.kp / PackOf<KD>::EPC + (1 << txs) - 1) >> txs;
        const unsigned spread = (unsigned)std::max<int64_t>(1, std::min(steps, 2048 / wgs));
        hipLaunchKernelGGL((pack_rows_kernel<KD, S>), dim3(grid_for(p.np, 256 >> txs), items, spread), dim3(256), 0, st, p,
                           txs);
    } else {
        const int64_t tiles_k = (p.kp + pack_tk<S>() - 1) / pack_tk<S>(), tiles = (p.np + 63) / 64 * tiles_k;
        hipLaunchKernelGGL((pack_cols_kernel<KD, S>), dim3(grid_for(tiles, 1), items), dim3(256), 0, st, p, tiles,
                           (int)tiles_k);
    }
    return hipGetLastError();
}

hipError_t launch_pack_kind(GemmKind kind, int src_dtype, const PackArgs& p, bool rows, int items, hipStream_t st) {
    switch (kind) {
        case KIND_F32:
            if (src_dtype == INGOT_DT_F32) return launch_pack<KIND_F32, float>(p, rows, items, st);
            if (src_dtype == INGOT_DT_BF16) return launch_pack<KIND_F32, uint16_t>(p, rows, items, st);
            break;
        case KIND_BF16:
            if (src_dtype == INGOT_DT_F32) return launch_pack<KIND_BF16, float>(p, rows, items, st);
            if (src_dtype == INGOT_DT_BF16) return launch_pack<KIND_BF16, uint16_t>(p, rows, items, st);
            break;
        case KIND_BF16X2:
            if (src_dtype == INGOT_DT_F32) return launch_pack<KIND_BF16X2, float>(p, rows, items, st);
            break;
        case KIND_I8:
            if (src_dtype == INGOT_DT_I8 || src_dtype == INGOT_DT_U8) return launch_pack<KIND_I8, uint8_t>(p, rows, items, st);
            break;
        default: break;
    }
    return hipErrorInvalidValue;
}

// The common activation pack — f32 rows already dense in whole k-tiles (lda = k = kl, one batch
// item), to bf16 (or the hi/lo planes) — as a flat stream: each thread converts U groups of 8
// elements per step, all U loads issued before any conversion, over a grid of a few workgroups
// per CU (grid-stride), so that the copy runs at streaming rate instead of one small workgroup
// per 2048 elements.
template <int KD, int U>
__global__ __launch_bounds__(256) void pack_a_flat_kernel(const float* __restrict__ src, uint16_t* __restrict__ dst,
                                                          int64_t groups, int64_t plane) {
    const int64_t stride = (int64_t)gridDim.x * 256 * U;
    for (int64_t g0 = (int64_t)blockIdx.x * 256 * U + threadIdx.x; g0 < groups; g0 += stride) {
        f32x4_t v[U][2];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t g = g0 + (int64_t)u * 256;
            if (g < groups) {
                v[u][0] = __builtin_nontemporal_load((const f32x4_t*)(src + g * 8));
                v[u][1] = __builtin_nontemporal_load((const f32x4_t*)(src + g * 8 + 4));
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t g = g0 + (int64_t)u * 256;
            if (g >= groups) continue;
            uint16_t h[8], l[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float x = v[u][e >> 2][e & 3];
                if (KD == KIND_BF16X2)
                    split_bf16(x, h[e], l[e]);
                else
                    h[e] = f32_to_bf16(x);
            }
            i32x4_t out;
            __builtin_memcpy(&out, h, 16);
            *(i32x4_t*)(dst + g * 8) = out;
            if (KD == KIND_BF16X2) {
                __builtin_memcpy(&out, l, 16);
                *(i32x4_t*)(dst + plane + g * 8) = out;
            }
        }
    }
}

// ---- elementwise passes ----
// A thread takes V neighbouring elements of the flat tensor, loaded and stored
// together at any element alignment. HBM-bound when large, by launch and load
// latency when small. A per-axis operand (scale, zero point, bias) costs two
// multiplications by a reciprocal per V elements, and its loads wait for nothing
// but the index, like the element's own. V is 4 where that fills the chip,
// else 1, which is done sooner (400 × 100 int32 per column 2.5 µs on MI355X, 2.9
// with four). DequantizeLinear and the GELU of its result, kernel times on
// MI355X: 4000 × 4000 int8 per row 15.0 and 19.7 µs (one element a thread with
// a 64-bit division each 38.6 and 30.9; a grid over rows and columns 17.9 and
// 20.6), 1024 × 3072 int32 per column 8.0 and 6.4 (9.5 and 8.1; 8.5 and 7.1),
// 100000 × 7 int32 per row 3.0 and 3.0 (3.8 and 3.4; 4.8 and 3.7), 4096 × 65 per
// column 2.7 and 2.6 (2.9 and 2.6; 3.2 and 3.0).

// Which of `count` operands element i takes: (i / inner) % count. Below 2^31
// elements both quotients are exact as the upper half of a product with
// ceil(2^(31 + l) / d), l = ceil(log2 d), shifted by l − 1 (Granlund and
// Montgomery); WIDE divides in 64 bits.
struct Axis {
    int64_t inner, count;
    uint32_t mi, mc;  // 0: a divisor of 1
    int si, sc;
    Axis(int64_t n, int64_t inner_, int64_t count_)
        : inner(std::min(std::max<int64_t>(inner_, 1), n)), count(std::min(count_, n)) {
        reciprocal(inner, &mi, &si);
        reciprocal(count, &mc, &sc);
    }
    static void reciprocal(int64_t d, uint32_t* m, int* s) {
        int l = 0;
        while (l < 31 && ((int64_t)1 << l) < d) ++l;
        *m = l ? (uint32_t)((((uint64_t)1 << (31 + l)) + d - 1) / d) : 0u;
        *s = l ? l - 1 : 0;
    }
};

// The operand index of element i and of the elements after it.
template <bool WIDE>
struct AxisAt {
    typedef std::conditional_t<WIDE, int64_t, uint32_t> I;
    I c, r;
    __device__ __forceinline__ AxisAt(const Axis& a, int64_t i) {
        if constexpr (WIDE) {
            const int64_t q = i / a.inner;
            r = i - q * a.inner, c = q % a.count;
        } else {
            const uint32_t u = (uint32_t)i;
            const uint32_t q = a.mi ? __umulhi(u, a.mi) >> a.si : u;
            r = u - q * (uint32_t)a.inner;
            c = q - (a.mc ? __umulhi(q, a.mc) >> a.sc : q) * (uint32_t)a.count;
        }
    }
    __device__ __forceinline__ void next(const Axis& a) {
        if (++r == (I)a.inner) {
            r = 0;
            if (++c == (I)a.count) c = 0;
        }
    }
};

struct Grid1 {
    int v;
    unsigned blocks;
    explicit Grid1(int64_t n) : v(n >> 19 ? 4 : 1), blocks(grid_for(n, 256 * v)) {}
};

// body(width, index of the first element): this thread's chunks of V, and the elements of a short last one singly (a
// chunk that may be short would be loaded in pieces).
template <int V, typename Body>
__device__ __forceinline__ void walk(int64_t n, Body body) {
    const int64_t step = (int64_t)gridDim.x * 256 * V;
    for (int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * V; i < n; i += step) {
        if (V == 1 || i + V <= n) {
            body(std::integral_constant<int, V>(), i);
        } else {
            for (; i < n; ++i) body(std::integral_constant<int, 1>(), i);
        }
    }
}

// z[e] = zero point c[e].
template <int W, typename Z, typename I>
__device__ __forceinline__ void load_zp(int32_t (&z)[W], const void* zp, const I (&c)[W]) {
#pragma unroll
    for (int e = 0; e < W; ++e) z[e] = (int32_t)((const Z*)zp)[c[e]];
}

// AXIS 0: one scale for all; 1: per axis; 2: per axis, 2^31 elements or more.
template <typename T, int AXIS, int V>
__global__ __launch_bounds__(256) void dequant_kernel(const T* x, int64_t n, const float* scale, Axis axis,
                                                      const void* zp, int zp_dt, int zp_each, float* y) {
    walk<V>(n, [&](auto width, int64_t i) {
        constexpr int W = decltype(width)::value;
        T v[W];
        __builtin_memcpy(v, x + i, sizeof v);
        // operand indexes of the elements
        std::conditional_t<AXIS == 2, int64_t, uint32_t> c[W] = {};
        if constexpr (AXIS != 0) {
            AxisAt<AXIS == 2> at(axis, i);
#pragma unroll
            for (int e = 0; e < W; ++e) c[e] = at.c, at.next(axis);
        }
        float sc[W];
#pragma unroll
        for (int e = 0; e < W; ++e) sc[e] = scale[c[e]];
        int32_t z[W] = {};
        if (zp) {
            if (AXIS != 0 && !zp_each) {
#pragma unroll
                for (int e = 0; e < W; ++e) c[e] = 0;
            }
            if (zp_dt == INGOT_DT_U8) load_zp<W, uint8_t>(z, zp, c);
            else if (zp_dt == INGOT_DT_I8) load_zp<W, int8_t>(z, zp, c);
            else load_zp<W, int32_t>(z, zp, c);
        }
        float f[W];
#pragma unroll
        for (int e = 0; e < W; ++e) f[e] = (float)wrap_add((int32_t)v[e], -z[e]) * sc[e];
        __builtin_memcpy(y + i, f, sizeof f);
    });
}

// y = post(act(x + bias[column])), bias optional (WIDE: 2^31 elements or more).
template <int ACT, bool WIDE, int V>
__global__ __launch_bounds__(256) void activation_kernel(const float* x, float* y, int64_t n, const float* bias, Axis axis,
                                                         float a, float b, int post, float ps, float pb) {
    walk<V>(n, [&](auto width, int64_t i) {
        constexpr int W = decltype(width)::value;
        float v[W];
        __builtin_memcpy(v, x + i, sizeof v);
        if (bias) {
            AxisAt<WIDE> at(axis, i);
#pragma unroll
            for (int e = 0; e < W; ++e) v[e] += bias[at.c], at.next(axis);
        }
#pragma unroll
        for (int e = 0; e < W; ++e) {
            if (ACT != INGOT_ACT_NONE) v[e] = apply_act(v[e], ACT, a, b);
            if (post) v[e] = v[e] * ps + pb;
        }
        __builtin_memcpy(y + i, v, sizeof v);
    });
}

template <int V>
__global__ __launch_bounds__(256) void cast_bf16_kernel(const float* x, uint16_t* y, int64_t n) {
    walk<V>(n, [&](auto width, int64_t i) {
        constexpr int W = decltype(width)::value;
        float v[W];
        __builtin_memcpy(v, x + i, sizeof v);
        uint16_t h[W];
#pragma unroll
        for (int e = 0; e < W; ++e) h[e] = f32_to_bf16(v[e]);
        __builtin_memcpy(y + i, h, sizeof h);
    });
}

// 16 bytes a thread and step; the bytes before the first and after the last aligned 16 one at a time.
__global__ void fill_kernel(uint8_t* d, uint8_t v, size_t bytes) {
    const size_t tid = blockIdx.x * (size_t)blockDim.x + threadIdx.x, threads = (size_t)gridDim.x * blockDim.x;
    const size_t head = min((size_t)(-(uintptr_t)d & 15), bytes), body = (bytes - head) / 16;
    const uint32_t w = v * 0x01010101u;
    for (size_t i = tid; i < body; i += threads) ((uint4*)(d + head))[i] = make_uint4(w, w, w, w);
    const size_t rest = bytes - body * 16;  // the head and the tail
    for (size_t i = tid; i < rest; i += threads) d[i < head ? i : i + body * 16] = v;
}

}  // namespace

hipError_t launch_pack_weight(const void* src, int src_dtype, int64_t ld, int trans, int64_t n, int64_t k, void* dst,
                              GemmKind dst_kind, int64_t np, int64_t kp, int64_t ldk, hipStream_t st, int items,
                              int64_t src_item, int64_t dst_item) {
    const PackArgs p = {src, ld, n, k, dst, np, kp, ldk, 0, src_item, dst_item, 0u};
    return launch_pack_kind(dst_kind, src_dtype, p, trans != 0, items, st);
}

hipError_t launch_colsum_i8(const int8_t* packed, int64_t kp, int64_t ldk, int64_t n, int32_t* colsum,
                            hipStream_t st) {
    hipLaunchKernelGGL(colsum_kernel, dim3((unsigned)((n + 3) / 4)), dim3(256), 0, st, packed, kp, ldk, n, colsum);
    return hipGetLastError();
}

hipError_t launch_pack_a(const void* src, int src_dtype, int64_t lda, int trans, int64_t m, int64_t k,
                         int64_t src_stride, void* dst, GemmKind dst_kind, int64_t kl, int64_t dst_stride, int batch,
                         hipStream_t st) {
    // (large activations only: at decode sizes the per-row grid below spreads the few rows over more CUs;
    // M = 16, K = 2048 took 5.4 us flat against 3.7)
    if ((dst_kind == KIND_BF16 || dst_kind == KIND_BF16X2) && src_dtype == INGOT_DT_F32 && !trans && batch == 1 &&
        lda == k && kl == k && k % 8 == 0 && m * k >= ((int64_t)1 << 22) && (((uintptr_t)src) & 15) == 0 &&
        (((uintptr_t)dst) & 15) == 0) {
        const int64_t groups = m * k / 8;
        const int64_t need = (groups + 256 * 4 - 1) / (256 * 4);
        const unsigned grid = (unsigned)std::max<int64_t>(1, std::min<int64_t>(need, 2048));
        if (dst_kind == KIND_BF16)
            hipLaunchKernelGGL((pack_a_flat_kernel<KIND_BF16, 4>), dim3(grid), dim3(256), 0, st, (const float*)src,
                               (uint16_t*)dst, groups, m * kl);
        else
            hipLaunchKernelGGL((pack_a_flat_kernel<KIND_BF16X2, 4>), dim3(grid), dim3(256), 0, st, (const float*)src,
                               (uint16_t*)dst, groups, m * kl);
        return hipGetLastError();
    }
    const PackArgs p = {src, lda, m, k, dst, m, kl, kl, m * kl, src_stride, dst_stride,
                        src_dtype == INGOT_DT_U8 ? 0x80u : 0u};
    return launch_pack_kind(dst_kind, src_dtype, p, trans == 0, batch, st);
}

hipError_t launch_dequant(const void* x, int x_dtype, int64_t n, const float* scale, int64_t n_scale, int64_t inner,
                          const void* zp, int zp_dtype, int64_t n_zp, float* y, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    const Grid1 g(n);
    const Axis axis(n, inner, n_scale);
    const auto launch = [&](auto kernel, auto t) {
        hipLaunchKernelGGL(kernel, dim3(g.blocks), dim3(256), 0, st, (const decltype(t)*)x, n, scale, axis, zp, zp_dtype,
                           n_zp > 1 ? 1 : 0, y);
        return hipGetLastError();
    };
    const auto go = [&](auto t) {
        typedef decltype(t) T;
        if (n_scale == 1) return g.v == 1 ? launch(dequant_kernel<T, 0, 1>, t) : launch(dequant_kernel<T, 0, 4>, t);
        if (n >> 31) return launch(dequant_kernel<T, 2, 4>, t);
        return g.v == 1 ? launch(dequant_kernel<T, 1, 1>, t) : launch(dequant_kernel<T, 1, 4>, t);
    };
    switch (x_dtype) {
        case INGOT_DT_U8: return go((uint8_t)0);
        case INGOT_DT_I8: return go((int8_t)0);
        case INGOT_DT_I32: return go((int32_t)0);
    }
    return hipErrorInvalidValue;
}

hipError_t launch_activation(const float* x, float* y, int64_t rows, int64_t cols, const float* bias, int act, float a,
                             float b, int post, float ps, float pb, hipStream_t st) {
    const int64_t n = rows * cols;
    if (n <= 0) return hipSuccess;
    const Grid1 g(n);
    const Axis axis(n, 1, cols);
    const auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(g.blocks), dim3(256), 0, st, x, y, n, bias, axis, a, b, post, ps, pb);
        return hipGetLastError();
    };
    switch (act) {
#define INGOT_ACT_CASE(A)                                      \
    case A:                                                    \
        return g.v == 1  ? launch(activation_kernel<A, false, 1>) \
               : n >> 31 ? launch(activation_kernel<A, true, 4>)  \
                         : launch(activation_kernel<A, false, 4>);
        INGOT_ACT_CASE(INGOT_ACT_NONE)
        INGOT_ACT_CASE(INGOT_ACT_RELU)
        INGOT_ACT_CASE(INGOT_ACT_GELU_ERF)
        INGOT_ACT_CASE(INGOT_ACT_GELU_TANH)
        INGOT_ACT_CASE(INGOT_ACT_SIGMOID)
        INGOT_ACT_CASE(INGOT_ACT_SILU)
        INGOT_ACT_CASE(INGOT_ACT_HARDSWISH)
        INGOT_ACT_CASE(INGOT_ACT_HARDSIGMOID)
        INGOT_ACT_CASE(INGOT_ACT_CLIP)
        INGOT_ACT_CASE(INGOT_ACT_LEAKYRELU)
#undef INGOT_ACT_CASE
    }
    return hipErrorInvalidValue;
}

hipError_t launch_cast_bf16(const float* x, uint16_t* y, int64_t n, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    const Grid1 g(n);
    if (g.v == 1)
        hipLaunchKernelGGL(cast_bf16_kernel<1>, dim3(g.blocks), dim3(256), 0, st, x, y, n);
    else
        hipLaunchKernelGGL(cast_bf16_kernel<4>, dim3(g.blocks), dim3(256), 0, st, x, y, n);
    return hipGetLastError();
}

hipError_t launch_fill(void* dst, int value, size_t bytes, hipStream_t st) {
    hipLaunchKernelGGL(fill_kernel, dim3(grid_for((int64_t)(bytes / 16 + 31), 256)), dim3(256), 0, st, (uint8_t*)dst,
                       (uint8_t)value, bytes);
    return hipGetLastError();
}

}  // namespace ingot
