// Memory-bound helper kernels: weight and activation packing, DequantizeLinear,
// the standalone activation / bias pass, the f32 → bf16 cast and fills.

#include <algorithm>

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
// and no thread divides.
template <int KD, typename S>
__global__ __launch_bounds__(256) void pack_rows_kernel(PackArgs p, int txs) {
    constexpr int EPC = PackOf<KD>::EPC;
    const int tx = threadIdx.x & ((1 << txs) - 1), ty = threadIdx.x >> txs;
    const int rows = 256 >> txs;
    const S* src = (const S*)p.src + (int64_t)blockIdx.y * p.src_item;
    char* dst = (char*)p.dst + (int64_t)blockIdx.y * p.dst_item * pack_esz<KD>();
    for (int64_t j = (int64_t)blockIdx.x * rows + ty; j < p.np; j += (int64_t)gridDim.x * rows) {
        const int64_t kin = j < p.n ? p.k : 0;
        for (int64_t k0 = (int64_t)tx * EPC; k0 < p.kp; k0 += (int64_t)EPC << txs) {
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
        hipLaunchKernelGGL((pack_rows_kernel<KD, S>), dim3(grid_for(p.np, 256 >> txs), items), dim3(256), 0, st, p, txs);
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
// A pass sees its tensor as rows × cols (the last row may be short: n counts
// the elements) with per-column or per-row operands, so that no element is
// divided for its index: 2^txs threads side by side on a row, V neighbouring
// elements each, loaded and stored together at any element alignment. HBM-bound:
// one element a thread with a 64-bit division and remainder for a per-axis
// scale, DequantizeLinear of 4000 × 4000 int8 per row took 53 µs on MI355X and
// the GELU of its result 31 µs; these take 27 and 21 µs. V is 4 where that
// fills the chip; small tensors take one element a thread, which is done
// sooner (400 × 100 int32 per column 2.6 µs, 2.9 with four).
struct Grid2 {
    int64_t n, rows, cols;
    int v, txs;
    Grid2(int64_t n_, int64_t cols_) : n(n_), rows((n_ + cols_ - 1) / cols_), cols(cols_), v(n_ >> 19 ? 4 : 1), txs(0) {
        while (txs < 8 && ((int64_t)v << txs) < cols) ++txs;
    }
    dim3 grid() const {
        const int64_t per = 256 >> txs;
        return dim3((unsigned)((((cols + v - 1) / v) + (1 << txs) - 1) >> txs),
                    (unsigned)std::min<int64_t>((rows + per - 1) / per, 65535));
    }
};

// This thread's first column; body(row, index of its first element, how many of the V are there) for its rows.
template <int V>
__device__ __forceinline__ int64_t first_col(int txs) {
    return (((int64_t)blockIdx.x << txs) + (threadIdx.x & ((1 << txs) - 1))) * V;
}
template <int V, typename Body>
__device__ __forceinline__ void walk_rows(int64_t n, int64_t rows, int64_t cols, int txs, int64_t col, Body body) {
    const int64_t step = (int64_t)gridDim.y * (256 >> txs);
    for (int64_t r = (int64_t)blockIdx.y * (256 >> txs) + (threadIdx.x >> txs); r < rows; r += step) {
        const int64_t i = r * cols + col;
        if (i < n) body(r, i, (int)min(min(cols - col, n - i), (int64_t)V));
    }
}

template <int V, typename T>
__device__ __forceinline__ void load_v(T (&v)[V], const T* p, int have) {
    if (have == V) {
        __builtin_memcpy(v, p, V * sizeof(T));
    } else {
#pragma unroll
        for (int e = 0; e < V; ++e)  // static indexes: v stays in registers
            if (e < have) v[e] = p[e];
    }
}
template <int V, typename T>
__device__ __forceinline__ void store_v(T* p, const T (&v)[V], int have) {
    if (have == V) {
        __builtin_memcpy(p, v, V * sizeof(T));
    } else {
#pragma unroll
        for (int e = 0; e < V; ++e)
            if (e < have) p[e] = v[e];
    }
}

__device__ __forceinline__ int32_t load_zp(const void* p, int dt, int64_t i) {
    switch (dt) {
        case INGOT_DT_U8: return (int32_t)((const uint8_t*)p)[i];
        case INGOT_DT_I8: return (int32_t)((const int8_t*)p)[i];
        default: return ((const int32_t*)p)[i];
    }
}

// COL: one scale (and zero point) per column; else one per row, row r taking r % n_scale.
template <typename T, bool COL, int V>
__global__ __launch_bounds__(256) void dequant_kernel(const T* x, int64_t n, int64_t rows, int64_t cols, int txs,
                                                      const float* scale, int64_t n_scale, const void* zp, int zp_dt,
                                                      int64_t n_zp, float* y) {
    const int64_t col = first_col<V>(txs);
    if (col >= cols) return;
    float sc[V];
    int32_t z[V];
    if constexpr (COL) {
#pragma unroll
        for (int e = 0; e < V; ++e) {
            const int64_t c = min(col + e, cols - 1);
            sc[e] = scale[c];
            z[e] = zp ? load_zp(zp, zp_dt, n_zp > 1 ? c : 0) : 0;
        }
    }
    walk_rows<V>(n, rows, cols, txs, col, [&](int64_t r, int64_t i, int have) {
        T v[V];
        load_v<V>(v, x + i, have);
        float rs = 0.f;
        int32_t rz = 0;
        if constexpr (!COL) {
            const int64_t c = n_scale == 1 ? 0 : rows >> 32 ? r % n_scale : (int64_t)((uint32_t)r % (uint32_t)n_scale);
            rs = scale[c];
            rz = zp ? load_zp(zp, zp_dt, n_zp > 1 ? c : 0) : 0;
        }
        float f[V];
#pragma unroll
        for (int e = 0; e < V; ++e) f[e] = (float)wrap_add((int32_t)v[e], -(COL ? z[e] : rz)) * (COL ? sc[e] : rs);
        store_v<V>(y + i, f, have);
    });
}

// y = post(act(x + bias[column])), bias optional.
template <int ACT, int V>
__global__ __launch_bounds__(256) void activation_kernel(const float* x, float* y, int64_t n, int64_t rows, int64_t cols,
                                                         int txs, const float* bias, float a, float b, int post, float ps,
                                                         float pb) {
    const int64_t col = first_col<V>(txs);
    if (col >= cols) return;
    float bi[V];
    if (bias) {
#pragma unroll
        for (int e = 0; e < V; ++e) bi[e] = bias[min(col + e, cols - 1)];
    }
    walk_rows<V>(n, rows, cols, txs, col, [&](int64_t, int64_t i, int have) {
        float v[V];
        load_v<V>(v, x + i, have);
#pragma unroll
        for (int e = 0; e < V; ++e) {
            if (bias) v[e] += bi[e];
            if (ACT != INGOT_ACT_NONE) v[e] = apply_act(v[e], ACT, a, b);
            if (post) v[e] = v[e] * ps + pb;
        }
        store_v<V>(y + i, v, have);
    });
}

template <int V>
__global__ __launch_bounds__(256) void cast_bf16_kernel(const float* x, uint16_t* y, int64_t n, int64_t rows,
                                                        int64_t cols, int txs) {
    const int64_t col = first_col<V>(txs);
    if (col >= cols) return;
    walk_rows<V>(n, rows, cols, txs, col, [&](int64_t, int64_t i, int have) {
        float v[V];
        load_v<V>(v, x + i, have);
        uint16_t h[V];
#pragma unroll
        for (int e = 0; e < V; ++e) h[e] = f32_to_bf16(v[e]);
        store_v<V>(y + i, h, have);
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
    if (inner < 1) inner = 1;
    // element i takes scale (i / inner) % n_scale: per column when inner is 1,
    // per row of `inner` else; one scale for all: any row length
    const bool col = n_scale > 1 && inner == 1;
    const Grid2 g(n, n_scale == 1 ? std::min<int64_t>(n, 1024) : (col ? n_scale : inner));
    const auto launch = [&](auto kernel, auto t) {
        typedef decltype(t) T;
        hipLaunchKernelGGL(kernel, g.grid(), dim3(256), 0, st, (const T*)x, n, g.rows, g.cols, g.txs, scale, n_scale, zp,
                           zp_dtype, n_zp, y);
        return hipGetLastError();
    };
    const auto go = [&](auto t) {
        typedef decltype(t) T;
        if (g.v == 1) return col ? launch(dequant_kernel<T, true, 1>, t) : launch(dequant_kernel<T, false, 1>, t);
        return col ? launch(dequant_kernel<T, true, 4>, t) : launch(dequant_kernel<T, false, 4>, t);
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
    const Grid2 g(n, bias ? cols : std::min<int64_t>(n, 1024));
    const auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, g.grid(), dim3(256), 0, st, x, y, n, g.rows, g.cols, g.txs, bias, a, b, post, ps, pb);
        return hipGetLastError();
    };
    switch (act) {
#define INGOT_ACT_CASE(A) \
    case A: return g.v == 1 ? launch(activation_kernel<A, 1>) : launch(activation_kernel<A, 4>);
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
    const Grid2 g(n, std::min<int64_t>(n, 1024));
    if (g.v == 1)
        hipLaunchKernelGGL(cast_bf16_kernel<1>, g.grid(), dim3(256), 0, st, x, y, n, g.rows, g.cols, g.txs);
    else
        hipLaunchKernelGGL(cast_bf16_kernel<4>, g.grid(), dim3(256), 0, st, x, y, n, g.rows, g.cols, g.txs);
    return hipGetLastError();
}

hipError_t launch_fill(void* dst, int value, size_t bytes, hipStream_t st) {
    hipLaunchKernelGGL(fill_kernel, dim3(grid_for((int64_t)(bytes / 16 + 31), 256)), dim3(256), 0, st, (uint8_t*)dst,
                       (uint8_t)value, bytes);
    return hipGetLastError();
}

}  // namespace ingot
