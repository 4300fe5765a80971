// Tile configuration tables and dispatch of the MFMA GEMM (the kernel itself
// is in gemm_mfma.hpp; each kind's instances are in their own source file).

#include "gemm_mfma.hpp"

namespace ingot {

namespace {

// Tile configurations per kind. occupancy: workgroups per CU the LDS and
// register footprint allow. A k-tile of a small tile costs its LDS traffic and
// its barrier, not its MFMAs, so what pays is wave tiles that share fragments,
// eight waves (two per SIMD) and three or four stages: bf16 128×128 0.35–0.43 µs
// with eight waves and three stages against 0.57 with four waves and two, hi/lo
// 64×128 0.45–0.50 with four stages against 0.67 for two 64×64 tiles of two.
// The bf16 kinds' costs (pick_config adds them up) are those that lose least
// over 500 (bf16) and 469 (hi/lo) products, M = 17–8192, K = 64–16384, N = 64–16384
// at random and the decoder's, encoder's and diffusion block's, every tile timed
// on each on MI355X with the operands cached and from HBM: the picks take 0.4%
// and 0.2% more than the best tile of each. Costs of full rounds measured on
// forty of them, with 4 µs a round for every tile, lost up to 15% on large tiles
// of short K and on products from HBM (hi/lo 1024 × 768 → 3072 22.9 µs, 20.9 now;
// 4096 × 12288 → 3072 560, 512 now).
// Tiles with two stages serve what they divide best: 192×256 (M around multiples
// of 192: hi/lo 3000 × 4096 → 4096 181 µs against 194 with 128×128, bf16 6912 × 3256
// → 2944 145 against 173); hi/lo 64×96, two per CU (N around multiples of 96: 1088 ×
// 1920 → 2432 33 against 35, 1728 × 9826 → 1280 134 against 155). bf16 128×192 with
// three stages has the products of one round that 192×128 and 128×128 divide worse
// (2048 × 768 → 3072, bf16 out, 18.6 µs; 24.4 with 192×192).
// Entry 9 is entry 1 with the weight staged through registers (gemm_kernel's
// RS = 2): every load issued two k-tiles ahead instead of one. On MI355X, the
// DiT MLP-down (M = 4096, N = 3072, K = 12288) right after the MLP-up GEMM
// (whose 201 MB of output fill the Infinity Cache) took 253–257 µs instead of
// 293–294, and after a 1 GiB fill 241 instead of 310; with its operands
// already cached it is 8–12% slower (249 vs 230 µs), so the runtime takes it
// only for products whose operands are too large to stay cached.
const GemmConfig kBF16Cfgs[] = {{256, 256, 1, -1, 0.61f, 5.96f, {1.341f}},
                                {256, 192, 1, 9, 0.66f, 4.47f, {1.104f}},
                                {128, 128, 1, -1, 0.67f, 1.49f, {0.457f}},
                                {192, 128, 1, -1, 0.64f, 2.23f, {0.603f}},
                                {64, 128, 1, -1, 0.60f, 0.74f, {0.264f}},
                                {32, 64, 3, -1, 1.00f, 0.19f, {0.143f, 0.284f, 0.397f}},
                                {128, 256, 1, -1, 0.89f, 2.98f, {0.775f}},
                                {32, 32, 3, -1, 1.00f, 0.09f, {0.127f, 0.169f, 0.272f}},
                                {64, 64, 2, -1, 0.73f, 0.37f, {0.195f, 0.381f}},
                                {256, 192, 1, 9, 0.66f, 4.47f, {1.094f}},
                                {192, 256, 1, -1, 0.64f, 4.47f, {1.112f}},
                                {192, 192, 1, -1, 0.71f, 3.35f, {0.798f}},
                                {128, 192, 1, -1, 0.66f, 2.23f, {0.655f}}};
// hi/lo: tiles of 128 rows hold both activation planes in a stage, which costs
// fewer operand bytes than the taller tiles' second pass over the weight (1.29
// against 2.42 µs for 128×192 and 256×192, half the area). 16×32 with five stages
// serves up to 16 rows and long K: half the activation bytes a k-tile of 32×32,
// and one wave's chain of fragment reads and MFMAs hidden by the fragments read
// ahead and by up to three workgroups per CU (M = 16, weights from HBM / cached:
// 2048 → 6144 13.6 / 10.6 → 12.5 / 9.7 µs, 5632 → 4096 27.3 / 20.0 → 23.3 / 16.9,
// 3584 → 19712 36.6 / 30.5 → 32.9 / 26.8); 32×64 stays better where it is one
// round of one per CU (2048 → 11264 12.5 against 13.2). 32×32 has six stages:
// with four the loads of a k-tile come too late (M = 64, 5632 → 4096 28.9 / 21.4
// → 27.8 / 20.6). 16×64, 16×48, 16×16 and eight stages were level or slower.
const GemmConfig kBF16X2Cfgs[] = {{256, 256, 1, -1, 0.65f, 5.17f, {2.993f}},
                                  {256, 192, 1, 9, 0.63f, 3.88f, {2.417f}},
                                  {128, 128, 1, -1, 0.63f, 1.29f, {0.916f}},
                                  {64, 256, 1, -1, 0.66f, 1.29f, {0.911f}},
                                  {64, 128, 1, -1, 0.72f, 0.65f, {0.468f}},
                                  {32, 64, 2, -1, 1.00f, 0.16f, {0.229f, 0.435f}},
                                  {128, 256, 1, -1, 0.63f, 2.58f, {1.509f}},
                                  {32, 32, 2, -1, 1.00f, 0.08f, {0.175f, 0.321f}},
                                  {64, 64, 1, -1, 0.64f, 0.32f, {0.320f}},
                                  {256, 192, 1, 9, 0.65f, 3.88f, {2.392f}},
                                  {128, 192, 1, -1, 0.64f, 1.94f, {1.287f}},
                                  {16, 32, 3, -1, 1.00f, 0.04f, {0.154f, 0.293f, 0.416f}},
                                  {192, 256, 1, -1, 0.64f, 3.88f, {2.402f}},
                                  {64, 96, 2, -1, 0.68f, 0.48f, {0.521f, 0.742f}}};
// f32: a k-tile is bound by its MFMAs (a tile's area per µs of cost is 7.1–9.0
// thousand outputs, 9.0 being 147 of the 157 TFLOP/s peak), so the tiles differ
// little but for how they divide a product over 256 CUs; 32×32 serves products
// of few tiles (128 × 256 → 512: 64 of them, 3.8 against 6.2 µs with 32×96), the
// four-stage 32×96 ones of one tile per CU (1024 × 3072 → 768 42.5 against 45.9
// with two stages), 64×64 and 64×96 with three stages the rest (1024 × 768 →
// 3072 38.5 against 39.7 µs with two; 260 × 2048 → 4096 50.9 against 55.7 with
// 32×96; 2048 × 768 → 2304 56.7 against 61). Measured like the bf16 kinds'
// costs, over M = 16–2048; the picks are within 0.5% of the best of 18 tiles.
const GemmConfig kF32Cfgs[] = {{128, 128, 2, -1, 1.00f, 0.00f, {1.816f, 3.670f}},
                               {128, 64, 3, -1, 1.00f, 0.00f, {0.936f, 1.826f, 2.750f}},
                               {64, 64, 3, -1, 1.00f, 0.00f, {0.484f, 0.924f, 1.368f}},
                               {32, 96, 3, -1, 1.00f, 0.00f, {0.432f, 0.755f, 1.229f}},
                               {32, 32, 3, -1, 1.00f, 0.00f, {0.169f, 0.294f, 0.429f}},
                               {32, 96, 2, -1, 1.00f, 0.00f, {0.387f, 0.740f}},
                               {64, 96, 2, -1, 1.00f, 0.00f, {0.723f, 1.407f}}};
// int8: costs fitted like the bf16 kinds' over 425 products (M = 1–100352, N = 16–
// 16384, K = 64–12288, f32 and byte outputs); the picks take 0.9% more than the best
// tile of each, where one efficiency per tile taken from a single product took up
// to 27% more (MI355X: 4096 × 4096 → 4096 84 µs with 128×128, 70 with 256×256; 8192 ×
// 4096 → 4096 172 / 135; 4096 × 1024 → 4096 37 / 31; 2048 × 768 → 3072 16.5, 13.7 with
// 64×96; 2048 × 4096 → 4096 42 with 128×128, 54 with 256×256). With K this short the
// stores count as much as the k-tiles, most for 256×256, whose CUs all store at
// once (7744 × 67 → 16320 213 µs, 126 with 64×96). 32×32 and 64×64 with four stages
// serve products of few tiles (M = 1–128 at K = 768–2048 3.8–5.3 µs; 196 tiles of 18
// k-tiles 9.8–10.4, 13.2–14.1 with two stages); 128×128 has eight waves and four
// stages. 128×96, 32×96, 64×128, 64×192, 32×64 to 32×128 and deeper rings were slower.
const GemmConfig kI8Cfgs[] = {{256, 256, 1, -1, 0.96f, 16.66f, {1.247f}},
                              {128, 128, 1, -1, 0.90f, 2.07f, {0.629f}},
                              {128, 64, 3, -1, 0.79f, 1.05f, {0.554f, 0.674f, 0.904f}},
                              {64, 64, 4, -1, 0.80f, 0.44f, {0.344f, 0.381f, 0.594f, 0.682f}},
                              {64, 96, 3, -1, 0.85f, 0.59f, {0.428f, 0.552f, 0.758f}},
                              {32, 32, 4, -1, 1.00f, 0.16f, {0.148f, 0.194f, 0.301f, 0.301f}},
                              {64, 64, 2, -1, 0.82f, 0.67f, {0.270f, 0.333f}}};

}  // namespace

int gemm_configs(GemmKind kind, const GemmConfig** out) {
    switch (kind) {
        case KIND_BF16: *out = kBF16Cfgs; return (int)(sizeof(kBF16Cfgs) / sizeof(kBF16Cfgs[0]));
        case KIND_F32: *out = kF32Cfgs; return (int)(sizeof(kF32Cfgs) / sizeof(kF32Cfgs[0]));
        case KIND_I8: *out = kI8Cfgs; return (int)(sizeof(kI8Cfgs) / sizeof(kI8Cfgs[0]));
        case KIND_BF16X2: *out = kBF16X2Cfgs; return (int)(sizeof(kBF16X2Cfgs) / sizeof(kBF16X2Cfgs[0]));
        default: break;
    }
    return 0;
}

float gemm_round_us(GemmKind kind) {
    return kind == KIND_I8 ? 2.32f : kind == KIND_BF16 ? 4.06f : kind == KIND_BF16X2 ? 4.05f : 4.f;
}

hipError_t launch_gemm(GemmKind kind, int cfg, const GemmArgs& a, int batch, hipStream_t st) {
    switch (kind) {
        case KIND_BF16: return launch_gemm_bf16(cfg, a, batch, st);
        case KIND_BF16X2: return launch_gemm_bf16x2(cfg, a, batch, st);
        case KIND_F32: return launch_gemm_f32(cfg, a, batch, st);
        case KIND_I8: return a.conv.cpc ? launch_gemm_i8_conv(cfg, a, batch, st) : launch_gemm_i8(cfg, a, batch, st);
        default: break;
    }
    return hipErrorInvalidValue;
}

}  // namespace ingot
