// sq8_gemm.h — host/device interface of the gfx950 weight-quantized GEMM kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "sq8_device.h"

namespace sq8 {

// One launch's operands; all pointers are device pointers.
struct GemmArgs {
    const uint16_t *a;      // bf16 [M, K], leading dimension lda (elements)
    int64_t lda;
    const uint8_t *w;       // codes: [K, N] (W_KN) or [N, K] (W_NK), leading dimension ldw
    int64_t ldw;
    const float *scale;     // fp32 [N] (scale_per_col) or [1]
    const float *bias;      // fp32 [N] or null
    void *c[3];             // outputs; c[1], c[2] only with `split`
    int64_t c_d1, c_d2;     // byte offsets of c[1], c[2] from c[0] (the device never indexes c[])
    int64_t ldc;
    int split;              // > 0: output columns [i·split, (i+1)·split) go to c[i]
    int head_dim;           // > 0: each output is [cols/head_dim, M, head_dim]
    int M, N, K;            // N: weight columns (2h for a GLU epilogue)
    int glu_half;           // h for GLU epilogues
    int scale_per_col;
    int a_vec, w_vec, c_vec; // 16-byte loads of A, wide loads of W, wide stores of C allowed
    int c_vec16;            // 16-byte stores of C allowed (aligned base, stride, split and head size)
    int sb_vec;             // 16-byte loads of 4 scales / biases allowed (aligned bases, GLU half % 4 == 0)
    int kt;                 // K steps of 64 (the packed layout's K extent); W8A8: K steps of 128
    int tiles_m, tiles_n;   // set by the launcher
    const float *gate;      // EPI_RESIDUAL: per-column gate fp32 [N], or null (1)
    const float *sx;        // W8A8: the activation's row scales fp32 [M] (`a` then holds int8 codes)
    int kt_w;               // W8A8: K steps of 64 of the packed weight; weight-direct kernels: the weight's
                            // K steps when the activation holds several parts along K (0: kt)
    float *part;            // the skinny kernel's K split: fp32 partial sums, skinny_part_bytes() of them
    int splits;             // > 1: the skinny kernel's K steps split over this many workgroups per tile, whose
                            // sums a second launch adds in split order before the epilogue
    int cus;                // the device's compute units (0: 256), for launch shapes chosen per product
    int epi, out;           // set by the launcher of a kernel that reads them at run time (sq8_group_kernel.h)
};

enum Tile { TILE_256x256 = 0, TILE_128x128 = 1 };

int choose_tile(int M, int N_out, bool glu, int cus);
// `fast`: the branch-free kernels on [K, N] codes, valid when A rows and W columns can be read with vector loads
// (alignment), K is a positive multiple of 64, and the weight columns (per GLU half) are a positive multiple of 4.
hipError_t launch_gemm(const GemmArgs &p, bool fast, int tile, int wt, int wl, int epi, int out, hipStream_t stream);

// The weight-direct kernels (sq8_wdirect_inst.hip): [N, K] or packed weights, K a multiple of 64,
// A aligned for 16-byte loads. `tile`: WD_256 (256 × 256, one workgroup per CU), WD_224 (224 × 256, the
// same kernel), WD_128 (128 × 256, two workgroups per CU), WD_GEMV (M ≤ 16 in 16-column groups on 16 × 16 MFMAs, every
// K step's loads issued far ahead), the skinny-M kernel with 64- or 32-row tiles of one 64-column slab and the K steps
// split over four waves (WD_SKINNY64, WD_SKINNY32), a K-group tile's id (below), or 64 rows without groups in WD_128's order of sums: WD_64
// (64 × 256, one per CU), WD_64N (64 × 128, a 32-column block a wave, two per CU; not GLU). By the SQ8_TILE knob only:
// WD_32 (32 × 256, two per CU), WD_64x192 (64 × 192, six waves of one 32-column block; not GLU), WD_SKINNY64.
enum WdTile { WD_256 = 0, WD_128 = 1, WD_SKINNY64 = 2, WD_SKINNY32 = 3, WD_64 = 4, WD_32 = 5, WD_224 = 6, WD_64N = 7, WD_64x192 = 8,
              WD_GEMV = 9 };
// The tile for an M × N product (GLU: N = 2h) of `steps` weight K steps of 64, `f32` on the fp32 route (three parts of
// an fp32 activation): by the shape alone, so that a call's bits depend on nothing else.
int choose_wd_tile(int M, int N, bool glu, int cus, int steps, bool f32);
// The short-M kernel (sq8_gemv_kernel.h): the activation staged in LDS (M rows of K' = kt · 64 bf16, rows
// gemv_xpitch bytes apart: 16 more than a row, so the 16 rows a fragment read touches start on different banks)
// when it fits GEMV_XLDS bytes and each row is whole 1 KB runs (K' a multiple of 512), the unit of a direct load.
constexpr int GEMV_XLDS = 100 * 1024;
__host__ __device__ constexpr int64_t gemv_xpitch(int kt) { return (int64_t)kt * 128 + 16; }
__host__ __device__ constexpr bool gemv_x_in_lds(int m, int kt) {
    return kt % 8 == 0 && (int64_t)m * gemv_xpitch(kt) <= GEMV_XLDS;
}
// Bytes of the partial sums of a split skinny product (tile height bm, `splits` splits).
int64_t skinny_part_bytes(int M, int N, bool glu, int bm, int splits);
hipError_t launch_wdirect(const GemmArgs &p, int tile, int wt, int wl, int epi, int out, hipStream_t stream);

// The K-group kernels (sq8_group_kernel.h): `rows` × `cols` tiles (cols: weight columns) whose K steps split over
// `groups` wave groups; GLU products take those of an even number of 32-column blocks. What a round of tiles on
// the CUs, one a CU, takes by kind of product: us + us_step · (weight K steps) microseconds, the launch's own 2.5 µs (and
// the fp32 route's split pass) taken off; us_step 0: not built for it. W8A8: fitted to 256 and 512 tiles at K = 1024, 3072
// and 8192; the others to 857 and 596 shapes of 17 to 5000 rows, K 256 to 12288, plain and GLU, weights in and out of
// the caches (each within 4 to 7 %).
enum GroupMath { GM_BF16 = 0, GM_I8 = 1, GM_F32 = 2 };
struct GroupCost {
    float us, us_step;
};
struct GroupShape {
    int rows, cols, groups;
    const char *name;   // the SQ8_TILE knob's name for it
    GroupCost cost[3];  // by GroupMath
};
constexpr int GROUP_TILE0 = 100;  // tile ids of the K-group kernels: GROUP_TILE0 + index into group_shapes
constexpr GroupShape group_shapes[] = {
    {32, 32, 8, "g32x32k8", {{}, {0.65f, 0.104f}, {}}},
    {32, 64, 8, "g32x64k8", {{}, {0.55f, 0.165f}, {}}},
    {32, 32, 4, "g32x32k4", {{1.85f, 0.077f}, {}, {1.09f, 0.198f}}},
    {32, 64, 4, "g32x64k4", {{2.55f, 0.107f}, {}, {1.40f, 0.280f}}},
    {64, 64, 4, "g64x64k4", {{3.55f, 0.161f}, {1.60f, 0.204f}, {2.81f, 0.366f}}},
    {64, 96, 4, "g64x96k4", {{3.87f, 0.210f}, {2.65f, 0.243f}, {3.73f, 0.472f}}},
    {64, 128, 4, "g64x128k4", {{4.28f, 0.277f}, {2.30f, 0.325f}, {4.38f, 0.591f}}},
    {64, 128, 2, "g64x128k2", {{4.04f, 0.263f}, {}, {3.81f, 0.628f}}},
    {64, 192, 2, "g64x192k2", {{5.11f, 0.390f}, {}, {5.18f, 0.893f}}},
    {96, 96, 4, "g96x96k4", {{5.08f, 0.273f}, {3.60f, 0.312f}, {5.12f, 0.666f}}},
    {96, 128, 4, "g96x128k4", {{5.61f, 0.357f}, {4.40f, 0.408f}, {}}},
    {128, 96, 4, "g128x96k4", {{5.72f, 0.375f}, {4.70f, 0.402f}, {}}},
    {128, 128, 2, "g128x128k2", {{6.22f, 0.443f}, {6.30f, 0.493f}, {6.75f, 1.131f}}},
    {96, 192, 2, "g96x192k2", {{6.59f, 0.482f}, {6.30f, 0.560f}, {7.02f, 1.207f}}},
    {128, 192, 2, "g128x192k2", {{8.00f, 0.606f}, {8.70f, 0.694f}, {8.85f, 1.553f}}},
};
constexpr int kGroupShapes = (int)(sizeof(group_shapes) / sizeof(group_shapes[0]));
hipError_t launch_group(const GemmArgs &p, int math, int shape, int wt, int wl, int epi, int out, hipStream_t stream);

// Bytes of the packed layout of a weight with k rows of K and n columns (GLU: n = 2h, packed in
// pairs of 32-column blocks of the two halves).
int64_t packed_bytes(int k, int n, bool glu);
// Writes the packed layout of codes `w` (layout W_KN or W_NK, leading dimension ldw) into `out`.
hipError_t launch_pack(const uint8_t *w, int wl, int64_t ldw, int k, int n, bool glu, uint8_t *out,
                       hipStream_t stream);

// Codes with a scale per block of rows and column (GGUF Q8_0; sq8_blocks.hip): the packed Q8 layout
// (codes in block-aligned K order, then fp32 scales per step and column) and its product, int8
// codes, K a multiple of 64, A aligned for 16-byte loads. `tile`: choose_blocks_tile's: BL_128x256 (eight waves of one
// 32-column block each, one workgroup per CU), BL_64x256 (the same waves on half the rows), BL_128x128 (four, two per
// CU), or BLOCKS16_ROWS + rows (below). Scales
// [K/B, N] for W_KN codes, [N, K/B] for W_NK; B a multiple of 32 dividing K; scale dtype numbered as the C ABI's
// (fp32, bf16, fp16).
enum BlocksTile { BL_128x256 = 0, BL_128x128 = 1, BL_64x256 = 2 };
int64_t packed_blocks_bytes(int k, int n, bool glu);
hipError_t launch_pack_blocks(const uint8_t *w, int wl, int64_t ldw, const void *scale, int scale_dtype, int block,
                              int k, int n, bool glu, uint8_t *out, hipStream_t stream);
// Tiles of BLOCKS16_ROWS + rows: the narrow-wave kernel (sq8_blocks16_kernel.h: 16, 32, 48, 64 or 80 rows × 64
// columns, waves of 16 columns).
constexpr int BLOCKS16_ROWS = 100;
int choose_blocks_tile(int M, int N, bool glu, int cus, int kt);
hipError_t launch_blocks16(const GemmArgs &p, int rows, int epi, int out, hipStream_t stream);
hipError_t launch_blocks_product(const GemmArgs &p, int tile, int epi, int out, hipStream_t stream);

// Auxiliary kernels (sq8_aux.hip).
hipError_t launch_dequantize(const uint8_t *codes, int wt, int64_t rows, int64_t columns, const void *scale,
                             int scale_dtype, int scale_layout, int64_t block_rows, int64_t first_row, float *out,
                             hipStream_t stream);
hipError_t launch_round_bf16(const float *x, uint16_t *y, int64_t count, hipStream_t stream);
// rows × k values read ldx apart → rows × kp bf16 written kp apart (kp ≥ k, columns [k, kp) zero; one
// launch, any stride).
hipError_t launch_round_bf16_rows(const float *x, int64_t ldx, uint16_t *y, int64_t rows, int k, int kp,
                                  hipStream_t stream);
// bf16 rows × k read ldx apart → rows × kp written kp apart, columns [k, kp) zero.
hipError_t launch_pad_bf16_rows(const uint16_t *x, int64_t ldx, uint16_t *y, int64_t rows, int k, int kp,
                                hipStream_t stream);
// Columns [k, kp) of rows × ld bf16 set to zero.
hipError_t launch_zero_tail(uint16_t *y, int64_t ld, int64_t rows, int k, int kp, hipStream_t stream);
// fp32 [rows, k] (leading dimension ldx) → bf16 [rows, 3kp]: the three parts hi | mid | lo of each value
// (each the top 16 bits of what the one before leaves: hi + mid + lo = x, no part rounded), each part kp ≥ k
// wide with columns [k, kp) zero; the fp32 route's operand.
hipError_t launch_split3(const float *x, int64_t ldx, uint16_t *y, int64_t rows, int k, int kp, hipStream_t stream);

// ComfyUI's convrot (sq8_convrot.hip): the activation's rotation x·R by groups of `group` (4, 16,
// 64 or 256; k a multiple of it), fp32 or bf16 in, fp32 or bf16 (rounded to nearest even) out; and
// the rotated weight widened, Float(H·q)·(s/√G), codes [k, n] rotated along k.
bool is_rotation_group(int group);
hipError_t launch_rotate_groups(const void *x, bool x_bf16, int64_t ldx, void *y, bool y_bf16, int64_t ldy, int64_t rows,
                                int k, int group, hipStream_t stream);
hipError_t launch_dequantize_rotated(const int8_t *q, int64_t ldq, int k, int n, int group, const void *scale,
                                     int scale_dtype, bool per_column, float *out, int64_t ldo, hipStream_t stream);

// W8A8 (sq8_w8a8.hip, sq8_i8_inst.hip): the activation's per-row quantization (optionally rotated
// first) into int8 codes of rows k_pad ≥ k bytes (zero past k) and fp32 row scales; rows up to
// quantize_row_limit() values. The int8 × int8 product: `a` the codes (lda a multiple of 16,
// 16-byte aligned, kt = k_pad / 128 steps, zero past K), `sx` their scales, the weight packed
// (kt_w = its 64-steps) or [N, K] with K a multiple of 128.
int quantize_row_limit();
hipError_t launch_quantize_rows(const void *x, bool x_bf16, int64_t ldx, int rows, int k, int group, int8_t *codes,
                                int64_t ldq, int k_pad, float *scales, hipStream_t stream);
hipError_t launch_pad_codes(const int8_t *src, int64_t ld_src, int8_t *dst, int64_t ld_dst, int64_t rows, int k, int k_pad,
                            hipStream_t stream);
// `tile`: choose_i8_tile's: I8_128x256 (128 × 256, two workgroups a CU) or a K-group tile's id. kt: K steps of 128.
constexpr int I8_128x256 = 0;
int choose_i8_tile(int M, int N, bool glu, int cus, int kt, bool residual);
hipError_t launch_i8gemm(const GemmArgs &p, int tile, int wl, int epi, int out, hipStream_t stream);

// The DiT block's elementwise passes (sq8_block.hip).
hipError_t launch_norm_modulate(const float *x, int64_t ldx, const float *w, const float *scale, const float *shift,
                                float eps, uint16_t *out, int64_t ldo, int rows, int cols, hipStream_t stream);
// The modulated RMSNorm writing the next product's operand: y rotated by `group` (0: none) and
// rounded to bf16 into `out` (codes == nullptr), or quantized per row into codes (rows of k_pad) and
// scales; y itself into y_out when given. cols % 4 == 0, 16-byte aligned rows and vectors, cols ≤ 32 768.
hipError_t launch_norm_operand(const float *x, int64_t ldx, const float *w, const float *scale, const float *shift,
                               float eps, int rows, int cols, int group, float *y_out, int64_t ldy, uint16_t *out,
                               int64_t ldo, int8_t *codes, int64_t ldq, int k_pad, float *scales, hipStream_t stream);
hipError_t launch_rms_rows(uint16_t *t, int64_t ld, int64_t rows, int cols, const float *w, float eps, hipStream_t stream);
hipError_t launch_gated_residual(float *x, int64_t ldx, const void *y, bool y_bf16, int64_t ldy, const float *gate,
                                 int64_t rows, int cols, hipStream_t stream);

}  // namespace sq8
