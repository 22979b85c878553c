// sq8_gemm.hip — picks the GEMM kernel for a product: the branch-free kernels when the operands
// allow them (sq8_gemm_inst.hip), the guarded ones otherwise (sq8_gemm_general.hip).
#include "sq8_gemm.h"

#include <math.h>

namespace sq8 {

hipError_t launch_fast_0(const GemmArgs &p, int tile, int epi, int out, hipStream_t stream);
hipError_t launch_fast_1(const GemmArgs &p, int tile, int epi, int out, hipStream_t stream);
hipError_t launch_general(const GemmArgs &p, int wt, int wl, int epi, int out, hipStream_t stream);
hipError_t launch_short_0_1(const GemmArgs &p, int tile, int epi, int out, hipStream_t stream);
hipError_t launch_short_0_2(const GemmArgs &p, int tile, int epi, int out, hipStream_t stream);
hipError_t launch_short_1_1(const GemmArgs &p, int tile, int epi, int out, hipStream_t stream);
hipError_t launch_short_1_2(const GemmArgs &p, int tile, int epi, int out, hipStream_t stream);
hipError_t launch_wdirect_0_1(const GemmArgs &p, int tile, int epi, int out, hipStream_t stream);
hipError_t launch_wdirect_0_2(const GemmArgs &p, int tile, int epi, int out, hipStream_t stream);
hipError_t launch_wdirect_1_1(const GemmArgs &p, int tile, int epi, int out, hipStream_t stream);
hipError_t launch_wdirect_1_2(const GemmArgs &p, int tile, int epi, int out, hipStream_t stream);

hipError_t launch_wdirect(const GemmArgs &p, int tile, int wt, int wl, int epi, int out, hipStream_t stream) {
    if (tile >= GROUP_TILE0)
        return launch_group(p, p.kt_w > 0 ? GM_F32 : GM_BF16, tile - GROUP_TILE0, wt, wl, epi, out, stream);
    const bool shorter = tile == WD_GEMV || tile == WD_SKINNY64 || tile == WD_SKINNY32;
#define SQ8_CASE(T, L)                                                                                          \
    if (wt == T && wl == L)                                                                                     \
        return shorter ? launch_short_##T##_##L(p, tile, epi, out, stream) : launch_wdirect_##T##_##L(p, tile, epi, out, stream);
    SQ8_CASE(0, 1)
    SQ8_CASE(0, 2)
    SQ8_CASE(1, 1)
    SQ8_CASE(1, 2)
#undef SQ8_CASE
    return hipErrorInvalidValue;
}

hipError_t launch_group_0_0_1(const GemmArgs &p, int shape, int epi, int out, hipStream_t stream);
hipError_t launch_group_0_0_2(const GemmArgs &p, int shape, int epi, int out, hipStream_t stream);
hipError_t launch_group_0_1_1(const GemmArgs &p, int shape, int epi, int out, hipStream_t stream);
hipError_t launch_group_0_1_2(const GemmArgs &p, int shape, int epi, int out, hipStream_t stream);
hipError_t launch_group_1_0_1(const GemmArgs &p, int shape, int epi, int out, hipStream_t stream);
hipError_t launch_group_1_0_2(const GemmArgs &p, int shape, int epi, int out, hipStream_t stream);
hipError_t launch_group_2_0_1(const GemmArgs &p, int shape, int epi, int out, hipStream_t stream);
hipError_t launch_group_2_0_2(const GemmArgs &p, int shape, int epi, int out, hipStream_t stream);
hipError_t launch_group_2_1_1(const GemmArgs &p, int shape, int epi, int out, hipStream_t stream);
hipError_t launch_group_2_1_2(const GemmArgs &p, int shape, int epi, int out, hipStream_t stream);

hipError_t launch_group(const GemmArgs &p, int math, int shape, int wt, int wl, int epi, int out, hipStream_t stream) {
#define SQ8_CASE(M, T)                                                                                   \
    if (math == M && wt == T)                                                                            \
        return wl == W_NK ? launch_group_##M##_##T##_1(p, shape, epi, out, stream)                       \
                          : launch_group_##M##_##T##_2(p, shape, epi, out, stream);
    SQ8_CASE(0, 0)
    SQ8_CASE(0, 1)
    SQ8_CASE(1, 0)
    SQ8_CASE(2, 0)
    SQ8_CASE(2, 1)
#undef SQ8_CASE
    return hipErrorInvalidValue;
}

// Tiles of `rows` rows × `nb` of the weight's blocks; a count past 2^24 only rounds.
static inline float tile_count(int M, int rows, int blocks, int nb) {
    return (float)((M + rows - 1) / rows) * (float)((blocks + nb - 1) / nb);
}

// Microseconds of `tiles` workgroups, `cus` at a time, `round` each: a last, partly filled round is shorter (its
// workgroups share the memory system with fewer others: half the CUs 0.83 of a full round).
static float rounds_us(float tiles, int cus, float round) {
    const float rounds = tiles / (float)cus, full = floorf(rounds), rest = rounds - full;
    return round * (full + (rest > 0.0f ? 0.66f + 0.34f * rest : 0.0f));
}

// The same of a kernel of two workgroups a CU: `two` a round of them, `one` a last round of at most one a CU; a last round
// with two on some CUs and one on the others is shorter (384 of 512: 0.88 to 0.96 of `two` on the three routes).
static float pairs_us(float tiles, int cus, float two, float one) {
    const float full = floorf(tiles / (2.0f * (float)cus)), rest = tiles - full * 2.0f * (float)cus;
    if (rest > (float)cus) return two * (full + 0.86f + 0.14f * (rest / (float)cus - 1.0f));
    return full * two + rounds_us(rest, cus, one);
}

// Calls take(tile, µs) for every K-group shape that serves M rows × `blocks` 32-column blocks of weight and `steps` weight K
// steps (unrolled: each shape's divisions are by constants; the rule runs on every call); `value_us`: further µs a value of
// the tile, `round_us`: a round past the first.
template <int MATH, int I = 0, typename F>
static inline void each_group(int M, int blocks, bool glu, int cus, int steps, float value_us, float round_us, F &&take) {
    if constexpr (I < kGroupShapes) {
        constexpr GroupShape g = group_shapes[I];
        constexpr GroupCost c = g.cost[MATH];
        constexpr int nw = g.cols / 32;
        // bf16: four groups give the skinny kernel's bits at any K, two the 64 × 128 tiles' where the steps divide.
        if (c.us_step > 0.0f && !(glu && nw % 2 != 0) && !(MATH == GM_BF16 && steps % 2 != 0 && g.groups == 2)) {
            const float tiles = tile_count(M, g.rows, blocks, nw);
            take(GROUP_TILE0 + I, rounds_us(tiles, cus, c.us + c.us_step * (float)steps + value_us * (float)(g.rows * g.cols)) +
                                      round_us * floorf((tiles - 1.0f) / (float)cus));
        }
        each_group<MATH, I + 1>(M, blocks, glu, cus, steps, value_us, round_us, take);
    }
}

int choose_wd_tile(int M, int N, bool glu, int cus, int steps, bool f32) {
    if (cus <= 0) cus = 256;
    const int kt = f32 ? 3 * steps : steps;  // the activation's K steps
    // Up to 16 rows, the 16-column groups of the short-M kernel where they fit one round of one or two groups a
    // workgroup on the CUs (N ≤ 8192 on 256 CUs), for a single row without GLU three (N ≤ 12288): every K step's loads
    // in flight, the activation read once per workgroup. Kernel traces at K = 3072, N = 3072 (int8 packed, bias): M = 1
    // 4.10 µs against the skinny kernel's 7.44, M = 16 5.95 against 8.73; two groups, SiLU-GLU: M = 3, N = 8192 5.8
    // against 8.5, M = 16 7.3 against 9.4; three, M = 1: N = 9216 8.9 against 9.7, N = 12288 10.6 against 11.4. With the
    // activation not in its LDS, to four rows of up to two groups; one row of three to 32 steps (1 × 832 × 8447 4.7 against
    // 6.0 for a K-group tile, 1 × 7808 × 10944 23.5 against 18.8); ten rows of one group (6 × 12160 × 166 11.3 against 14.2,
    // 5 × 1472 × 2944 4.7 against 5.4; by 11 rows level, 16 × 6144 × 3072 11.3 against 8.5; the fp32 route four: 3 % on
    // average to six, and the K-group tiles' sums are nearer, 2.8e-7 against 3.6e-7 at K = 3136); one group of GLU columns
    // (SiLU-GLU 10 × 3840 × 3072 7.2 against 9.1, 5 × 1152 × 3200 4.8 against 5.9).
    const int groups16 = glu ? (N / 2 + 7) / 8 : (N + 15) / 16;
    const bool staged = gemv_x_in_lds(M, kt);
    if (M <= 16 && ((groups16 <= 2 * cus && (M <= 4 || staged)) || (groups16 <= cus && (glu || M <= (f32 ? 4 : 10))) ||
                    (M == 1 && !glu && (staged || kt <= 32) && groups16 <= 3 * cus)))
        return WD_GEMV;
    // Up to 16 rows on a weight wider than 3/4 of the CUs' 64-column slabs, the skinny kernel (a slab a workgroup, four
    // a CU): its many small workgroups stream the weight best (1 × 3072 × 18432 13.7 µs against 16.0 in 32 × 64 tiles, 8
    // × 9216 7.9 against 7.2), and on short K than half of them (12 × 640 × 11968 5.4 against 5.8; 10 × 6912 × 9216 15.1
    // against 14.2), unless its rows are stored value by value (below). The fp32 route's K-group tiles load the codes once for three parts (16 × 12288 17.8
    // against 21.9).
    const int blocks = glu ? 2 * ((N / 2 + 31) / 32) : (N + 31) / 32;  // 32-column blocks
    const int slabs = (blocks + 1) / 2;
    const bool ragged = (glu ? N / 2 : N) % 8 != 0;
    if (M <= 16 && !f32 && (slabs >= cus * 3 / 4 || (!glu && !ragged && slabs > cus / 2 && steps <= 40))) return WD_SKINNY32;
    // Else the tile of the least estimated time: µs a round of tiles, one a CU (128 × 256 and 64 × 128: two a CU, or one in a
    // round of at most one a CU), fitted as the K-group tiles' (GroupShape). Few tiles go to the K-group tiles: more CUs, and
    // eight to sixteen waves a CU with their loads in flight whatever the tile; many to the 256- and 224-row tiles of one
    // workgroup a CU (the least widening and operand traffic), the height whose rounds cover the fewest rows. Measured
    // (µs, thresholds on tile counts → estimates): 512 × 3072 × 3072 16.5 → 14.6, 1531 × 3072 × 3072 41.8 → 33.0, 200 × 3072 ×
    // 6144 16.4 → 14.0; SiLU-GLU 333 × 3840 × 20480 62.6 → 55.2, 77 × 3840 × 20480 30.6 → 24.1, 20 × 3072 × 6144 10.0 → 7.0, 43
    // × 3424 × 10880 23.1 → 14.8; fp32 route 1531 × 3072 × 3072 130 → 87, 18 × 6592 × 64 36 → 20, 176 × 8512 × 64 117 → 34.
    auto tiles = [&](int rows, int nb) { return tile_count(M, rows, blocks, nb); };
    float best = INFINITY;
    int tile = WD_128;
    auto take = [&](int t, float time) {
        if (time < best) {
            best = time;
            tile = t;
        }
    };
    struct One {  // a round of a tile of one workgroup a CU; `later`: more, past the first
        float us, us_step, later;
        float of(float n, int cus, int steps) const {
            return rounds_us(n, cus, us + us_step * (float)steps) + later * floorf((n - 1.0f) / (float)cus);
        }
    };
    struct Two {
        float two, two_step, one, one_step;
        float of(float n, int cus, int steps, float ragged_two, float ragged_one) const {
            return pairs_us(n, cus, two + two_step * (float)steps + ragged_two, one + one_step * (float)steps + ragged_one);
        }
    };
    // By the shape alone: the 256- and 224-row kernel also wants its scales and outputs aligned, but a choice by alignment
    // or output type would give one call two sets of bits (launch_wdirect takes 128-row tiles, the same sums, where that
    // kernel cannot serve the product).
    const bool whole = glu ? N / 2 % 32 == 0 : N % 64 == 0;
    // Output rows that are not whole 16 bytes of bf16 are stored value by value in these kernels, not in the K-group ones
    // (1032 × 512 × 6559 33.4 µs in 128 × 256 and 25.5 in 96 × 192 tiles). Where a tile of one sequence and one of K groups
    // are within 5 % the K groups, whose sums are nearer too (K = 3072, errors against 64 bits: fp32 route 7.2e-7 in one
    // sequence, 3.8e-7 in two groups, 2.7e-7 in four; bf16 route 1.5e-7, 1.0e-7, 0.8e-7).
    const float nearer = f32 ? 1.05f : 1.0f;
    const Two t128 = f32 ? Two{10.2f, 4.14f, 7.3f, 2.44f} : Two{7.7f, 1.478f, 5.8f, 0.908f};
    take(WD_128, nearer * t128.of(tiles(128, 8), cus, steps, ragged ? 20.0f : 0.0f, ragged ? 14.0f : 0.0f));
    if (whole) {
        take(WD_256, nearer * (f32 ? One{14.8f, 3.49f, 2.9f} : One{11.3f, 1.280f, 3.0f}).of(tiles(256, 8), cus, steps));
        take(WD_224, nearer * (f32 ? One{13.2f, 3.14f, 2.0f} : One{10.0f, 1.149f, 3.1f}).of(tiles(224, 8), cus, steps));
    }
    // 64 rows without groups: 64 × 128 of one-block waves, two a CU, and for the GLU epilogues (and wide plain ones) 64 × 256.
    // They win on few K steps (139 × 384 × 17856 8.2 µs against 12.6 in 64 × 128 of two groups; SiLU-GLU 652 × 3776 × 5120 33.1
    // against 40.1) and where an odd count of steps leaves only the tiles of four groups (2199 × 12096 × 1728). Not on the fp32
    // route.
    if (!f32) {
        if (!glu) take(WD_64N, 1.05f * Two{3.4f, 0.495f, 2.8f, 0.348f}.of(tiles(64, 4), cus, steps, ragged ? 5.2f : 0.0f, ragged ? 4.6f : 0.0f));
        take(WD_64, 1.05f * One{ragged ? 12.2f : 4.4f, 0.530f, -0.8f}.of(tiles(64, 8), cus, steps));
    }
    // From 4096 rows on and past 1024 columns no K groups: the tiles above sum each output's K in one sequence, so a host that
    // chunks its rows by that many gets the bits of one call. What it costs where 128 × 192 tiles of two groups would fill
    // the rounds better (µs): 5760 × 3072 × 3072 115.9 → 119.9, with the residual 124.6 → 141.8, fp32 route 309 → 375.
    if (M >= 4096 && N > 1024) return tile;
    // A K-group round past the first costs 0.8 µs more.
    if (f32)
        each_group<GM_F32>(M, blocks, glu, cus, steps, 0.0f, 0.8f, take);
    else
        each_group<GM_BF16>(M, blocks, glu, cus, steps, 0.0f, 0.8f, take);
    return tile;
}

int choose_i8_tile(int M, int N, bool glu, int cus, int kt, bool residual) {
    // The tile of the least estimated time. Every tile gives the same bits (int32 sums), so only time decides; the
    // 128 × 256 kernel's rounds (two workgroups a CU: 11.2 + 1.70 µs a K step; one: 9.6 + 0.91) are measured as the
    // K-group tiles' (GroupShape). It has the least operand traffic per output and wins where its tiles fill the
    // chip (K = 3072: 4096 × 12288 150 µs against 203 in 128 × 192); with fewer the K-group tiles spread the work
    // over more CUs and hold more loads in flight a CU. Measured, K = 3072, product alone, µs, 128 × 256 tiles
    // against the rule's: 1 × 3072 20.8 → 4.9, 77 × 12288 22.6 → 12.9, 512 × 3072 23.0 → 10.8, 1021 × 3072 24.5 →
    // 17.0, 333 × 9216 25.0 → 20.0; K = 12288, 68 × 512 62.9 → 9.7. The residual epilogue reads and writes 8 bytes a value
    // past the sums, a round's at the CU's share of the memory's rate (0.4 ns a value) where one workgroup fills the CU,
    // half of that under the other's K steps where two do: 3742 × 3072 × 3072 62.9 µs in 128 × 256 and 71.3 in 128 × 192
    // tiles, at K = 12288 163 and 159. Rounds of K-group tiles past the first cost about 1 µs more than it (their loads wait
    // for an epilogue): 3277 × 1024 × 1024 with SiLU-GLU 14.8 µs in 1.6 rounds of 64 × 128, 11.0 in one of 128 × 128; 1975
    // × 3072 × 6144 57.1 in 128 × 192, 49.4 in 128 × 256.
    if (cus <= 0) cus = 256;
    const int blocks = glu ? 2 * ((N / 2 + 31) / 32) : (N + 31) / 32;  // 32-column blocks
    const float two = residual ? 22.2f : 11.2f, one = residual ? 15.6f : 9.6f;
    float best = pairs_us(tile_count(M, 128, blocks, 8), cus, two + 1.70f * (float)kt, one + 0.91f * (float)kt);
    int tile = I8_128x256;
    each_group<GM_I8>(M, blocks, glu, cus, kt, residual ? 4e-4f : 0.0f, 1.0f, [&](int t, float time) {
        if (time < best) {
            best = time;
            tile = t;
        }
    });
    return tile;
}

int choose_blocks_tile(int M, int N, bool glu, int cus, int kt) {
    // Every tile gives the same bits (each sum in K order), so only time decides: the least estimate for the CU that holds
    // the most workgroups, `at_once` of them side by side (registers): µs of a launch, of a workgroup (`group`), and of a K
    // step, a workgroup's chain alone or the CU's work for each of several. Fitted to 270 to 370 shapes of 1 to 5000 rows, K
    // 768 to 12288, plain and GLU, weights in and out of the caches (each tile's estimate within 4 % in the median; the
    // choice 0.1 % past the best tile in the mean, 8 % at most). Narrow waves (16 … 80 rows × 64 columns) where tiles are
    // few; measured against 128 × 256 tiles (µs, K = 3072): 77 × 12288 54 → 22, 512 × 3072 54 → 25, 16 × 128 (K = 2816) 48 →
    // 11; K = 9728, 148 × 960 152 → 31. 64 × 256 where it fits a round that the taller tiles leave part empty or exceed
    // (before it → with it: SiLU-GLU 575 × 1024 × 7040 23.5 → 17.5, 1065 × 1536 × 7488 51.5 → 42.2; GELU 300 × 3456 × 10944
    // 54.1 → 40.3). 128 × 128, two a CU, past that (1021 × 3072 54.9 → 40.3), and 128 × 256 on a full chip and many steps
    // (GELU, 4096 × 12288 385 against 396: one activation tile for twice the columns).
    if (cus <= 0) cus = 256;
    const float steps = (float)kt;
    const int slabs = glu ? (N / 2 + 31) / 32 : (N + 63) / 64;
    struct Tile { int tile, rows, slabs, at_once; float launch, group, chain, work; };
    static const Tile tiles[] = {
        {BLOCKS16_ROWS + 16, 16, 1, 4, 3.9f, 0.45f, 0.172f, 0.131f}, {BLOCKS16_ROWS + 32, 32, 1, 4, 4.1f, 0.65f, 0.195f, 0.142f},
        {BLOCKS16_ROWS + 48, 48, 1, 3, 4.1f, 0.92f, 0.255f, 0.180f}, {BLOCKS16_ROWS + 64, 64, 1, 2, 3.3f, 1.78f, 0.309f, 0.206f},
        {BLOCKS16_ROWS + 80, 80, 1, 2, 3.6f, 1.99f, 0.358f, 0.250f}, {BL_128x128, 128, 2, 2, 6.3f, 2.47f, 0.434f, 0.548f},
        {BL_128x256, 128, 4, 1, 2.0f, 7.70f, 0.814f, 0.992f},        {BL_64x256, 64, 4, 1, 2.0f, 5.00f, 0.524f, 0.608f}};
    float best = INFINITY;
    int tile = BL_128x256;
    for (const Tile &t : tiles) {
        const float n = ceilf(tile_count(M, t.rows, slabs, t.slabs) / (float)cus), at_once = (float)t.at_once;
        auto together = [&](float j) { return j > 0.0f ? j * t.group + steps * fmaxf(t.chain, j * t.work) : 0.0f; };
        const float full = floorf(n / at_once);
        const float us = t.launch + (t.at_once == 1 ? n * (t.group + steps * (n > 1.0f ? t.work : t.chain))
                                                    : full * together(at_once) + together(n - full * at_once));
        if (us < best) {
            best = us;
            tile = t.tile;
        }
    }
    return tile;
}

int64_t skinny_part_bytes(int M, int N, bool glu, int bm, int splits) {
    const long slabs = glu ? (N / 2 + 31) / 32 : (N + 63) / 64;
    const long tiles = (long)((M + bm - 1) / bm) * slabs;
    return (int64_t)splits * tiles * (2 * (bm / 32)) * 1024 * 4;
}

int choose_tile(int M, int N_out, bool glu, int cus) {
    // Tiles of 256 × 256 while they fill the CUs at least 3/4 of the way; 128 × 128 below.
    if (cus <= 0) cus = 256;
    const int n_virtual = glu ? 2 * N_out : N_out;
    const long big = (long)((M + 255) / 256) * ((n_virtual + 255) / 256);
    return big >= (long)cus * 3 / 4 ? TILE_256x256 : TILE_128x128;
}

hipError_t launch_gemm(const GemmArgs &p, bool fast, int tile, int wt, int wl, int epi, int out, hipStream_t stream) {
    if (!fast) return launch_general(p, wt, wl, epi, out, stream);
    if (wl != W_KN) return hipErrorInvalidValue;
    return wt == W_INT8 ? launch_fast_0(p, tile, epi, out, stream) : launch_fast_1(p, tile, epi, out, stream);
}

}  // namespace sq8
