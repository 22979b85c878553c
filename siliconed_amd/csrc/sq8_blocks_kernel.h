// sq8_blocks_kernel.h — the gfx950 product on codes with a scale per block of rows and column (GGUF
// Q8_0: int8 q [K, N], fp32 s [K/B, N], B = 32 or a multiple of it):
//
//     C = act(A · W + b),  W[k, n] = q[k, n] · s[k / B, n]
//
// (Sources/Siliconed/TensorGEMM.swift:137-171, `linear_q8`, which widens q · s into threadgroup
// memory and multiplies in fp32). Here the codes go to bf16 MFMAs as they are (exact), and each
// block's fp32 partial sum is scaled once it is complete:
//
//     C[m, n] = Σ_blocks s[blk, n] · (Σ_{k ∈ blk} a[m, k] · q[k, n])
//
// equal to the reference's sum in exact arithmetic, rounded differently: one fp32 product and sum
// per block instead of one fp32 product per weight.
//
// The weight-direct kernel's structure (sq8_wdirect_kernel.h: activation tiles through an LDS ring, each wave
// streaming its packed codes straight into registers) with these differences:
//   * the activation is the MFMA's first operand and the codes the second, so each lane's 16
//     results of a 32 × 32 block share one column (lane & 31) and one scale per block of K;
//   * a 64-step's K order keeps each block of 32 in two MFMA sub-steps: sub-step ks takes
//     k ∈ [16·ks, 16·ks + 16), lane half h the 8 at 16·ks + 8·h — the packed Q8 layout stores the
//     codes in that order, the activation fragment of (ks, h) is LDS chunk 2·ks + h;
//   * per block: P = MFMA(A, q) over its two sub-steps (from zero), then acc += P · s (fp32 FMA).
//
// What bounds it, and the schedule. Per MFMA (32 cycles of a SIMD's matrix core) a wave issues 8 rescale FMAs and
// 3 widening operations, 44 cycles of the vector ALU: the kernel can only approach the vector ALU's time if the two
// run side by side, and waves that run all their MFMAs and then all their FMAs, in step with each other between
// barriers, add them (measured: 32 + 54 cycles). So the step is cut into four groups of one K block × two row
// blocks: a group issues its four MFMAs (P of this group), and between them the 32 FMAs of the group before (whose P
// is complete), a quarter of the widening and the next group's four fragment reads; the groups run on across steps
// (the next step's first fragments and codes are taken during the last group). The order of every sum is unchanged.
// Measured (µs, the groups against the plain order): one row of tiles alone, K = 3072, 52.4 → 46.5 in 128 × 256 and
// 33.6 in 128 × 128; 1021 × 3072 × 3072 54.9 → 40.3 (128 × 128, two workgroups a CU: one's epilogue under the other's
// MFMAs). On a full chip the two still add (4096 × 3072 × 12288: 81.5 cycles an MFMA, 32 + 12.7 vector instructions of 4),
// 400 → 378 to 391 µs; a fifth of that is the clock under power (303 µs with every activation or every
// code zero).
// 64 × 256 tiles (two row blocks a wave: two groups a step, each widening a whole K block) serve products that leave a
// round of the taller ones part empty: SiLU-GLU 575 × 1024 × 7040 17.5 µs (28 tiles of 128 × 256 a row 23.5), 1065 ×
// 1536 × 7488 42.2 (128 × 128 51.5).
// Measured and not kept: eight activation stages with a barrier every two steps (402 against 406 µs, two registers
// spilled).
//
// Packed Q8 layout (sq8_pack_blocks): the codes as the packed layout's chunks — chunk c =
// ((slab·kt + t)·4 + j)·64 + lane, 16 bytes: k = 64t + 32(j&1) + 8h + [0, 8) then
// 64t + 32(j&1) + 16 + 8h + [0, 8) of virtual column 32(j>>1) + (lane & 31) — then, at byte
// slabs·kt·4096, the scales: per (slab, t), per column nl < 32, 16 bytes {s(block 0 of the step,
// column nl), s(block 1, nl), s(block 0, 32 + nl), s(block 1, 32 + nl)} (virtual columns; GLU:
// the slab's 32 output columns of each half). Zeros past K and past the columns.
#pragma once

#include "sq8_group_kernel.h"

namespace sq8 {
namespace blk {

using wd::BK;
using wd::glb_ptr;
using wd::lds_ptr;
using wd::step_barrier;
using wd::swz;
using wd::wait_vmcnt;
using wd::widen8;

// Byte offset of the packed scales of a weight of kt steps and `slabs` slabs from the packed base.
__host__ __device__ inline int64_t scales_offset(int64_t slabs, int64_t kt) { return slabs * kt * 4096; }

template <int BM, int NW>
__global__ void __attribute__((amdgpu_flat_work_group_size(64 * NW, 64 * NW), amdgpu_waves_per_eu(2, 2)))
gemm_blocks_kernel(const GemmArgs p) {
    static_assert(NW % 2 == 0, "wave w: block w & 1 of slab w ÷ 2 of the tile's");
    constexpr int FM = BM / 32;
    static_assert(FM % 2 == 0, "row blocks in pairs");
    constexpr int NAS = 4;                    // activation stages and code buffers
    constexpr int SA = BM * 128;
    constexpr int A_PER_WAVE = BM / 8 / NW;
    static_assert(BM / 8 % NW == 0, "the activation blocks split evenly over the waves");
    constexpr int GROUPS = FM;                // groups a step: two K blocks × FM/2 pairs of row blocks
    static_assert(A_PER_WAVE <= GROUPS, "a group issues one activation load, the one before the last a second");
    constexpr int WLOADS = 3;                 // two code loads and a scale load per step
    constexpr int LDS_BYTES = NAS * SA > NW * grp::SLOT ? NAS * SA : NW * grp::SLOT;

    __shared__ __attribute__((aligned(1024))) uint8_t lds[LDS_BYTES];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int tm, tn;
    kern::tile_of(blockIdx.x, p.tiles_m, p.tiles_n, tm, tn);
    const int m0 = tm * BM;
    const bool glu = p.glu_half > 0;
    const int slabs = glu ? (p.glu_half + 31) / 32 : (p.N + 63) / 64;
    const int slab = min(tn * (NW / 2) + (wave >> 1), slabs - 1);  // a wave past the last slab reads the last
    const int b0 = wave & 1;
    const kern::gbytes Wg = (kern::gbytes)p.w;
    const int KT = p.kt;

    uint32_t a_goff[A_PER_WAVE];
#pragma unroll
    for (int i = 0; i < A_PER_WAVE; ++i) {
        const int r = 8 * (wave + NW * i) + (lane >> 3);
        const int lc = (lane & 7) ^ ((r ^ (r >> 3)) & 7);
        a_goff[i] = (uint32_t)((int64_t)min(m0 + r, p.M - 1) * p.lda * 2) + lc * 16;
    }
    const wd::i32x4 a_rsrc = wd::buffer_rsrc(p.a);
    auto issue_a1 = [&](int t, auto stage, auto ic) {  // load ic of step t
        constexpr int S = decltype(stage)::value, i = decltype(ic)::value;
        const int soff = __builtin_amdgcn_readfirstlane((int)((uint32_t)min(t, KT - 1) * 128));
        wd::raw_buffer_load_lds(a_rsrc, (wd::lds_u32)(lds + S * SA + (wave + NW * i) * 1024), 16, (int)a_goff[i], soff, 0, 0);
    };
    auto issue_a = [&](int t, auto stage) {
        static_for<0, A_PER_WAVE>([&](auto ic) { issue_a1(t, stage, ic); });
    };

    // Codes: 2 × 16 bytes per lane per step (the two K blocks); scales: the lane's column's two, 8 bytes. The weight's
    // K steps: KT, or kt_w when the activation holds several parts along K that each face the whole weight (the fp32
    // route), the weight's step then t modulo kt_w.
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    const int KW = p.kt_w > 0 ? p.kt_w : KT;
    const uint32_t w_off = (uint32_t)((int64_t)slab * KW * 4096) + b0 * 2048 + lane * 16;
    const uint32_t s_off = (uint32_t)(scales_offset(slabs, KW) + (int64_t)slab * KW * 512) + (lane & 31) * 16 + 8 * b0;
    u32x4 raw[NAS][2];
    f32x2 sraw[NAS];
    auto issue_w = [&](int t, auto buf) {
        constexpr int B = decltype(buf)::value;
        const int tt = wd::weight_step(p, min(t, KT - 1));
        const kern::gbytes base = Wg + (uint32_t)tt * 4096;
        raw[B][0] = kern::gld<u32x4>(base, w_off);
        raw[B][1] = kern::gld<u32x4>(base, w_off + 1024);
        sraw[B] = kern::gld<f32x2>(Wg + (uint32_t)tt * 512, s_off);
    };

    const int h = lane >> 5;
    int xo[2][4];
#pragma unroll
    for (int par = 0; par < 2; ++par)
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) xo[par][ks] = swz(32 * par + (lane & 31), 2 * ks + h) - 32 * 128 * par;

    f32x16 acc[FM];
    f32x16 pp[2][2];       // [group & 1][row block of the pair]
    bf16x8 xf[2][2][2];    // [group & 1][row block of the pair][sub-step of the K block]
    bf16x8 wk[2][2];       // [K block][sub-step]
#pragma unroll
    for (int bm = 0; bm < FM; ++bm)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[bm][r] = 0.0f;
    // The first step's "group before": sums of zero.
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) pp[1][i][r] = 0.0f;
    float sp = 0.0f;       // the scale of the group before

    auto read_x = [&](auto stage, auto gc, auto dst) {  // group gc's fragments
        constexpr int S = decltype(stage)::value, g = decltype(gc)::value, D = decltype(dst)::value;
        constexpr int kb = g / (FM / 2), pair = g % (FM / 2);
        static_for<0, 2>([&](auto kc) {
            constexpr int ks = decltype(kc)::value;
            static_for<0, 2>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                xf[D][i][ks] = kern::lds_load_frag(lds + S * SA + 32 * 128 * (2 * pair + i), xo[i][2 * kb + ks]);
            });
        });
    };
    auto widen = [&](auto buf, auto bc, auto kc) {
        constexpr int B = decltype(buf)::value, kb = decltype(bc)::value, ks = decltype(kc)::value;
        wk[kb][ks] = widen8<W_INT8>(raw[B][kb][2 * ks], raw[B][kb][2 * ks + 1]);
    };
    auto rescale = [&](auto gc, float s) {  // group gc's P into the totals
        constexpr int g = decltype(gc)::value, pair = g % (FM / 2);
        static_for<0, 2>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[2 * pair + i][r] = __builtin_fmaf(pp[g & 1][i][r], s, acc[2 * pair + i][r]);
        });
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;

    // Prologue: W(0 .. 2) and A(0 .. 2), all landed (the compiler's own waits for the codes of the first steps then
    // count from here; behind loads in flight they would drain the loop's prefetch too).
    static_for<0, NAS - 1>([&](auto vc) { issue_w(decltype(vc)::value, vc); });
    static_for<0, NAS - 1>([&](auto vc) { issue_a(decltype(vc)::value, vc); });
    wait_vmcnt<0>();
    step_barrier();
    read_x(I0{}, I0{}, I0{});
    widen(I0{}, I0{}, I0{});
    widen(I0{}, I0{}, I1{});

    // Step t on stage and code buffer U = t mod 4. TAIL: one of the last steps, whose code loads no later step uses and the
    // compiler drops: the wait counts the activation's loads only (as if every code load had been dropped).
    auto step = [&](int t, auto uc, auto tail) {
        constexpr bool TAIL = decltype(tail)::value;
        constexpr int U = decltype(uc)::value;
        using SU = std::integral_constant<int, U>;
        using S1 = std::integral_constant<int, (U + 1) % NAS>;
        using S3 = std::integral_constant<int, (U + 3) % NAS>;
        static_for<0, GROUPS>([&](auto gc) {
            constexpr int g = decltype(gc)::value, kb = g / (FM / 2), pair = g % (FM / 2);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (g + 1 < GROUPS)
                read_x(SU{}, std::integral_constant<int, g + 1>{}, std::integral_constant<int, (g + 1) & 1>{});
            else
                read_x(S1{}, I0{}, I0{});  // the next step's first
            // The next K block's codes: one sub-step each in the K block's last two groups (both where it has one).
            static_for<0, 2>([&](auto ks) {
                if constexpr (FM == 2 || pair == FM / 2 - 2 + decltype(ks)::value) {
                    if constexpr (kb == 0) widen(SU{}, I1{}, ks);
                    else widen(S1{}, I0{}, ks);
                }
            });
            // Into the stage and buffer last read during step t − 1 (its barrier saw every wave's reads): the activation's loads
            // in the groups before the last, the code loads in the last, so that the step's wait counts them in this order
            // (within a group the compiler orders loads as it likes).
            if constexpr (g < A_PER_WAVE && g < GROUPS - 1) issue_a1(t + 3, S3{}, gc);
            if constexpr (g == GROUPS - 2 && A_PER_WAVE == GROUPS) issue_a1(t + 3, S3{}, std::integral_constant<int, GROUPS - 1>{});
            if constexpr (g == GROUPS - 1) issue_w(t + 3, S3{});
            static_for<0, 2>([&](auto kc) {
                constexpr int ks = decltype(kc)::value;
                static_for<0, 2>([&](auto ic) {
                    constexpr int i = decltype(ic)::value;
                    if constexpr (ks == 0)
                        pp[g & 1][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xf[g & 1][i][0], wk[kb][0], f32x16{}, 0, 0, 0);
                    else
                        pp[g & 1][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xf[g & 1][i][1], wk[kb][1], pp[g & 1][i], 0, 0, 0);
                });
            });
            rescale(std::integral_constant<int, (g + GROUPS - 1) % GROUPS>{}, sp);
            sp = sraw[U][kb];
            static_for<0, 4>([&](auto) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, FM == 2 ? 8 : 6, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, FM == 2 ? 6 : 5, 0);
                __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
            });
            __builtin_amdgcn_sched_barrier(0);
        });
        // A(t + 2) landed: W(t + 2) and step t + 3's loads may fly.
        wait_vmcnt<A_PER_WAVE + (TAIL ? 0 : 2 * WLOADS)>();
        step_barrier();
    };
    int t = 0;
    for (; t + NAS <= KT; t += NAS) static_for<0, NAS>([&](auto uc) { step(t + decltype(uc)::value, uc, std::false_type{}); });
    static_for<0, NAS - 1>([&](auto uc) {
        if (t + decltype(uc)::value < KT) step(t + decltype(uc)::value, uc, std::true_type{});
    });
    rescale(std::integral_constant<int, GROUPS - 1>{}, sp);
    wait_vmcnt<0>();
    __syncthreads();

    // ---- epilogue: 32 rows at a time through LDS, then four columns a thread, whole rows of the tile ----------
    // A thread's column (and so its bias) is the same for every row block.
    const int n_out = glu ? p.glu_half : p.N;
    const int cols = (glu ? 16 : 32) * NW, per_row = cols / 4;
    const int chunk = tid % per_row;
    const int col = tn * cols + 4 * chunk, blk = chunk >> 3;   // blk: the 32-column output block
    const bool has_bias = p.bias != nullptr;
    const grp::Out4 to = grp::out4(p, min(col, n_out - 1), n_out);
    const int64_t row_bytes = grp::row_bytes(p);
    float bi[4], bu[4];
    if (col < n_out) {
        grp::column4(p.bias, true, p.sb_vec, col, n_out, 0, bi);
        if (glu) grp::column4(p.bias, true, p.sb_vec, col, n_out, p.glu_half, bu);
    }
    static_for<0, FM>([&](auto bmc) {
        constexpr int bm = decltype(bmc)::value;
#pragma unroll
        for (int r = 0; r < 16; ++r)  // row 8·(r >> 2) + 4h + (r & 3), column lane & 31 of the wave's block
            *reinterpret_cast<float *>(lds + wave * grp::SLOT + (8 * (r >> 2) + 4 * h + (r & 3)) * grp::PITCH + (lane & 31) * 4) =
                acc[bm][r];
        __syncthreads();
        if (col < n_out) {
            const uint8_t *src = lds + (glu ? 2 * blk : blk) * grp::SLOT + (chunk & 7) * 16;
            for (int row = tid / per_row; row < 32; row += 64 * NW / per_row) {
                const int m = m0 + 32 * bm + row;
                if (m >= p.M) break;
                const f32x4 x = *reinterpret_cast<const f32x4 *>(src + row * grp::PITCH);
                float v[4], u[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = has_bias ? __fadd_rn(x[e], bi[e]) : x[e];
                if (glu) {
                    const f32x4 y = *reinterpret_cast<const f32x4 *>(src + grp::SLOT + row * grp::PITCH);
#pragma unroll
                    for (int e = 0; e < 4; ++e) u[e] = has_bias ? __fadd_rn(y[e], bu[e]) : y[e];
                }
                grp::activate4(p.epi, v, u);
                grp::store4(p, to, m * row_bytes, col, n_out, v);
            }
        }
        if constexpr (bm + 1 < FM) __syncthreads();
    });
}

template <int BM, int NW>
hipError_t launch_blocks_product(const GemmArgs &args, int epi, int out, hipStream_t stream) {
    GemmArgs p = args;
    p.epi = epi;
    p.out = out;
    p.tiles_m = (p.M + BM - 1) / BM;
    const int slabs = p.glu_half > 0 ? (p.glu_half + 31) / 32 : (p.N + 63) / 64;
    p.tiles_n = (slabs + NW / 2 - 1) / (NW / 2);
    const int blocks = p.tiles_m * p.tiles_n;
    if (blocks == 0) return hipSuccess;
    hipLaunchKernelGGL((gemm_blocks_kernel<BM, NW>), dim3(blocks), dim3(64 * NW), 0, stream, p);
    return hipGetLastError();
}

}  // namespace blk
}  // namespace sq8
