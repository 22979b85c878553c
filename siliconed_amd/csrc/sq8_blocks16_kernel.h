// sq8_blocks16_kernel.h — the block-scaled product (sq8_blocks_kernel.h: GGUF Q8_0) where its 128 × 256 tiles are
// too few to fill the chip: one wave owns 16 columns for RB·16 rows, so the same output spreads over many more
// waves, without splitting K (every output's sums stay in K order, one fused rounding per block of 32:
// acc = fl(P·s + acc), the same bits as the 128 × 256 kernel's).
//
// v_mfma_f32_16x16x32_bf16 takes exactly one block of 32 K: P = A · q from zero, then four FMAs a lane per 16 rows
// (lane l: column l & 15, rows 4·(l >> 4) + e). Lane group q = l >> 4 holds k = 8q + [0, 8) of the block: in the
// packed Q8 layout those are bytes 8·(q >> 1) + [0, 8) of chunk (half q & 1), one 8-byte load; the activation's are
// chunk 4·kb + q of its 128-byte row.
//
// A workgroup is four waves on one 64-column slab; the activation tile (RB·16 rows of 64 K) goes through an LDS
// ring of NAS stages by direct loads, rows XOR-swizzled, its fragments read a step ahead; the codes and scales
// stream into registers PF steps ahead. What bounds it: the vector ALU (per wave and step 24 widening operations
// and 8 FMAs per 16 rows) where waves are many, the chain of K steps (0.18 µs a step at 16 rows, 0.38 at 80) where
// they are few. Measured against the 128 × 256 tiles (µs): 1 × 3072 × 3072 52.4 → 11.9, 77 × 3072 × 12288 54.0 → 21.9,
// 512 × 3072 × 3072 54.3 → 25.2, 148 × 9728 × 960 152 → 31.5. Not kept: fragments straight from global memory without
// the ring and its barriers (one row 10.6, but 17.4 at 16 rows and 70 against 33 at 77 × 12288: the four waves of a
// CU each fetch them), and taller tiles (96 rows 28 against 21.5 of 80 on one row: the registers end the overlap).
//
// Epilogue: the sums go through LDS as 64-column rows; all threads add the bias, activate and store four
// columns each (grp::store4), the kind of epilogue and the output type read at run time.
#pragma once

#include "sq8_blocks_kernel.h"

namespace sq8 {
namespace blk {

template <int RB, int NAS, int PF>
__global__ void __attribute__((amdgpu_flat_work_group_size(256, 256), amdgpu_waves_per_eu(2, 4)))
gemm_blocks16_kernel(const GemmArgs p) {
    constexpr int NW = 4;
    constexpr int BM = 16 * RB;
    constexpr int SA = BM * 128;                       // bytes per activation stage
    constexpr int A_BLOCKS = BM / 8;                   // 1 KB (8-row) blocks per stage
    constexpr int A_PER_WAVE = (A_BLOCKS + NW - 1) / NW;
    constexpr int WLD = 3;                             // two code loads and a scale load per step
    constexpr int OUT_PITCH = 64 * 4 + 16;             // bytes a row of 64 staged sums takes
    constexpr int LDS_BYTES = NAS * SA > BM * OUT_PITCH ? NAS * SA : BM * OUT_PITCH;
    // Loads in flight at the end of step t, A(t + 2) landed (its fragments are read in step t + 1): in issue order
    // per step s: A(s + NAS − 1), then W(s + PF).
    static_assert(PF >= NAS, "the codes run at least as far ahead as the activation");
    constexpr int STEP_WAIT = (NAS - 3) * (A_PER_WAVE + WLD) + WLD;
    static_assert(NAS >= 3 && STEP_WAIT < 64, "vmcnt budget");

    __shared__ __attribute__((aligned(1024))) uint8_t lds[LDS_BYTES];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int tm, tn;
    kern::tile_of(blockIdx.x, p.tiles_m, p.tiles_n, tm, tn);
    const int m0 = tm * BM;
    const bool glu = p.glu_half > 0;
    const int slabs = glu ? (p.glu_half + 31) / 32 : (p.N + 63) / 64;
    const int slab = tn;
    const int c = lane & 15, q = lane >> 4;
    const kern::gbytes Wg = (kern::gbytes)p.w;
    const int KT = p.kt;
    const int KW = p.kt_w > 0 ? p.kt_w : KT;           // the weight's steps (the fp32 route: three parts of them)

    // ---- codes (8 bytes per block of 32) and scales (both blocks of the step) of the lane's column ----
    const int vc = 16 * wave + c, half = vc >> 5, nl = vc & 31;  // virtual column of the slab
    const uint32_t w_off = (uint32_t)((int64_t)slab * KW * 4096) + half * 2048 + (nl + 32 * (q & 1)) * 16 + 8 * (q >> 1);
    const uint32_t s_off = (uint32_t)(scales_offset(slabs, KW) + (int64_t)slab * KW * 512) + nl * 16 + 8 * half;
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    u32x2 raw[PF][2];
    f32x2 sraw[PF];
    auto issue_w = [&](int t, auto buf) {
        constexpr int B = decltype(buf)::value;
        const int tt = wd::weight_step(p, min(t, KT - 1));
        const kern::gbytes base = Wg + (uint32_t)tt * 4096;
        raw[B][0] = kern::gld<u32x2>(base, w_off);
        raw[B][1] = kern::gld<u32x2>(base, w_off + 1024);
        sraw[B] = kern::gld<f32x2>(Wg + (uint32_t)tt * 512, s_off);
    };

    f32x4 acc[RB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) acc[rb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    // ---- activation: block b of 8 rows, lane → row 8b + lane/8, chunk lane%8 (the last loads of some waves
    // repeat one of their own blocks where the blocks do not split evenly) ----
    uint32_t a_goff[A_PER_WAVE];
    int a_blk[A_PER_WAVE];
#pragma unroll
    for (int i = 0; i < A_PER_WAVE; ++i) {
        int b = wave + NW * i;
        if constexpr (A_BLOCKS % NW != 0) b = b < A_BLOCKS ? b : A_BLOCKS >= NW ? b - NW : b % A_BLOCKS;
        a_blk[i] = b;
        const int r = 8 * b + (lane >> 3);
        const int lc = (lane & 7) ^ ((r ^ (r >> 3)) & 7);
        a_goff[i] = (uint32_t)((int64_t)min(m0 + r, p.M - 1) * p.lda * 2) + lc * 16;
    }
    const wd::i32x4 a_rsrc = wd::buffer_rsrc(p.a);
    auto issue_a = [&](int t, auto stage) {
        constexpr int S = decltype(stage)::value;
        const int soff = __builtin_amdgcn_readfirstlane((int)((uint32_t)min(t, KT - 1) * 128));
#pragma unroll
        for (int i = 0; i < A_PER_WAVE; ++i)
            wd::raw_buffer_load_lds(a_rsrc, (wd::lds_u32)(lds + S * SA + a_blk[i] * 1024), 16, (int)a_goff[i], soff, 0, 0);
    };

    // Fragment (row block rb, K block kb): row 16·rb + (lane & 15), chunk 4·kb + q. The swizzle of row r + 16·rb is
    // r's with bits 1 and 2 flipped by rb's low bits.
    int xo[4][2];
#pragma unroll
    for (int rb = 0; rb < 4; ++rb)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) xo[rb][kb] = wd::swz(16 * rb + c, 4 * kb + q) - 16 * 128 * rb;

    bf16x8 xf[2][RB][2];  // fragments of the step and of the next one
    auto read_x = [&](auto stage, auto dst) {
        constexpr int S = decltype(stage)::value, D = decltype(dst)::value;
        static_for<0, RB>([&](auto rc) {
            constexpr int rb = decltype(rc)::value;
            static_for<0, 2>([&](auto kc) {
                constexpr int kb = decltype(kc)::value;
                xf[D][rb][kb] = kern::lds_load_frag(lds + S * SA + 16 * 128 * rb, xo[rb & 3][kb]);
            });
        });
    };

    // Prologue: the loads of the steps before the loop in its issue order — A(0), A(1), then A(s), W(s) pairs
    // (kept in it: the compiler would move the codes' loads past the others, and the waits count on the order).
    __builtin_amdgcn_sched_barrier(0);
    issue_a(0, std::integral_constant<int, 0>{});
    issue_a(1, std::integral_constant<int, 1>{});
    __builtin_amdgcn_sched_barrier(0);
    static_for<0, PF>([&](auto vc_) {
        constexpr int v = decltype(vc_)::value;
        // W(v) belongs to step v − PF, whose A is A(v − PF + NAS − 1).
        constexpr int a = v - PF + NAS - 1;
        if constexpr (a >= 2) issue_a(a, std::integral_constant<int, a>{});
        __builtin_amdgcn_sched_barrier(0);
        issue_w(v, vc_);
        __builtin_amdgcn_sched_barrier(0);
    });
    wait_vmcnt<STEP_WAIT>();
    step_barrier();
    read_x(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{});

    // Step t: activation stage t mod NAS, code buffer t mod PF, fragments t mod 2. TAIL: one of the last steps, whose code
    // loads no later step uses and the compiler drops: the wait counts the activation's loads only.
    auto step = [&](int t, auto uc, auto tail) {
        constexpr bool TAIL = decltype(tail)::value;
        constexpr int U = decltype(uc)::value;
        constexpr int S = U % NAS, P = U % PF, D = U & 1;
        __builtin_amdgcn_sched_barrier(0);
        // Into the stage of step t − 1, whose fragments were read during step t − 2 (two barriers ago); the next step's
        // fragments come from a stage that the previous barrier published.
        issue_a(t + NAS - 1, std::integral_constant<int, (S + NAS - 1) % NAS>{});
        read_x(std::integral_constant<int, (S + 1) % NAS>{}, std::integral_constant<int, 1 - D>{});
        f32x4 pp[2][RB];
        static_for<0, 2>([&](auto kc) {
            constexpr int kb = decltype(kc)::value;
            const bf16x8 w = widen8<W_INT8>(raw[P][kb][0], raw[P][kb][1]);
            static_for<0, RB>([&](auto rc) {
                constexpr int rb = decltype(rc)::value;
                pp[kb][rb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[D][rb][kb], w, f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
            });
        });
        const f32x2 s = sraw[P];
        static_for<0, 2>([&](auto kc) {
            constexpr int kb = decltype(kc)::value;
            static_for<0, RB>([&](auto rc) {
                constexpr int rb = decltype(rc)::value;
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[rb][e] = __builtin_fmaf(pp[kb][rb][e], s[kb], acc[rb][e]);
            });
        });
        __builtin_amdgcn_sched_barrier(0);
        issue_w(t + PF, std::integral_constant<int, P>{});
        __builtin_amdgcn_sched_barrier(0);
        wait_vmcnt<TAIL ? (NAS - 3) * A_PER_WAVE : STEP_WAIT>();
        step_barrier();
    };
    // The stages, buffers and fragment halves repeat every lcm(NAS, PF, 2) steps.
    constexpr int CYCLE = PF % NAS == 0 && PF % 2 == 0 ? PF : 2 * NAS * PF;
    static_assert(CYCLE <= 16, "unrolled steps");
    int t = 0;
    for (; t + CYCLE <= KT; t += CYCLE) static_for<0, CYCLE>([&](auto uc) { step(t + decltype(uc)::value, uc, std::false_type{}); });
    static_for<0, CYCLE - 1>([&](auto uc) {
        constexpr int u = decltype(uc)::value;
        if (t + u < KT) step(t + u, uc, std::true_type{});
    });
    wait_vmcnt<0>();
    __syncthreads();

    // ---- epilogue: sums to LDS [row][64 virtual columns], then four output columns a thread ----------------
    static_for<0, RB>([&](auto rc) {
        constexpr int rb = decltype(rc)::value;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            *reinterpret_cast<float *>(lds + (16 * rb + 4 * q + e) * OUT_PITCH + vc * 4) = acc[rb][e];
    });
    __syncthreads();
    const int n_out = glu ? p.glu_half : p.N;
    const int per_row = glu ? 8 : 16;                  // chunks of four output columns
    const int chunk = tid & (per_row - 1);
    const int col = slab * (glu ? 32 : 64) + 4 * chunk;
    const bool has_bias = p.bias != nullptr;
    float bi[4], bu[4];
    if (col < n_out) {
        grp::column4(p.bias, true, p.sb_vec, col, n_out, 0, bi);
        if (glu) grp::column4(p.bias, true, p.sb_vec, col, n_out, p.glu_half, bu);
    }
    for (int row = tid / per_row; row < BM; row += 256 / per_row) {
        const int m = m0 + row;
        if (m >= p.M || col >= n_out) break;
        const f32x4 x = *reinterpret_cast<const f32x4 *>(lds + row * OUT_PITCH + 16 * chunk);
        float v[4], u[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = has_bias ? __fadd_rn(x[e], bi[e]) : x[e];
        if (glu) {
            const f32x4 y = *reinterpret_cast<const f32x4 *>(lds + row * OUT_PITCH + 128 + 16 * chunk);
#pragma unroll
            for (int e = 0; e < 4; ++e) u[e] = has_bias ? __fadd_rn(y[e], bu[e]) : y[e];
        }
        grp::activate4(p.epi, v, u);
        grp::store4(p, grp::out4(p, col, n_out), m * grp::row_bytes(p), col, n_out, v);
    }
}

template <int RB, int NAS, int PF>
hipError_t launch_blocks16(const GemmArgs &args, int epi, int out, hipStream_t stream) {
    GemmArgs p = args;
    p.epi = epi;
    p.out = out;
    p.tiles_m = (p.M + 16 * RB - 1) / (16 * RB);
    p.tiles_n = p.glu_half > 0 ? (p.glu_half + 31) / 32 : (p.N + 63) / 64;
    const int blocks = p.tiles_m * p.tiles_n;
    if (blocks == 0) return hipSuccess;
    hipLaunchKernelGGL((gemm_blocks16_kernel<RB, NAS, PF>), dim3(blocks), dim3(256), 0, stream, p);
    return hipGetLastError();
}

}  // namespace blk
}  // namespace sq8
