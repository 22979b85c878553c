// sq8_group_kernel.h — products whose output tiles are too few to fill the chip: each workgroup's K
// steps split over KS groups of NW waves (group g takes the steps g, g + KS, …, with its own activation
// stages), so one workgroup a CU holds eight waves and their loads in flight whatever its tile; the groups'
// sums meet in LDS and are added in group order (deterministic; exact for int32).
//
// Three kinds of product (MATH):
//   GM_BF16 — bf16 activation × 8-bit codes widened to bf16 (sq8_wdirect_kernel.h's arithmetic, K steps of 64;
//             every K-group count a family of bits of its own, the same over all tile shapes);
//   GM_F32  — the same codes under an fp32 activation's three bf16 parts along K (the fp32 route): a weight step's
//             codes are loaded and widened once and meet the three parts' activation steps in turn (as 3·K steps each
//             code is loaded and widened three times); the steps split over the groups are the weight's;
//   GM_I8   — int8 activation codes × int8 codes, int32 sums (sq8_i8_kernel.h's, K steps of 128): the same
//             bits as every other W8A8 kernel whatever the split.
// Both stage 128 bytes of every activation row per K step, so the rings, swizzles and direct loads are shared.
// A wave owns one 32-column block (half a slab of the packed layout) for all BM rows: twice the waves of a
// 64-column one for the same tile, and the waves' loads in flight are what these shapes are short of.
//
// Epilogue: a row block (32 rows) at a time, every wave writes its sums to LDS as they are, then all the
// workgroup's threads add the groups' sums, scale, bias, activate and store, four columns a thread (GLU: the gate
// block's and the up block's, neighbouring waves'). The kind of
// epilogue and the output type are read at run time (p.epi, p.out): they are a few instructions per four
// values here, and one kernel a tile then serves them all (nine instances a tile compiled for minutes).
#pragma once

#include "sq8_i8_kernel.h"

namespace sq8 {
namespace grp {

using wd::BK;
using wd::buffer_rsrc;
using wd::lds_u32;
using wd::raw_buffer_load_lds;
using wd::step_barrier;
using wd::swz;
using wd::wait_vmcnt;

constexpr int PITCH = 144;           // bytes a row of 32 staged sums takes (16-byte aligned, banks spread)
constexpr int SLOT = 32 * PITCH;     // one 32 × 32 block of sums

constexpr int lds_bytes(int bm, int nw, int ks, int nas) {
    const int stages = ks * nas * bm * 128, sums = ks * nw * SLOT;
    return stages > sums ? stages : sums;
}

// Where four output columns [col, col + 4) go, rows 0: in the residual stream, or the output tensor and head out_index says;
// `whole`: all four at at[0], aligned for one store. Worked out once a thread, before the row blocks: out_index divides
// (by the split and the head), and its code in every row block's stores made kernels of up to 61 KB (now 46), which each
// product reads past a cold instruction cache: 432 × 2048 × 8192 with GELU inside a block 27.1 → 25.5 µs. (A loop over the row
// blocks, 33 KB, 26.3 there, but 0.5 µs more on every product alone.)
struct Out4 {
    uint8_t *at[4];
    bool whole;
};

__device__ __forceinline__ Out4 out4(const GemmArgs &p, int col, int n_out) {
    Out4 o;
    if (p.epi == EPI_RESIDUAL) {
        o.whole = p.c_vec16 && col + 4 <= n_out;
#pragma unroll
        for (int e = 0; e < 4; ++e) o.at[e] = reinterpret_cast<uint8_t *>(p.c[0]) + (int64_t)(col + e) * 4;
        return o;
    }
    const int esz = p.out == OUT_F32 ? 4 : 2;
    o.whole = p.c_vec && col + 4 <= n_out && (p.split % 4) == 0;  // the four in one output and head
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        if (e > 0 && o.whole) {
            o.at[e] = o.at[0];
        } else {
            int which = 0;
            const int64_t off = p.split > 0 || p.head_dim > 0 ? wd::out_index(p, 0, min(col + e, n_out - 1), which) : col + e;
            o.at[e] = kern::out_base(p, which) + off * esz;
        }
    }
    return o;
}

// Bytes from one output row to the next.
__device__ __forceinline__ int64_t row_bytes(const GemmArgs &p) {
    return p.epi == EPI_RESIDUAL ? p.ldc * 4 : (p.head_dim > 0 ? p.head_dim : p.ldc) * (p.out == OUT_F32 ? 4 : 2);
}

// Stores the values v (scaled, biased, activated) of columns [col, col + 4), `row` bytes past their rows 0.
__device__ __forceinline__ void store4(const GemmArgs &p, const Out4 &o, int64_t row, int col, int n_out, const float (&v)[4]) {
    if (p.epi == EPI_RESIDUAL) {
        if (o.whole) {
            float *xr = reinterpret_cast<float *>(o.at[0] + row);
            const f32x4 xv = *reinterpret_cast<const f32x4 *>(xr);
            const f32x4 gv = p.gate ? *reinterpret_cast<const f32x4 *>(p.gate + col) : f32x4{1.0f, 1.0f, 1.0f, 1.0f};
            f32x4 y;
#pragma unroll
            for (int e = 0; e < 4; ++e) y[e] = __fadd_rn(xv[e], __fmul_rn(gv[e], v[e]));
            *reinterpret_cast<f32x4 *>(xr) = y;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (col + e < n_out) {
                    float *xr = reinterpret_cast<float *>(o.at[e] + row);
                    *xr = __fadd_rn(*xr, __fmul_rn(p.gate ? p.gate[col + e] : 1.0f, v[e]));
                }
        }
    } else if (o.whole) {
        if (p.out == OUT_F32)
            *reinterpret_cast<f32x4 *>(o.at[0] + row) = f32x4{v[0], v[1], v[2], v[3]};
        else
            *reinterpret_cast<u32x2 *>(o.at[0] + row) = u32x2{pack_bf16_rne(v[0], v[1]), pack_bf16_rne(v[2], v[3])};
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (col + e >= n_out) break;
            if (p.out == OUT_F32)
                *reinterpret_cast<float *>(o.at[e] + row) = v[e];
            else
                *reinterpret_cast<uint16_t *>(o.at[e] + row) = (uint16_t)(pack_bf16_rne(v[e], 0.0f) & 0xFFFFu);
        }
    }
}

// The activation of four finished values (GLU: with the up half's four `u`), as block_values applies it.
__device__ __forceinline__ void activate4(int epi, float (&v)[4], const float (&u)[4]) {
    if (epi == EPI_GELU) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = gelu_tanh(v[e]);
    } else if (epi == EPI_SILU_GLU) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = silu_glu(v[e], u[e]);
    } else if (epi == EPI_SITU_GLU) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = situ(v[e], u[e]);
    }
}

// Four scales or biases of columns [col, col + 4) (clamped to the last of n_out; `off`: the GLU half).
__device__ __forceinline__ void column4(const float *src, bool per_column, bool vec, int col, int n_out, int off,
                                        float (&v)[4]) {
    if (!src) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = 0.0f;
    } else if (!per_column) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = src[0];
    } else if (vec && col + 4 <= n_out) {
        const f32x4 t = *reinterpret_cast<const f32x4 *>(src + col + off);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = t[e];
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = src[min(col + e, n_out - 1) + off];
    }
}

template <int MATH, int WT, int WL, int BM, int NW, int KS, int NAS>
__global__ void __attribute__((amdgpu_flat_work_group_size(64 * NW * KS, 64 * NW * KS),
                               amdgpu_waves_per_eu(NW *KS / 4, NW *KS / 4)))
gemm_group_kernel(const GemmArgs p) {
    static_assert(NW * KS % 4 == 0, "the workgroup's waves spread evenly over the four SIMDs");
    constexpr bool I8 = MATH == GM_I8, F32 = MATH == GM_F32;
    constexpr int FM = BM / 32;
    constexpr int SA = BM * 128;                 // bytes per activation stage
    // 1 KB direct loads per wave per step; where the blocks do not split evenly over a group's waves the last loads
    // of some repeat one of their own blocks, so every wave issues the same count (one vmcnt value fits them all).
    constexpr int A_BLOCKS = BM / 8;
    constexpr int A_PER_WAVE = (A_BLOCKS + NW - 1) / NW;
    constexpr int WLD = I8 ? 4 : 2;              // 16-byte weight loads per lane per step
    constexpr int THREADS = 64 * NW * KS;
    using acc_t = std::conditional_t<I8, wd::i32x16, f32x16>;
    using v4 = std::conditional_t<I8, wd::i32x4, f32x4>;
    // Loads a wave may leave in flight at the end of step t, A(t+1) and W(t+1) landed.
    constexpr int STEP_WAIT = WLD + (NAS - 2) * (A_PER_WAVE + WLD);
    static_assert(STEP_WAIT < 64, "vmcnt budget");
    static_assert(!F32 || NAS == 3, "the fp32 route's activation stages are its three parts");
    constexpr int NWB = F32 ? 2 : NAS;           // code buffers

    __shared__ __attribute__((aligned(1024))) uint8_t lds[lds_bytes(BM, NW, KS, NAS)];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave_all = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int group = wave_all / NW, wave = wave_all - group * NW;
    uint8_t *const ldg = lds + group * (NAS * SA);
    int tm, tn;
    kern::tile_of(blockIdx.x, p.tiles_m, p.tiles_n, tm, tn);
    const int m0 = tm * BM;
    const bool glu = p.glu_half > 0;             // NW even only (the launcher's rule): a pair of blocks is one tile's
    const int slab = (tn * NW + wave) >> 1, b0 = (tn * NW + wave) & 1;  // the wave's block: b0 of slab
    const kern::gbytes Wg = (kern::gbytes)p.w;
    const int KT = F32 ? p.kt_w : p.kt;          // the weight's steps

    // ---- activation: wave block b = wave + NW·i of 8 rows, lane → row 8b + lane/8, chunk lane%8 ----
    uint32_t a_goff[A_PER_WAVE];
    int a_blk[A_PER_WAVE];
#pragma unroll
    for (int i = 0; i < A_PER_WAVE; ++i) {
        int b = wave + NW * i;
        if constexpr (A_BLOCKS % NW != 0) b = b < A_BLOCKS ? b : b - NW;
        a_blk[i] = b;
        const int r = 8 * b + (lane >> 3);
        const int lc = (lane & 7) ^ ((r ^ (r >> 3)) & 7);
        const int row = min(m0 + r, p.M - 1);
        a_goff[i] = (uint32_t)((int64_t)row * p.lda * (I8 ? 1 : 2)) + lc * 16;
    }
    const wd::i32x4 a_rsrc = buffer_rsrc(p.a);
    auto issue_a = [&](int t, auto stage) {
        constexpr int S = decltype(stage)::value;
        // Fp32 route: t counts activation steps, three (stages 0, 1, 2: the parts, KT · 128 bytes apart) a weight step.
        const int soff = __builtin_amdgcn_readfirstlane(
            (int)((uint32_t)min((F32 ? t / 3 : t) * KS + group, KT - 1) * 128 + (F32 ? (uint32_t)(S * KT) * 128 : 0u)));
#pragma unroll
        for (int i = 0; i < A_PER_WAVE; ++i)
            raw_buffer_load_lds(a_rsrc, (lds_u32)(ldg + S * SA + a_blk[i] * 1024), 16, (int)a_goff[i], soff, 0, 0);
    };

    // ---- weight: WLD × 16 bytes per lane per step, straight into registers ---------------------------
    // Load j of a packed step: half j of the block's codes (W8A8: two packed steps).
    uint32_t w_off[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        if constexpr (WL == W_PACKED) {
            const int slabs = glu ? (p.glu_half + 31) / 32 : (p.N + 63) / 64;
            const int s = slab < slabs ? slab : slabs - 1;
            const int kt = I8 ? p.kt_w : KT;
            w_off[j] = (uint32_t)(((int64_t)s * kt * 4 + 2 * b0 + j) * 1024 + lane * 16);
        } else {
            const int hl = lane >> 5, nl = lane & 31;
            const int n = glu ? min(slab * 32 + nl, p.glu_half - 1) + b0 * p.glu_half : min(slab * 64 + b0 * 32 + nl, p.N - 1);
            w_off[j] = (uint32_t)((int64_t)n * p.ldw + 32 * hl + 16 * j);
        }
    }
    constexpr uint32_t w_step = WL == W_PACKED ? 4096 : 64;
    u32x4 raw[NWB][WLD];
    auto issue_w = [&](int t, auto buf) {
        constexpr int B = decltype(buf)::value;
        const int tt = min(t * KS + group, KT - 1);
        if constexpr (I8) {
            // The last packed step twice when they are odd (against zero activation codes).
            const kern::gbytes b0p = Wg + (uint32_t)min(2 * tt, p.kt_w - 1) * w_step;
            const kern::gbytes b1p = Wg + (uint32_t)min(2 * tt + 1, p.kt_w - 1) * w_step;
#pragma unroll
            for (int j = 0; j < 2; ++j) raw[B][j] = kern::gld<u32x4>(b0p, w_off[j]);
#pragma unroll
            for (int j = 0; j < 2; ++j) raw[B][2 + j] = kern::gld<u32x4>(b1p, w_off[j]);
        } else {
            const kern::gbytes base = Wg + (uint32_t)tt * w_step;
#pragma unroll
            for (int j = 0; j < 2; ++j) raw[B][j] = kern::gld<u32x4>(base, w_off[j]);
        }
    };

    // Fragment read offsets: sub-step s, row 32·bm + (lane & 31); the 16-byte chunk of lane half h.
    const int h = lane >> 5;
    int xo[2][4];
#pragma unroll
    for (int par = 0; par < 2; ++par)
#pragma unroll
        for (int s = 0; s < 4; ++s)
            xo[par][s] = swz(32 * par + (lane & 31), I8 ? 4 * (s >> 1) + 2 * h + (s & 1) : 4 * h + s) - 32 * 128 * par;

    acc_t acc[FM];
#pragma unroll
    for (int bm = 0; bm < FM; ++bm)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[bm][r] = 0;

    // The prologue's loads in the order the waits count on (the compiler would move the codes' loads past the others).
    auto ordered = [&](auto &&f) {
        f();
        __builtin_amdgcn_sched_barrier(0);
    };
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (F32) {
        // A(0), A(1) (parts 0 and 1 of the first weight step) and W(0), W(1): A(0) and W(0) landed.
        using S0 = std::integral_constant<int, 0>;
        using S1 = std::integral_constant<int, 1>;
        ordered([&] { issue_w(0, S0{}); });
        ordered([&] { issue_a(0, S0{}); });
        ordered([&] { issue_w(1, S1{}); });
        ordered([&] { issue_a(1, S1{}); });
        wait_vmcnt<WLD + A_PER_WAVE>();
    } else {
        // The steps' issue order: A(0 .. NAS−2) and W(0 .. NAS−1); A(0) and W(0) landed.
        static_for<0, NAS>([&](auto vc) {
            constexpr int v = decltype(vc)::value;
            if constexpr (v > 0) ordered([&] { issue_a(v - 1, std::integral_constant<int, v - 1>{}); });
            ordered([&] { issue_w(v, vc); });
        });
        wait_vmcnt<STEP_WAIT>();
    }
    step_barrier();

    using I0 = std::integral_constant<int, 0>;
    u32x4 wf[F32 ? 4 : 1];  // fp32 route: the weight step's widened codes, kept for its three parts
    // Step t on stage U; its codes in buffer B (fp32 route: part U of the weight step in buffer B).
    // TAIL: one of the last steps, whose code loads no later step uses and the compiler drops: the wait counts the
    // activation's loads only (as if every code load had been dropped).
    auto step = [&](int t, auto uc, auto bc, auto tail) {
        constexpr bool TAIL = decltype(tail)::value;
        constexpr int U = decltype(uc)::value, B = decltype(bc)::value;
        u32x4 wk[2];                            // the sub-step's codes (widened, or as they are)
        u32x4 xf[2][FM];
        auto codes = [&](auto sc) {
            constexpr int s = decltype(sc)::value;
            if constexpr (I8) {
                wk[s & 1] = raw[B][s];
            } else if constexpr (F32 && U > 0) {
                wk[s & 1] = wf[s];
            } else {
                const u32x4 &r = raw[B][s >> 1];
                wk[s & 1] = __builtin_bit_cast(u32x4, wd::widen8<WT>(r[2 * (s & 1)], r[2 * (s & 1) + 1]));
                if constexpr (F32) wf[s] = wk[s & 1];
            }
        };
        auto read_x = [&](auto sc) {
            constexpr int s = decltype(sc)::value;
            static_for<0, FM>([&](auto bmc) {
                constexpr int bm = decltype(bmc)::value;
                xf[s & 1][bm] = __builtin_bit_cast(u32x4, kern::lds_load_frag(ldg + U * SA + 32 * 128 * bm, xo[bm & 1][s]));
            });
        };
        __builtin_amdgcn_sched_barrier(0);
        read_x(I0{});
        codes(I0{});
        // Into the stage read in step t − 1 (the barrier that ended it saw every wave's reads).
        issue_a(t + NAS - 1, std::integral_constant<int, (U + NAS - 1) % NAS>{});
        static_for<0, 4>([&](auto sc) {
            constexpr int s = decltype(sc)::value;
            if constexpr (s < 3) {
                read_x(std::integral_constant<int, s + 1>{});
                codes(std::integral_constant<int, s + 1>{});
            }
            // The buffer's last codes are read (bf16: widened) by sub-step 2; the A loads stay ahead of
            // these in issue order (the vmcnt counts rely on it).
            if constexpr (!I8 && s == 2 && (!F32 || U == 0)) {
                __builtin_amdgcn_sched_barrier(0);
                issue_w(F32 ? t / 3 + NWB : t + NAS, bc);
                __builtin_amdgcn_sched_barrier(0);
            }
            static_for<0, FM>([&](auto bmc) {
                constexpr int bm = decltype(bmc)::value;
                if constexpr (I8)
                    acc[bm] = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(wd::i32x4, wk[s & 1]),
                                                                    __builtin_bit_cast(wd::i32x4, xf[s & 1][bm]), acc[bm],
                                                                    0, 0, 0);
                else
                    acc[bm] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, wk[s & 1]),
                                                                      __builtin_bit_cast(bf16x8, xf[s & 1][bm]), acc[bm],
                                                                      0, 0, 0);
            });
            if constexpr (!I8 && s < 3) {
                static_for<0, FM>([&](auto) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, 12 / FM, 0);
                });
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (I8) {
            issue_w(t + NAS, bc);
            __builtin_amdgcn_sched_barrier(0);
        }
        // Fp32 route: A(t + 1) landed; A(t + 2) may fly, and the codes issued in part 0 beside it.
        if constexpr (F32) wait_vmcnt<A_PER_WAVE + (U < 2 && !TAIL ? WLD : 0)>();
        else wait_vmcnt<TAIL ? (NAS - 2) * A_PER_WAVE : STEP_WAIT>();
        // A group of one wave shares no LDS within the K loop (it reads only the stages it loads itself).
        if constexpr (NW > 1) step_barrier();
        else asm volatile("" ::: "memory");
    };
    // Every group runs the same number of step rounds (the barriers are the workgroup's); a step past K — the
    // last round of the later groups when the steps do not divide — is left out, its loads repeat the last step's.
    const int mine = group < KT ? (KT - group + KS - 1) / KS : 0;
    const int rounds = (KT + KS - 1) / KS;
    int t = 0;
    if constexpr (F32) {
        auto three = [&](int i, auto bc, auto tail) {
            static_for<0, 3>([&](auto uc) { step(3 * i + decltype(uc)::value, uc, bc, tail); });
        };
        for (; t + 2 <= mine; t += 2)
            static_for<0, 2>([&](auto bc) { three(t + decltype(bc)::value, bc, std::false_type{}); });
        if (t < mine) three(t, I0{}, std::true_type{});
    } else {
        for (; t + NAS <= mine; t += NAS) static_for<0, NAS>([&](auto uc) { step(t + decltype(uc)::value, uc, uc, std::false_type{}); });
        static_for<0, NAS>([&](auto uc) {
            constexpr int u = decltype(uc)::value;
            if (t + u < mine) step(t + u, uc, uc, std::true_type{});
        });
    }
    if constexpr (NW > 1) {
        if (mine < rounds) static_for<0, F32 ? 3 : 1>([&](auto) { step_barrier(); });
    }
    wait_vmcnt<0>();
    __syncthreads();

    // ---- the groups' sums added, the epilogue, the stores --------------------------------------------
    // A thread's items of a row block: four columns (chunk) of one row of one output block; its block and
    // chunk, and so its columns' scales and biases, are the same for every row block.
    const int n_out = glu ? p.glu_half : p.N;
    constexpr int IT = (4 + KS - 1) / KS;                    // items a thread at most
    const int items = (glu ? NW / 2 : NW) * 256;             // 32 rows × 8 chunks a block of output columns
    const int chunk = tid & 7;
    float sc[IT][4], bi[IT][4], su[IT][4], bu[IT][4];
    int col[IT];
    Out4 to[IT];
#pragma unroll
    for (int i = 0; i < IT; ++i) {
        const int it = tid + i * THREADS, blk = it >> 8;
        if (it < items) {
            col[i] = (glu ? tn * NW / 2 + blk : tn * NW + blk) * 32 + 4 * chunk;
            to[i] = out4(p, min(col[i], n_out - 1), n_out);
            column4(p.scale, p.scale_per_col, p.sb_vec, col[i], n_out, 0, sc[i]);
            column4(p.bias, true, p.sb_vec, col[i], n_out, 0, bi[i]);
            if (glu) {
                column4(p.scale, p.scale_per_col, p.sb_vec, col[i], n_out, p.glu_half, su[i]);
                column4(p.bias, true, p.sb_vec, col[i], n_out, p.glu_half, bu[i]);
            }
        } else {
            col[i] = n_out;
        }
    }
    const bool has_bias = p.bias != nullptr;
    const int64_t row_stride = row_bytes(p);
    static_for<0, FM>([&](auto bmc) {
        constexpr int bm = decltype(bmc)::value;
        uint8_t *dst = lds + wave_all * SLOT + (lane & 31) * PITCH + 16 * h;
        static_for<0, 4>([&](auto gc) {
            constexpr int g = decltype(gc)::value;  // columns 8g + 4h + [0, 4) of row lane & 31
            *reinterpret_cast<v4 *>(dst + 32 * g) = v4{acc[bm][4 * g], acc[bm][4 * g + 1], acc[bm][4 * g + 2], acc[bm][4 * g + 3]};
        });
        __syncthreads();
#pragma unroll
        for (int i = 0; i < IT; ++i) {
            const int it = tid + i * THREADS, blk = it >> 8, row = (it >> 3) & 31;
            const int m = m0 + 32 * bm + row;
            if (col[i] < n_out && m < p.M) {
                const uint8_t *src = lds + (glu ? 2 * blk : blk) * SLOT + row * PITCH + 16 * chunk;
                float v[4], u[4];
                auto total = [&](const uint8_t *s, float (&o)[4]) {
                    v4 x = *reinterpret_cast<const v4 *>(s);
#pragma unroll
                    for (int g = 1; g < KS; ++g) {
                        const v4 y = *reinterpret_cast<const v4 *>(s + g * NW * SLOT);
#pragma unroll
                        for (int e = 0; e < 4; ++e) x[e] += y[e];
                    }
#pragma unroll
                    for (int e = 0; e < 4; ++e) o[e] = (float)x[e];
                };
                const float sx = I8 ? p.sx[m] : 1.0f;
                total(src, v);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    v[e] = __fmul_rn(v[e], I8 ? __fmul_rn(sx, sc[i][e]) : sc[i][e]);
                    if (has_bias) v[e] = __fadd_rn(v[e], bi[i][e]);
                }
                if (glu) {
                    total(src + SLOT, u);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        u[e] = __fmul_rn(u[e], I8 ? __fmul_rn(sx, su[i][e]) : su[i][e]);
                        if (has_bias) u[e] = __fadd_rn(u[e], bu[i][e]);
                    }
                }
                activate4(p.epi, v, u);
                store4(p, to[i], m * row_stride, col[i], n_out, v);
            }
        }
        if constexpr (bm + 1 < FM) __syncthreads();
    });
}

template <int MATH, int WT, int WL, int BM, int NW, int KS, int NAS>
hipError_t launch_group(const GemmArgs &args, int epi, int out, hipStream_t stream) {
    GemmArgs p = args;
    if (p.glu_half > 0 && NW % 2 != 0) return hipErrorInvalidValue;
    p.epi = epi;
    p.out = out;
    p.tiles_m = (p.M + BM - 1) / BM;
    const int blocks_n = p.glu_half > 0 ? 2 * ((p.glu_half + 31) / 32) : (p.N + 31) / 32;  // 32-column blocks
    p.tiles_n = (blocks_n + NW - 1) / NW;
    const int blocks = p.tiles_m * p.tiles_n;
    if (blocks == 0) return hipSuccess;
    hipLaunchKernelGGL((gemm_group_kernel<MATH, WT, WL, BM, NW, KS, NAS>), dim3(blocks), dim3(64 * NW * KS), 0, stream, p);
    return hipGetLastError();
}

}  // namespace grp
}  // namespace sq8
