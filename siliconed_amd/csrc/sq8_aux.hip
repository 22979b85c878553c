// sq8_aux.hip — the device dequantiser and the bf16 rounding pass.
//
// dequantize: out[i] = Float(code[i]) · s, one fp32 multiply, never fused
// (Sources/Siliconed/Widen.swift:81-97, :129-271). The code goes through the same widening the
// GEMM uses (sq8_device.h), so the bit-exact test of this kernel is the test of that conversion.
// round_bf16: fp32 → bf16 nearest-even, a NaN kept quiet (TensorGEMMBF16.swift:41-48, 67-73).
#include <hip/hip_fp16.h>

#include "sq8_gemm.h"

namespace sq8 {

namespace {

// Scale kinds, numbered as the C ABI's sq8_dtype.
constexpr int S_BF16 = 1, S_F16 = 5;  // 2, fp32, otherwise
constexpr int L_TENSOR = 0, L_COLUMNS = 1, L_BLOCKS = 2;  // 3, rows, otherwise

__device__ __forceinline__ float scale_at(const void *s, int kind, int64_t i) {
    if (kind == S_BF16) return __uint_as_float((uint32_t)reinterpret_cast<const uint16_t *>(s)[i] << 16);
    if (kind == S_F16) return __half2float(reinterpret_cast<const __half *>(s)[i]);
    return reinterpret_cast<const float *>(s)[i];
}

template <int WT>
__global__ void __launch_bounds__(256) dequantize_kernel(const uint8_t *__restrict__ codes, int64_t rows,
                                                         int64_t columns, const void *__restrict__ scale,
                                                         int scale_kind, int layout, int64_t block_rows,
                                                         int64_t first_row, float *__restrict__ out) {
    const int64_t count = rows * columns;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (int64_t)gridDim.x * blockDim.x) {
        const float v = widen1<WT>(codes[i]);
        if (!scale) {
            out[i] = v;
            continue;
        }
        const int64_t r = i / columns, c = i - r * columns;
        float s;
        switch (layout) {
        case L_TENSOR: s = scale_at(scale, scale_kind, 0); break;
        case L_COLUMNS: s = scale_at(scale, scale_kind, c); break;
        case L_BLOCKS: s = scale_at(scale, scale_kind, ((first_row + r) / block_rows) * columns + c); break;
        default: s = scale_at(scale, scale_kind, first_row + r); break;
        }
        out[i] = __fmul_rn(v, s);
    }
}

__global__ void __launch_bounds__(256) round_bf16_kernel(const float *__restrict__ x, uint16_t *__restrict__ y,
                                                         int64_t count) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (int64_t)gridDim.x * blockDim.x)
        y[i] = (uint16_t)round_bf16(x[i]);
}

// The passes that write the products' operands, `rows` rows of k values read `ldx` apart, four values a thread:
//   ROUND  fp32 → bf16, rows kp ≥ k apart with columns [k, kp) zero;
//   COPY   bf16 as they are, padded the same way (a K of no whole 64-wide steps, an operand not aligned for 16-byte loads);
//   SPLIT3 fp32 → three bf16 parts along K: y[r, c] = hi, y[r, kp + c] = mid, y[r, 2kp + c] = lo (columns [k, kp) of each
//          part zero), each part the top 16 bits of what the one before leaves (hi = x truncated to bf16, mid = (x − hi)
//          truncated, lo = x − hi − mid): 24 significant bits in three parts of 8, every difference exact, no part
//          rounded, so hi + mid + lo = x and every product of a part with a code is exact. Every part is a normal bf16 for
//          |x| ≥ 2^−103; an infinity or NaN is its hi part alone.
// Memory-bound: 2^lg threads a row (up to 1024 columns a workgroup, several short rows in one), 16- or 8-byte loads where
// the rows are aligned for them (VEC) and 8-byte stores where kp and y are (`wide`). One value a thread and a 64-bit
// division each took 12.6 µs for SPLIT3 of 1531 × 3072 values (47 MB); this takes 10.9.
enum RowPass { ROUND = 0, COPY = 1, SPLIT3 = 2 };

template <int PASS, bool VEC>
__global__ void __launch_bounds__(256) row_pass_kernel(const void *__restrict__ x, int64_t ldx, uint16_t *__restrict__ y,
                                                       int64_t rows, int lg, int per_row, int k, int kp, int wide) {
    const uint32_t part = blockIdx.x / (uint32_t)per_row;
    const int64_t row = ((int64_t)part << (8 - lg)) + (threadIdx.x >> lg);
    const int c = ((int)(blockIdx.x - part * (uint32_t)per_row) * 256 + (int)(threadIdx.x & ((1u << lg) - 1))) * 4;
    if (c >= kp || row >= rows) return;
    const int64_t at = row * ldx + c;
    uint32_t hi[4] = {0, 0, 0, 0}, mid[4] = {0, 0, 0, 0}, lo[4] = {0, 0, 0, 0};
    if constexpr (PASS == COPY) {
        const uint16_t *src = static_cast<const uint16_t *>(x) + at;
        if (VEC && wide && c + 4 <= k) {
            *reinterpret_cast<u32x2 *>(y + row * kp + c) = *reinterpret_cast<const u32x2 *>(src);
            return;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (c + e < k) hi[e] = src[e];
    } else {
        const float *src = static_cast<const float *>(x) + at;
        float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if (VEC && c + 4 <= k) {
            const f32x4 t = *reinterpret_cast<const f32x4 *>(src);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = t[e];
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (c + e < k) v[e] = src[e];
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if constexpr (PASS == ROUND) {
                hi[e] = round_bf16(v[e]);
            } else {
                const uint32_t u = __float_as_uint(v[e]);
                hi[e] = u >> 16;
                if ((u & 0x7f800000u) != 0x7f800000u) {
                    const float r1 = v[e] - __uint_as_float(u & 0xffff0000u);  // the low 16 bits of x: exact
                    mid[e] = __float_as_uint(r1) >> 16;
                    lo[e] = __float_as_uint(r1 - __uint_as_float(mid[e] << 16)) >> 16;  // ≤ 8 bits left: a bf16 value
                }
            }
        }
    }
    auto put = [&](uint16_t *dst, const uint32_t (&d)[4]) {
        if (wide) {
            *reinterpret_cast<u32x2 *>(dst) = u32x2{d[0] | d[1] << 16, d[2] | d[3] << 16};
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (c + e < kp) dst[e] = (uint16_t)d[e];
        }
    };
    if constexpr (PASS == SPLIT3) {
        uint16_t *dst = y + row * 3 * kp + c;
        put(dst, hi);
        put(dst + kp, mid);
        put(dst + 2 * (int64_t)kp, lo);
    } else {
        put(y + row * kp + c, hi);
    }
}

// Columns [k, kp) of `rows` bf16 rows `ld` apart set to zero (the padding after a pass that wrote
// only the first k).
__global__ void __launch_bounds__(256) zero_tail_kernel(uint16_t *__restrict__ y, int64_t ld, int64_t rows, int k,
                                                        int kp) {
    const int w = kp - k;
    const int64_t count = rows * w;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t r = i / w;
        y[r * ld + k + (i - r * w)] = 0;
    }
}

int grid_for(int64_t count) {
    const int64_t blocks = (count + 255) / 256;
    return (int)(blocks < 8192 ? (blocks > 0 ? blocks : 1) : 8192);
}

// One row pass: `size` the input's bytes a value.
template <int PASS>
hipError_t row_pass(const void *x, int64_t ldx, int size, uint16_t *y, int64_t rows, int k, int kp, hipStream_t stream) {
    if (rows == 0 || kp == 0) return hipSuccess;
    int lg = 0;
    while (lg < 8 && (4 << lg) < kp) ++lg;
    const int64_t per_row = (kp + 1023) / 1024, blocks = ((rows + (256 >> lg) - 1) >> (8 - lg)) * per_row;
    if (blocks > INT32_MAX) return hipErrorInvalidValue;
    const int wide = kp % 4 == 0 && (reinterpret_cast<uintptr_t>(y) % 8) == 0;
    const bool vec = ldx % 4 == 0 && (reinterpret_cast<uintptr_t>(x) % (4 * size)) == 0;
    if (vec)
        hipLaunchKernelGGL((row_pass_kernel<PASS, true>), dim3((unsigned)blocks), dim3(256), 0, stream, x, ldx, y, rows,
                           lg, (int)per_row, k, kp, wide);
    else
        hipLaunchKernelGGL((row_pass_kernel<PASS, false>), dim3((unsigned)blocks), dim3(256), 0, stream, x, ldx, y, rows,
                           lg, (int)per_row, k, kp, wide);
    return hipGetLastError();
}

// [N, K] codes, one thread per 16-byte chunk of the packed layout: chunk c = ((slab·kt + t)·4 + j)·64 + lane holds
// codes k ∈ [64t + 32h + 16(j&1), +16) of virtual column 32·(j>>1) + (lane & 31) of the slab
// (h = lane >> 5); virtual columns are the weight's own, or for GLU the slab's 32 output columns of
// the first half then the same of the second. Zeros past K and past the columns.
__global__ void __launch_bounds__(256) pack_kernel(const uint8_t *__restrict__ w, int64_t ldw, int k, int n, int glu, int kt,
                                                   int64_t chunks, uint8_t *__restrict__ out) {
    for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < chunks; c += (int64_t)gridDim.x * blockDim.x) {
        const int lane = (int)(c & 63), j = (int)((c >> 6) & 3);
        const int64_t st = c >> 8;
        const int t = (int)(st % kt), slab = (int)(st / kt);
        const int b = j >> 1, h = lane >> 5, nl = lane & 31;
        int col;
        bool valid;
        if (glu) {
            const int half = n / 2, oc = slab * 32 + nl;
            valid = oc < half;
            col = oc + b * half;
        } else {
            col = slab * 64 + b * 32 + nl;
            valid = col < n;
        }
        const int k0 = 64 * t + 32 * h + 16 * (j & 1);
        u32x4 v = {0, 0, 0, 0};
        if (valid && k0 + 16 <= k) {
            // The chunk is 16 contiguous codes of row `col` (at any byte address).
            __builtin_memcpy(&v, w + (int64_t)col * ldw + k0, 16);
        } else {
            uint32_t d[4] = {0, 0, 0, 0};
            for (int e = 0; e < 16; ++e)
                if (valid && k0 + e < k) d[e >> 2] |= (uint32_t)w[(int64_t)col * ldw + k0 + e] << (8 * (e & 3));
            v = u32x4{d[0], d[1], d[2], d[3]};
        }
        *reinterpret_cast<u32x4 *>(out + c * 16) = v;
    }
}

// [K, N] codes: one workgroup per (slab, 4 K steps) — 256 rows of K × the slab's 64
// (virtual) columns. Each thread loads 4 consecutive rows × 16 columns (four 16-byte loads),
// transposes the 4 × 16 bytes in registers into 16 words of 4 consecutive K of one column, and
// writes them to an LDS tile [column][K]; the packed chunks (16 consecutive K of one column) are then
// 16-byte LDS reads. WHOLE: k % 256 == 0, whole slabs (n % 64 == 0, GLU: half % 32 == 0), ldw %
// 16 == 0 and a 16-byte aligned base; else any k, n, row stride and base: 16-byte loads at any byte address where a
// row holds the 16 columns, single codes at the edges, zeros past them (4672 × 11563 codes 38.1 µs, 40.6 by a gather of
// single bytes; 3072 × 12288, whole, 17.8).
constexpr int PK_KSTEPS = 4;
constexpr int PK_PITCH = 64 * PK_KSTEPS + 16;  // bytes per LDS column row (16-byte aligned, bank spread)

__device__ __forceinline__ uint32_t byte_of(const u32x4 &v, int e) { return (v[e >> 2] >> (8 * (e & 3))) & 0xFF; }

template <bool WHOLE>
__global__ void __launch_bounds__(256) pack_kn_kernel(const uint8_t *__restrict__ w, int64_t ldw, int k, int n, int glu, int kt,
                                                      uint8_t *__restrict__ out) {
    __shared__ __attribute__((aligned(16))) uint8_t tile[64 * PK_PITCH];
    const int groups = (kt + PK_KSTEPS - 1) / PK_KSTEPS;
    const int slab = blockIdx.x / groups, tq = blockIdx.x - slab * groups;
    const int tid = threadIdx.x;
    const int seg = tid & 3, kq = tid >> 2;  // columns [16·seg, +16) of the slab, rows 4·kq .. 4·kq + 3
    const int vc0 = 16 * seg, b = vc0 >> 5;
    const int oc0 = glu ? slab * 32 + (vc0 & 31) : slab * 64 + vc0;
    const int left = (glu ? n / 2 : n) - oc0;  // columns of this half from oc0 on
    const int col0 = glu ? oc0 + b * (n / 2) : oc0;
    const int row0 = tq * 64 * PK_KSTEPS + 4 * kq;
    u32x4 r[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint8_t *src = w + (int64_t)(row0 + i) * ldw + col0;
        if constexpr (WHOLE) {
            r[i] = *reinterpret_cast<const u32x4 *>(src);
        } else {
            r[i] = u32x4{0, 0, 0, 0};
            if (row0 + i < k) {
                if (left >= 16) {
                    __builtin_memcpy(&r[i], src, 16);
                } else {
#pragma unroll
                    for (int e = 0; e < 16; ++e)
                        if (e < left) r[i][e >> 2] |= (uint32_t)src[e] << (8 * (e & 3));
                }
            }
        }
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const uint32_t word = byte_of(r[0], e) | byte_of(r[1], e) << 8 | byte_of(r[2], e) << 16 | byte_of(r[3], e) << 24;
        *reinterpret_cast<uint32_t *>(tile + (vc0 + e) * PK_PITCH + 4 * kq) = word;
    }
    __syncthreads();
    // 4 K steps × 4 loads × 64 lanes = 1024 chunks, 4 per thread.
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int c = tid + 256 * i;
        const int lane = c & 63, j = (c >> 6) & 3, ts = c >> 8;
        const int vc = 32 * (j >> 1) + (lane & 31);
        const int kr = 64 * ts + 32 * (lane >> 5) + 16 * (j & 1);
        const u32x4 v = *reinterpret_cast<const u32x4 *>(tile + vc * PK_PITCH + kr);
        const int t = tq * PK_KSTEPS + ts;
        if (WHOLE || t < kt) *reinterpret_cast<u32x4 *>(out + (((int64_t)slab * kt + t) * 4 + j) * 1024 + lane * 16) = v;
    }
}

}  // namespace

int64_t packed_bytes(int k, int n, bool glu) {
    const int64_t kt = (k + 63) / 64;
    const int64_t slabs = glu ? ((int64_t)n / 2 + 31) / 32 : ((int64_t)n + 63) / 64;
    return slabs * kt * 4096;
}

hipError_t launch_pack(const uint8_t *w, int wl, int64_t ldw, int k, int n, bool glu, uint8_t *out, hipStream_t stream) {
    const int kt = (k + 63) / 64;
    const int64_t chunks = packed_bytes(k, n, glu) / 16;
    if (chunks == 0) return hipSuccess;
    if (wl == W_KN) {
        const bool whole = k % (64 * PK_KSTEPS) == 0 && (glu ? (n / 2) % 32 == 0 : n % 64 == 0) && ldw % 16 == 0 &&
                           ((uintptr_t)w & 15) == 0;
        const int64_t slabs = packed_bytes(k, n, glu) / ((int64_t)kt * 4096);
        const dim3 grid((unsigned)(slabs * ((kt + PK_KSTEPS - 1) / PK_KSTEPS)));
        if (whole)
            hipLaunchKernelGGL(pack_kn_kernel<true>, grid, dim3(256), 0, stream, w, ldw, k, n, glu ? 1 : 0, kt, out);
        else
            hipLaunchKernelGGL(pack_kn_kernel<false>, grid, dim3(256), 0, stream, w, ldw, k, n, glu ? 1 : 0, kt, out);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(pack_kernel, dim3(grid_for(chunks)), dim3(256), 0, stream, w, ldw, k, n, glu ? 1 : 0, kt, chunks, out);
    return hipGetLastError();
}

hipError_t launch_dequantize(const uint8_t *codes, int wt, int64_t rows, int64_t columns, const void *scale,
                             int scale_dtype, int scale_layout, int64_t block_rows, int64_t first_row, float *out,
                             hipStream_t stream) {
    const int64_t count = rows * columns;
    if (count == 0) return hipSuccess;
    if (wt == W_INT8)
        hipLaunchKernelGGL(dequantize_kernel<W_INT8>, dim3(grid_for(count)), dim3(256), 0, stream, codes, rows, columns,
                           scale, scale_dtype, scale_layout, block_rows, first_row, out);
    else
        hipLaunchKernelGGL(dequantize_kernel<W_FP8>, dim3(grid_for(count)), dim3(256), 0, stream, codes, rows, columns,
                           scale, scale_dtype, scale_layout, block_rows, first_row, out);
    return hipGetLastError();
}

hipError_t launch_split3(const float *x, int64_t ldx, uint16_t *y, int64_t rows, int k, int kp, hipStream_t stream) {
    return row_pass<SPLIT3>(x, ldx, 4, y, rows, k, kp, stream);
}

hipError_t launch_round_bf16(const float *x, uint16_t *y, int64_t count, hipStream_t stream) {
    if (count == 0) return hipSuccess;
    hipLaunchKernelGGL(round_bf16_kernel, dim3(grid_for(count)), dim3(256), 0, stream, x, y, count);
    return hipGetLastError();
}

hipError_t launch_round_bf16_rows(const float *x, int64_t ldx, uint16_t *y, int64_t rows, int k, int kp,
                                  hipStream_t stream) {
    return row_pass<ROUND>(x, ldx, 4, y, rows, k, kp, stream);
}

hipError_t launch_pad_bf16_rows(const uint16_t *x, int64_t ldx, uint16_t *y, int64_t rows, int k, int kp,
                                hipStream_t stream) {
    return row_pass<COPY>(x, ldx, 2, y, rows, k, kp, stream);
}

hipError_t launch_zero_tail(uint16_t *y, int64_t ld, int64_t rows, int k, int kp, hipStream_t stream) {
    if (rows == 0 || kp <= k) return hipSuccess;
    hipLaunchKernelGGL(zero_tail_kernel, dim3(grid_for(rows * (kp - k))), dim3(256), 0, stream, y, ld, rows, k, kp);
    return hipGetLastError();
}

}  // namespace sq8
