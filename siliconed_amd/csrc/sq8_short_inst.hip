// sq8_short_inst.hip — instantiates the short-M kernels (the 16-column groups of sq8_gemv_kernel.h and the skinny kernel)
// for one weight type (SQ8_WT) and layout (SQ8_WL: 1 [N, K], 2 packed).
#include "sq8_gemv_kernel.h"
#include "sq8_skinny_kernel.h"

#if !defined(SQ8_WT) || !defined(SQ8_WL)
#error "compile with -DSQ8_WT=<0 int8 | 1 fp8> -DSQ8_WL=<1 [N,K] | 2 packed>"
#endif

#define SQ8_CAT2(a, b) a##b
#define SQ8_CAT(a, b) SQ8_CAT2(a, b)

namespace sq8 {

hipError_t SQ8_CAT(launch_short_, SQ8_CAT(SQ8_WT, SQ8_CAT(_, SQ8_WL)))(const GemmArgs &p, int tile, int epi, int out,
                                                                     hipStream_t stream) {
    if (tile == WD_GEMV) {
        // Up to 16 rows (one group of 16 × 16 MFMAs); more rows take the skinny kernel.
        if (p.M <= 16) return wd::dispatch_gemv<SQ8_WT, SQ8_WL>(p, epi, out, stream);
        tile = p.M <= 128 ? WD_SKINNY32 : WD_SKINNY64;
    }
    if (tile == WD_SKINNY64) return wd::dispatch_skinny<64, 4, 2, SQ8_WT, SQ8_WL>(p, epi, out, stream);
    if (tile == WD_SKINNY32) return wd::dispatch_skinny<32, 4, 2, SQ8_WT, SQ8_WL>(p, epi, out, stream);
    return hipErrorInvalidValue;
}

}  // namespace sq8
