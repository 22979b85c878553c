// sq8_group_inst.hip — the K-group kernels' instantiations (sq8_group_kernel.h) for one kind of product (SQ8_MATH:
// 0 bf16 × widened codes, 1 int8 × int8), weight type (SQ8_WT) and layout (SQ8_WL: 1 [N, K], 2 packed).
#include "sq8_group_kernel.h"

#if !defined(SQ8_MATH) || !defined(SQ8_WT) || !defined(SQ8_WL)
#error "compile with -DSQ8_MATH=<0|1> -DSQ8_WT=<0 int8 | 1 fp8> -DSQ8_WL=<1 [N,K] | 2 packed>"
#endif

#define SQ8_CAT2(a, b) a##b
#define SQ8_CAT(a, b) SQ8_CAT2(a, b)

namespace sq8 {

hipError_t SQ8_CAT(launch_group_, SQ8_CAT(SQ8_MATH, SQ8_CAT(_, SQ8_CAT(SQ8_WT, SQ8_CAT(_, SQ8_WL)))))(
    const GemmArgs &p, int shape, int epi, int out, hipStream_t stream) {
    constexpr int MATH = SQ8_MATH, WT = SQ8_WT, WL = SQ8_WL;
    switch (shape) {
    //                                         rows, waves, groups, stages
    case 0: return grp::launch_group<MATH, WT, WL, 32, 1, 8, 4>(p, epi, out, stream);
    case 1: return grp::launch_group<MATH, WT, WL, 32, 2, 8, 2>(p, epi, out, stream);
    case 2: return grp::launch_group<MATH, WT, WL, 64, 2, 4, 4>(p, epi, out, stream);
    case 3: return grp::launch_group<MATH, WT, WL, 64, 3, 4, 3>(p, epi, out, stream);
    case 4: return grp::launch_group<MATH, WT, WL, 64, 4, 4, 2>(p, epi, out, stream);
    case 5: return grp::launch_group<MATH, WT, WL, 96, 3, 4, 3>(p, epi, out, stream);
    case 6: return grp::launch_group<MATH, WT, WL, 96, 4, 4, 2>(p, epi, out, stream);
    case 7: return grp::launch_group<MATH, WT, WL, 128, 3, 4, 2>(p, epi, out, stream);
    case 8: return grp::launch_group<MATH, WT, WL, 128, 4, 2, 3>(p, epi, out, stream);
    case 9: return grp::launch_group<MATH, WT, WL, 96, 6, 2, 3>(p, epi, out, stream);
    case 10: return grp::launch_group<MATH, WT, WL, 128, 6, 2, 3>(p, epi, out, stream);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace sq8
