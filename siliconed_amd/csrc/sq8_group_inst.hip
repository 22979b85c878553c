// sq8_group_inst.hip — the K-group kernels' instantiations (sq8_group_kernel.h) for one kind of product (SQ8_MATH:
// 0 bf16 × widened codes, 1 int8 × int8, 2 the fp32 route), weight type (SQ8_WT) and layout (SQ8_WL: 1 [N, K], 2 packed).
#include "sq8_group_kernel.h"

#if !defined(SQ8_MATH) || !defined(SQ8_WT) || !defined(SQ8_WL)
#error "compile with -DSQ8_MATH=<0|1|2> -DSQ8_WT=<0 int8 | 1 fp8> -DSQ8_WL=<1 [N,K] | 2 packed>"
#endif

#define SQ8_CAT2(a, b) a##b
#define SQ8_CAT(a, b) SQ8_CAT2(a, b)

namespace sq8 {

hipError_t SQ8_CAT(launch_group_, SQ8_CAT(SQ8_MATH, SQ8_CAT(_, SQ8_CAT(SQ8_WT, SQ8_CAT(_, SQ8_WL)))))(
    const GemmArgs &p, int shape, int epi, int out, hipStream_t stream) {
    constexpr int MATH = SQ8_MATH, WT = SQ8_WT, WL = SQ8_WL;
    // The shapes of group_shapes, each with its activation stages by kind of product (bf16, int8, fp32 route; 0: not
    // built for it), as many as fit the LDS beside the groups'.
#define SQ8_SHAPE(I, BM, NW, KS, BF16, I8, F32)                                                                       \
    case I: {                                                                                                         \
        constexpr int NAS = MATH == GM_I8 ? I8 : MATH == GM_F32 ? F32 : BF16;                                         \
        static_assert(group_shapes[I].rows == BM && group_shapes[I].cols == 32 * NW && group_shapes[I].groups == KS); \
        static_assert((NAS > 0) == (group_shapes[I].cost[MATH].us_step > 0.0f), "priced where it is built");          \
        if constexpr (NAS > 0) return grp::launch_group<MATH, WT, WL, BM, NW, KS, NAS>(p, epi, out, stream);          \
        break;                                                                                                        \
    }
    static_assert(kGroupShapes == 15, "a case for each");
    switch (shape) {
        SQ8_SHAPE(0, 32, 1, 8, 0, 4, 0)
        SQ8_SHAPE(1, 32, 2, 8, 0, 2, 0)
        SQ8_SHAPE(2, 32, 1, 4, 4, 0, 3)
        SQ8_SHAPE(3, 32, 2, 4, 4, 0, 3)
        SQ8_SHAPE(4, 64, 2, 4, 4, 4, 3)
        SQ8_SHAPE(5, 64, 3, 4, 3, 3, 3)
        SQ8_SHAPE(6, 64, 4, 4, 2, 2, 3)
        SQ8_SHAPE(7, 64, 4, 2, 3, 0, 3)
        SQ8_SHAPE(8, 64, 6, 2, 3, 0, 3)
        SQ8_SHAPE(9, 96, 3, 4, 3, 3, 3)
        SQ8_SHAPE(10, 96, 4, 4, 2, 2, 0)
        SQ8_SHAPE(11, 128, 3, 4, 2, 2, 0)
        SQ8_SHAPE(12, 128, 4, 2, 3, 3, 3)
        SQ8_SHAPE(13, 96, 6, 2, 3, 3, 3)
        SQ8_SHAPE(14, 128, 6, 2, 3, 3, 3)
    default: break;
    }
#undef SQ8_SHAPE
    return hipErrorInvalidValue;
}

}  // namespace sq8
