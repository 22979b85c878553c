// sq8_gemm_inst.hip — instantiates the branch-free (FAST) GEMM kernels on [K, N] codes for one weight type, chosen at
// compile time: the build compiles this file once per SQ8_WT so the sets compile in parallel. ([N, K] codes that these
// could read go to the weight-direct kernels.)
#include "sq8_gemm_kernel.h"

#if !defined(SQ8_WT)
#error "compile with -DSQ8_WT=<0 int8 | 1 fp8>"
#endif

#define SQ8_CAT2(a, b) a##b
#define SQ8_CAT(a, b) SQ8_CAT2(a, b)

namespace sq8 {

hipError_t SQ8_CAT(launch_fast_, SQ8_WT)(const GemmArgs &p, int tile, int epi, int out, hipStream_t stream) {
    switch (tile) {
    case TILE_256x256: return kern::dispatch_epi_out<256, 256, SQ8_WT, W_KN, true>(p, epi, out, stream);
    case TILE_128x128: return kern::dispatch_epi_out<128, 128, SQ8_WT, W_KN, true>(p, epi, out, stream);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace sq8
