// sq8_blocks16_inst.hip — the narrow-wave block-scaled kernel's instantiations (sq8_blocks16_kernel.h), by rows.
#include "sq8_blocks16_kernel.h"

namespace sq8 {

hipError_t launch_blocks16(const GemmArgs &p, int rows, int epi, int out, hipStream_t stream) {
    switch (rows) {
    case 16: return blk::launch_blocks16<1, 8, 8>(p, epi, out, stream);
    case 32: return blk::launch_blocks16<2, 8, 8>(p, epi, out, stream);
    case 48: return blk::launch_blocks16<3, 4, 8>(p, epi, out, stream);
    case 64: return blk::launch_blocks16<4, 4, 8>(p, epi, out, stream);
    case 80: return blk::launch_blocks16<5, 4, 8>(p, epi, out, stream);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace sq8
