// Kernel instantiations of the wave-split mmt4d for one operand type (see
// mmt4d_wave_k_kernels.h).
#include "mmt4d_wave_k_kernels.h"

namespace uk {

hipError_t launch_wave_k_f16(const MfmaArgs& m, int gather, int shape, bool streamed, hipStream_t stream) {
  switch (gather) {
    case 16: return launch_wave_k_piece<kF16, false, false, 16>(m, shape, streamed, stream);
    case 8: return launch_wave_k_piece<kF16, false, false, 8>(m, shape, streamed, stream);
    case 4: return launch_wave_k_piece<kF16, false, false, 4>(m, shape, streamed, stream);
    default: return launch_wave_k_piece<kF16, false, false, 2>(m, shape, streamed, stream);
  }
}

}  // namespace uk
