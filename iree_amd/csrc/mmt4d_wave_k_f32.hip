// Kernel instantiations of the wave-split mmt4d for one operand type (see
// mmt4d_wave_k_kernels.h).
#include "mmt4d_wave_k_kernels.h"

namespace uk {
namespace {

// Tile number `shape` of kWaveKShapesF32, from number SHAPE on.
template <int G, int SHAPE = 0>
hipError_t launch_shape(const MfmaArgs& m, int shape, bool streamed, hipStream_t stream) {
  if constexpr (SHAPE < (int)(sizeof kWaveKShapesF32 / sizeof kWaveKShapesF32[0])) {
    constexpr WaveKShape s = kWaveKShapesF32[SHAPE];
    if (shape != SHAPE) return launch_shape<G, SHAPE + 1>(m, shape, streamed, stream);
    if constexpr (SHAPE == 0) {
      if (two_steps_ahead<kF32, G>(m)) return launch_wave_k_tile<kF32, false, false, G, 1, 1, 8, 3>(m, streamed, stream);
    }
    return launch_wave_k_tile<kF32, false, false, G, s.fa, s.fb, 8, 2>(m, streamed, stream);
  } else {
    return hipErrorInvalidValue;
  }
}

}  // namespace

hipError_t launch_wave_k_f32(const MfmaArgs& m, int gather, int shape, bool streamed, hipStream_t stream) {
  switch (gather) {
    case 16: return launch_shape<16>(m, shape, streamed, stream);
    case 8: return launch_shape<8>(m, shape, streamed, stream);
    default: return launch_shape<4>(m, shape, streamed, stream);
  }
}

}  // namespace uk
