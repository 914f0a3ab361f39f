// Instantiation unit of the runtime-radix line kernel: FP32.
#include "fft_mixed_launch.hpp"

namespace dfft {

int mixed_lanes_f32(int n) { return mix_length<float, 16>(n).lanes; }

hipError_t launch_mixed_f32(const LinePass& p, hipStream_t s) { return launch_mixed<float, 16>(p, s); }

}  // namespace dfft
