// Host interface of the runtime-radix line kernel (fft_mixed_impl.hpp).
#pragma once

#include "fft_kernels.hpp"

namespace dfft {

// true if every prime factor of n is at most 13 and a block holds a line of it
bool mixed_length(int n, bool fp64);
// true if pass p suits the kernels that hold whole lines (this one and
// fft_smooth): the line axis undistributed on both sides, no adjoint of a real pass
bool whole_line_pass(const LinePass& p);
int mixed_lanes_f64(int n);  // lanes per line, 0: not a length of the kernel
int mixed_lanes_f32(int n);
hipError_t launch_mixed_f64(const LinePass& p, hipStream_t s);
hipError_t launch_mixed_f32(const LinePass& p, hipStream_t s);

}  // namespace dfft
