// Host interface of the compiled kernels of lengths 2^a 3^b 5^c up to 1024, and
// with factors 7 up to 256 (fft_smooth_impl.hpp).
#pragma once

#include "fft_kernels.hpp"

namespace dfft {

// true if whole lines (whole_line_pass) of length n have a compiled kernel here
bool smooth_length(int n);
hipError_t launch_smooth_f64(const LinePass& p, hipStream_t s);
hipError_t launch_smooth_f32(const LinePass& p, hipStream_t s);
// kept-mode passes (launch_band_pass), FP64: even 2^a 3^b 5^c from 36 to 384
bool smooth_band_length(int n);
hipError_t launch_smooth_band(const LinePass& p, hipStream_t s);

// one per instantiation unit; hipErrorNotSupported for other lengths
hipError_t smooth_f64_a(const LinePass& p, hipStream_t s);
hipError_t smooth_f64_b(const LinePass& p, hipStream_t s);
hipError_t smooth_f64_c(const LinePass& p, hipStream_t s);
hipError_t smooth_f64_d(const LinePass& p, hipStream_t s);
hipError_t smooth_f64_e(const LinePass& p, hipStream_t s);
hipError_t smooth_f32_a(const LinePass& p, hipStream_t s);
hipError_t smooth_f32_b(const LinePass& p, hipStream_t s);
hipError_t smooth_f32_c(const LinePass& p, hipStream_t s);
hipError_t smooth_f32_d(const LinePass& p, hipStream_t s);
hipError_t smooth_f32_e(const LinePass& p, hipStream_t s);
hipError_t smooth_band_a(const LinePass& p, hipStream_t s);
hipError_t smooth_band_b(const LinePass& p, hipStream_t s);
hipError_t smooth_band_c(const LinePass& p, hipStream_t s);

}  // namespace dfft
