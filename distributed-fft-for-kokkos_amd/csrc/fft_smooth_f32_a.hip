// Instantiation unit of the compiled 2^a 3^b 5^c lengths: F32, 3 to 100 (the
// units are compiled in parallel).
#include "fft_smooth.hpp"
#include "fft_smooth_impl.hpp"

namespace dfft {

hipError_t smooth_f32_a(const LinePass& p, hipStream_t s) {
  return dispatch_smooth<float,
      3, 5, 6, 9, 10, 12, 15, 18, 20, 24, 25, 27, 30, 36, 40, 45, 48, 50, 54, 60, 72, 75, 80, 81,
      90, 96, 100>(p, s);
}

hipError_t launch_smooth_f32(const LinePass& p, hipStream_t s) {
  if (p.n % 7 == 0) return smooth_f32_e(p, s);
  return p.n <= 100 ? smooth_f32_a(p, s) : p.n <= 250 ? smooth_f32_b(p, s) : p.n <= 500 ? smooth_f32_c(p, s) : smooth_f32_d(p, s);
}

}  // namespace dfft
