// Instantiation unit of the kept-mode passes of the lengths 2^a 3^b 5^c: even
// lengths 36 to 120, FP64 (the units are compiled in parallel).
#include "fft_smooth.hpp"
#include "fft_smooth_impl.hpp"

namespace dfft {

hipError_t smooth_band_a(const LinePass& p, hipStream_t s) {
  return dispatch_smooth_band<
      36, 40, 48, 50, 54, 60, 72, 80, 90, 96, 100, 108, 120>(p, s);
}

bool smooth_band_length(int n) { return n % 2 == 0 && n % 7 != 0 && n >= 36 && n <= 384 && smooth_length(n); }

hipError_t launch_smooth_band(const LinePass& p, hipStream_t s) {
  return p.n <= 120 ? smooth_band_a(p, s) : p.n <= 240 ? smooth_band_b(p, s) : smooth_band_c(p, s);
}

}  // namespace dfft
