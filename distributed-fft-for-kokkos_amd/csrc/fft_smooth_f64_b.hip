// Instantiation unit of the compiled 2^a 3^b 5^c lengths: F64, 108 to 250 (the
// units are compiled in parallel).
#include "fft_smooth.hpp"
#include "fft_smooth_impl.hpp"

namespace dfft {

hipError_t smooth_f64_b(const LinePass& p, hipStream_t s) {
  return dispatch_smooth<double,
      108, 120, 125, 135, 144, 150, 160, 162, 180, 192, 200, 216, 225, 240, 243, 250>(p, s);
}

}  // namespace dfft
