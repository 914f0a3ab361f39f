// Instantiation unit of the compiled 2^a 3^b 5^c lengths: F64, 270 to 500 (the
// units are compiled in parallel).
#include "fft_smooth.hpp"
#include "fft_smooth_impl.hpp"

namespace dfft {

hipError_t smooth_f64_c(const LinePass& p, hipStream_t s) {
  return dispatch_smooth<double,
      270, 288, 300, 320, 324, 360, 375, 384, 400, 405, 432, 450, 480, 486, 500>(p, s);
}

}  // namespace dfft
