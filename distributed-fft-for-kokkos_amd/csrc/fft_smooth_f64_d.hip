// Instantiation unit of the compiled 2^a 3^b 5^c lengths: F64, 540 to 1000 (the
// units are compiled in parallel).
#include "fft_smooth.hpp"
#include "fft_smooth_impl.hpp"

namespace dfft {

hipError_t smooth_f64_d(const LinePass& p, hipStream_t s) {
  return dispatch_smooth<double,
      540, 576, 600, 625, 640, 648, 675, 720, 729, 750, 768, 800, 810, 864, 900, 960, 972, 1000>(p, s);
}

}  // namespace dfft
