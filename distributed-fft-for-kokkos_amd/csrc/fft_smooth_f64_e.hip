// Instantiation unit of the compiled lengths with a factor 7: F64, 7 to 252 (the
// units are compiled in parallel).
#include "fft_smooth.hpp"
#include "fft_smooth_impl.hpp"

namespace dfft {

hipError_t smooth_f64_e(const LinePass& p, hipStream_t s) {
  return dispatch_smooth<double,
      7, 14, 21, 28, 35, 42, 49, 56, 63, 70, 84, 98, 105, 112, 126, 140, 147, 168, 175, 189, 196,
      210, 224, 245, 252>(p, s);
}

}  // namespace dfft
