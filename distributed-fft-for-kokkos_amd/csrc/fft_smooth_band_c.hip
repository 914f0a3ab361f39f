// Instantiation unit of the kept-mode passes of the lengths 2^a 3^b 5^c: even
// lengths 250 to 384, FP64 (the units are compiled in parallel).
#include "fft_smooth.hpp"
#include "fft_smooth_impl.hpp"

namespace dfft {

hipError_t smooth_band_c(const LinePass& p, hipStream_t s) {
  return dispatch_smooth_band<
      250, 270, 288, 300, 320, 324, 360, 384>(p, s);
}

}  // namespace dfft
