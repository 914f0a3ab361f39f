// Instantiation unit of the kept-mode passes of the lengths 2^a 3^b 5^c: even
// lengths 144 to 240, FP64 (the units are compiled in parallel).
#include "fft_smooth.hpp"
#include "fft_smooth_impl.hpp"

namespace dfft {

hipError_t smooth_band_b(const LinePass& p, hipStream_t s) {
  return dispatch_smooth_band<
      144, 150, 160, 162, 180, 192, 200, 216, 240>(p, s);
}

}  // namespace dfft
