// Instantiation unit of the compiled 2^a 3^b 5^c lengths: F64, 3 to 100 (the
// units are compiled in parallel).
#include "fft_smooth.hpp"
#include "fft_smooth_impl.hpp"

namespace dfft {

hipError_t smooth_f64_a(const LinePass& p, hipStream_t s) {
  return dispatch_smooth<double,
      3, 5, 6, 9, 10, 12, 15, 18, 20, 24, 25, 27, 30, 36, 40, 45, 48, 50, 54, 60, 72, 75, 80, 81,
      90, 96, 100>(p, s);
}

bool smooth_length(int n) {
  if (n < 3 || n > 1024 || (n & (n - 1)) == 0) return false;
  if (n <= 256)
    while (n % 7 == 0) n /= 7;
  if (n == 1) return true;
  for (int r : {2, 3, 5})
    while (n % r == 0) n /= r;
  return n == 1;
}

hipError_t launch_smooth_f64(const LinePass& p, hipStream_t s) {
  if (p.n % 7 == 0) return smooth_f64_e(p, s);
  return p.n <= 100 ? smooth_f64_a(p, s) : p.n <= 250 ? smooth_f64_b(p, s) : p.n <= 500 ? smooth_f64_c(p, s) : smooth_f64_d(p, s);
}

}  // namespace dfft
