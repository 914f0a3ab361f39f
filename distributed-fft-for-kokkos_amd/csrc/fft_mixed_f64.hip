// Instantiation unit of the runtime-radix line kernel: FP64.
#include "fft_mixed_launch.hpp"

namespace dfft {

bool mixed_length(int n, bool fp64) {
  return n >= 2 && line_length_single_pass(n, fp64) && (fp64 ? mixed_lanes_f64(n) : mixed_lanes_f32(n)) > 0;
}

bool whole_line_pass(const LinePass& p) {
  if (p.long_n1 > 0 || p.products) return false;
  if (p.in.ntopo[p.axis] != 1 || p.out.ntopo[p.axis] != 1) return false;
  return p.kind == kC2C || (p.kind == kR2C ? !p.inverse : p.inverse != 0);
}

static bool wide(int n) { return n % 11 == 0 || n % 13 == 0; }

int mixed_lanes_f64(int n) { return wide(n) ? mix_length<double, 13>(n).lanes : mix_length<double, 10>(n).lanes; }

hipError_t launch_mixed_f64(const LinePass& p, hipStream_t s) {
  return wide(p.n) ? launch_mixed<double, 13>(p, s) : launch_mixed<double, 10>(p, s);
}

}  // namespace dfft
