// Instantiation unit of the FP64 passes over the kept modes of dealiased
// fields: lengths 8 ... 1024.
#include "fft_line_impl.hpp"

namespace dfft {

namespace {
template <int N> hipError_t band(const LinePass& p, hipStream_t s) {
  return p.nontemporal ? launch_band<N, true>(p, s) : launch_band<N, false>(p, s);
}
}  // namespace

hipError_t dispatch_band_f64(const LinePass& p, hipStream_t s) {
  switch (p.n) {
    case 8: return band<8>(p, s);
    case 16: return band<16>(p, s);
    case 32: return band<32>(p, s);
    case 64: return band<64>(p, s);
    case 128: return band<128>(p, s);
    case 256: return band<256>(p, s);
    case 512: return band<512>(p, s);
    case 1024: return band<1024>(p, s);
    default: return hipErrorNotSupported;
  }
}

}  // namespace dfft
