// Radix plan, block shape and launcher of the runtime-radix line kernel, one
// instantiation per precision (fft_mixed_f64.hip, fft_mixed_f32.hip).
#pragma once

#include "fft_mixed.hpp"
#include "fft_mixed_impl.hpp"

#include <algorithm>
#include <map>
#include <mutex>
#include <vector>

namespace dfft {
namespace {

inline int ceil_div(int a, int b) { return (a + b - 1) / b; }
inline int log2i(int v) {  // of a power of two, at most 6
  int k = 0;
  while (k < 6 && (2 << k) <= v) ++k;
  return k;
}

// lanes a line of length n needs when every lane carries as many butterflies
// of each stage as its registers hold
template <int V>
inline int mix_lanes_packed(int n, const std::vector<int>& rad) {
  int T = 1;
  for (int r : rad) T = std::max(T, ceil_div(n / r, mix_nb<V>(r)));
  return T;
}

// Radices of n: the fewest stages (each costs an exchange through LDS), then
// the fewest lanes per line (every stage then fills the lanes' registers
// alike: 375 = 15 * 5 * 5 takes 25 lanes of 15 values), the largest radix
// first (stage 0 multiplies by no twiddles).  Empty if n has a prime factor
// above V.
template <int V>
inline std::vector<int> mix_radices(int n) {
  static const int kRadix[] = {16, 15, 13, 12, 11, 10, 9, 8, 7, 6, 5, 4, 3, 2};
  std::vector<int> best, cur;
  int best_lanes = 0;
  auto search = [&](auto&& self, int rest, int from) -> void {
    if (rest == 1) {
      const int lanes = mix_lanes_packed<V>(n, cur);
      if (best.empty() || cur.size() < best.size() || (cur.size() == best.size() && lanes < best_lanes)) {
        best = cur;
        best_lanes = lanes;
      }
      return;
    }
    if (cur.size() + 1 > static_cast<std::size_t>(kMixStages) || (!best.empty() && cur.size() + 1 > best.size())) return;
    for (int i = from; i < static_cast<int>(sizeof(kRadix) / sizeof(int)); ++i) {
      if (rest % kRadix[i] || !mix_has<V>(kRadix[i])) continue;
      cur.push_back(kRadix[i]);
      self(self, rest / kRadix[i], i);
      cur.pop_back();
    }
  };
  if (n >= 2) search(search, n, 0);
  return best;
}

// Padding of the exchange after a stage of radix r over L positions: lanes
// write runs of L positions, one run every L r + pad.  Of the paddings up to
// an eighth of the run distance (at least one), the one with the fewest bank
// conflicts: a cycle serves 128 bytes, 16 lanes of 8 or 32 of 4, `across` of
// them adjacent for every position.
template <typename Real>
inline int mix_pad(int L, int r, int across) {
  constexpr int kSlots = 128 / static_cast<int>(sizeof(Real));
  int best = 0, best_sum = 1 << 30;
  for (int pad = 0; pad <= std::min(std::max(1, L * r / 8), kSlots - 1) && best_sum > 64 / kSlots; ++pad) {
    int sum = 0;
    for (int first = 0; first < 64; first += kSlots) {
      int hits[kSlots] = {}, most = 0;
      for (int lane = first; lane < first + kSlots; ++lane) {
        const int b = lane % across, beta = lane / across;
        const int at = ((beta / L) * (L * r + pad) + beta % L) * across + b;
        most = std::max(most, ++hits[at % kSlots]);
      }
      sum += most;
    }
    if (sum < best_sum) {
      best_sum = sum;
      best = pad;
    }
  }
  return best;
}

// what the kernel needs to know of a length, worked out once
struct MixLength {
  std::vector<int> rad;              // empty: not a length of this instance
  int lanes = 0;                     // per line, packed shape
  int pad[kMixStages][7] = {};       // by stage and log2 of the lanes across lines (at most 64)
};

template <typename Real, int V>
inline const MixLength& mix_length(int n) {
  static std::mutex lock;
  static std::map<int, MixLength> known;  // nodes stay where they are
  std::lock_guard<std::mutex> hold(lock);
  auto it = known.find(n);
  if (it != known.end()) return it->second;
  MixLength l;
  l.rad = mix_radices<V>(n);
  if (!l.rad.empty()) l.lanes = mix_lanes_packed<V>(n, l.rad);
  if (l.lanes > 1024) l = MixLength{};
  int L = 1;
  for (std::size_t i = 0; i + 1 < l.rad.size(); ++i) {
    for (int k = 0; k < 7; ++k) l.pad[i][k] = mix_pad<Real>(L, l.rad[i], 1 << k);
    L *= l.rad[i];
  }
  return known.emplace(n, l).first->second;
}

template <typename Real, int V, bool NT, int KIND>
hipError_t launch_mixed_kernel(const LinePass& p, const MixPlan& m, unsigned grid, unsigned threads, size_t smem,
                               hipStream_t s) {
  static std::atomic<size_t> limit{64 * 1024};
  const hipError_t e = raise_lds_limit(limit, reinterpret_cast<const void*>(&fft_mixed<Real, V, NT, KIND>), smem);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((fft_mixed<Real, V, NT, KIND>), dim3(grid), dim3(threads), smem, s, fast_pass(p, sizeof(Real) == 8), m);
  return hipGetLastError();
}

template <typename Real, int V>
hipError_t launch_mixed(LinePass p, hipStream_t s) {
  const int n = p.n;
  const MixLength& len = mix_length<Real, V>(n);
  const std::vector<int>& rad = len.rad;
  if (rad.empty()) return hipErrorNotSupported;
  int T = len.lanes;
  const int64_t units = p.nlines;
  if (units <= 0) return hipSuccess;

  // Lanes per line: full registers, or one butterfly per lane where the pass
  // would otherwise leave most of the chip's 1024 SIMDs without a wave.
  if (p.values_per_thread > 0) T = std::min(1024, std::max(T, ceil_div(n, p.values_per_thread)));
  else if (units * T < 1024 * 64) T = std::min(1024, std::max(T, n / *std::min_element(rad.begin(), rad.end())));
  // Lines per block: blocks of up to 256 lanes; across lines a power of two,
  // 8 to 32 adjacent lines (strided passes over 33.5M elements, GB/s read and
  // written with 8 / 16 / 32 lines: FP64 n = 50 4640 / 4790 / 4960, n = 100
  // 4680 / 4840 / -, n = 250 4100 / 4030 / -; FP32 n = 162 2250 / 1860 / 2000,
  // n = 250 2850 / 2550 / -, n = 50 - / 3500 / 3990).  Fewer lines while the
  // pass has less than two blocks per CU.
  int B = p.lines_per_block;
  if (B <= 0) {
    if (p.lines_fast) {
      B = 32;
      while (B > 8 && B * T > 256) B /= 2;
    } else {
      B = std::max(1, 256 / T);
    }
    while (B > 1 && (units + B - 1) / B < 512 && B * T > 64) B = (B + 1) / 2;
  }
  if (p.lines_fast) {
    B = std::min(B, 64);
    while (B & (B - 1)) B &= B - 1;
  }
  // LDS elements of a line with the paddings of its exchanges
  auto ldsn = [&](int lines) {
    const int k = p.lines_fast ? log2i(lines) : 0;
    int most = n;
    for (int i = 0, L = 1; i + 1 < static_cast<int>(rad.size()); ++i) {
      L *= rad[i];
      most = std::max(most, n + (n / L - 1) * len.pad[i][k]);
    }
    constexpr int kReal = static_cast<int>(sizeof(Real));
    return p.lines_fast ? most
                        : static_cast<int>(line_stride(static_cast<size_t>(most) * kReal, kReal, false, lines, T)) / kReal;
  };
  while (B > 1 && (B * T > 1024 || static_cast<size_t>(B) * ldsn(B) * sizeof(Real) > kGenericLdsMax)) B /= 2;
  const int line = ldsn(B);
  const size_t smem = static_cast<size_t>(B) * line * sizeof(Real);
  if (B * T > 1024 || smem > kGenericLdsMax) return hipErrorInvalidConfiguration;

  MixPlan m{};
  m.nst = static_cast<int32_t>(rad.size());
  m.T = T;
  m.dT = FastDiv(static_cast<uint32_t>(T));
  m.log2B = p.lines_fast ? log2i(B) : 0;
  m.ps = p.lines_fast ? B : 1;
  m.bs = p.lines_fast ? 1 : line;
  int L = 1;
  for (int i = 0; i < m.nst; ++i) {
    MixStage& st = m.st[i];
    st.r = rad[i];
    st.nr = n / rad[i];
    st.L = L;
    st.ts = n / (L * rad[i]);
    st.dL = FastDiv(static_cast<uint32_t>(L));
    st.in_pad = i > 0 ? m.st[i - 1].out_group - L : 0;
    st.in_step = (st.nr + st.nr / L * st.in_pad) * m.ps;
    st.out_group = L * rad[i] + (i + 1 < m.nst ? len.pad[i][m.log2B] : 0);
    L *= rad[i];
  }
  p.lines_per_block = B;
  p.swizzle = 0;
  const unsigned grid = static_cast<unsigned>((units + B - 1) / B);
  const unsigned threads = static_cast<unsigned>((B * T + 63) / 64 * 64);
  const bool nt = p.nontemporal != 0;
  switch (p.kind) {
    case kC2C:
      return nt ? launch_mixed_kernel<Real, V, true, kC2C>(p, m, grid, threads, smem, s)
                : launch_mixed_kernel<Real, V, false, kC2C>(p, m, grid, threads, smem, s);
    case kR2C:
      return nt ? launch_mixed_kernel<Real, V, true, kR2C>(p, m, grid, threads, smem, s)
                : launch_mixed_kernel<Real, V, false, kR2C>(p, m, grid, threads, smem, s);
    default:
      return nt ? launch_mixed_kernel<Real, V, true, kC2R>(p, m, grid, threads, smem, s)
                : launch_mixed_kernel<Real, V, false, kC2R>(p, m, grid, threads, smem, s);
  }
}

}  // namespace
}  // namespace dfft
