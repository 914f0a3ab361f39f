// Line passes of the lengths 2^a 3^b 5^c up to 1024 (without the powers of two,
// which fft_line_impl.hpp serves) and 2^a 3^b 5^c 7^d up to 256: a Stockham
// kernel compiled per length, with the radices, lanes per line and LDS
// paddings worked out at compile time.
//
// What bounds it: the runtime-radix kernel (fft_mixed_impl.hpp) spends 100 to
// 160 vector instructions per element on these lengths, most of them index
// arithmetic on plan fields, against 50 of a compiled length; its passes are
// bound by instruction issue.  Compiled, with LDS indices of a lane part and
// immediates and no radix branch, they take 45 to 75 and most complex passes
// are bound by memory again (FP64 3.7 to 6.2 TB/s, FP32 2.8 to 6.3, the shorter
// lines less); real lines, which run one by one, are bound by the latency of
// the exchanges (3.1 to 5.3 TB/s across the lines, 2.0 to 4.4 along them).
// Runtime radices -> this kernel over 39 lengths from 36 to 1000, both
// precisions, complex and real: 1.40 times as fast (passes of 24M elements, us:
// 384 real FP64 140 -> 106 along the lines, 104 -> 93 across; 375 FP32 95 -> 92,
// 128 -> 97; 1000 FP64 148 -> 133, 209 -> 173).  With factors 7 (42 to 252
// points) 1.39 times; longer ones are left to it.
// 96 and 160 against the compiled power-of-two kernel: complex FP64 160 4.4 to
// 6.0 -> 4.8 to 6.5 TB/s, FP32 160 5.0 -> 5.7 along the lines, real FP64 160 3.3 ->
// 4.1 and 2.6 -> 3.6, 96 3.2 -> 3.4 and 2.5 -> 3.2 (complex FP64 96 5.7 -> 5.4).
#pragma once

#include <hip/hip_runtime.h>

#include "fft_kernels.hpp"
#include "fft_line_impl.hpp"
#include "fft_mixed_impl.hpp"

namespace dfft {

constexpr int kSmoothStages = 6;
// Complex values a lane holds at most.  FP64 with 16 (fewer lanes, 120
// registers) ran the 39 lengths 2.6 % slower, FP32 with 20 2-13 % slower.
template <typename Real> constexpr int kSmoothValues = sizeof(Real) == 8 ? 12 : 16;
struct SmoothPlan {
  int nst = 0;
  int T = 0;  // lanes per line
  int V = 0;  // complex values a lane holds
  int rad[kSmoothStages] = {};
  int cost = 0;
};

constexpr int cdiv(int a, int b) { return (a + b - 1) / b; }
// instructions a lane spends on one value of a radix-r stage, roughly: twiddle
// and its powers, exchange, butterfly.  Counted, not fitted: the choices that
// these figures lead to were timed as a whole (above), not each against others.
constexpr int smooth_value_cost(int r) {
  return r >= 15 ? 26 : r >= 12 ? 25 : r >= 9 ? 24 : r == 8 ? 23 : r >= 5 ? 22 : r >= 4 ? 20 : 18;
}
constexpr int kSmoothLaneCost = 120;  // line addresses

// the lanes per line that suit the radices best
constexpr void smooth_try(SmoothPlan& best, const SmoothPlan& cur, int n, int most) {
  for (int T = 1; T <= n; ++T) {
    int V = 0, cost = kSmoothLaneCost;
    for (int s = 0; s < cur.nst; ++s) {
      const int values = cdiv(n / cur.rad[s], T) * cur.rad[s];
      V = values > V ? values : V;
      cost += values * smooth_value_cost(cur.rad[s]);
    }
    if (V > most) continue;
    cost *= T;
    if (best.nst == 0 || cost < best.cost) {
      best = cur;
      best.T = T;
      best.V = V;
      best.cost = cost;
    }
    if (V * 3 < most) break;
  }
}
constexpr void smooth_search(SmoothPlan& best, const SmoothPlan& cur, int n, int rest, int top, int most) {
  if (rest == 1) {
    smooth_try(best, cur, n, most);
    return;
  }
  if (cur.nst >= 4) return;
  constexpr int kRadix[] = {16, 15, 12, 10, 9, 8, 7, 6, 5, 4, 3, 2};
  for (int r : kRadix) {
    if (r > top || rest % r) continue;
    SmoothPlan next = cur;
    next.rad[next.nst++] = r;
    smooth_search(best, next, n, rest / r, r, most);
  }
}
// Radices in descending order (the first stage multiplies by no twiddles) and
// lanes per line of the least modelled work.
constexpr SmoothPlan smooth_plan(int n, int most) {
  SmoothPlan best;
  smooth_search(best, SmoothPlan{}, n, n, 16, most);
  return best;
}

// Padding of the exchange after a stage: lanes write runs of L positions, one
// run every L r + pad.  The one of fewest bank conflicts (a cycle serves 128
// bytes) of those up to an eighth of the run distance.
constexpr int smooth_pad(int L, int r, int T, int elem) {
  const int slots = 128 / elem;
  const int lim = L * r / 8 > 1 ? L * r / 8 : 1;
  int best = 0, best_sum = 1 << 30;
  for (int pad = 0; pad <= lim && pad < slots; ++pad) {
    int sum = 0;
    for (int first = 0; first < 64 && first < T; first += slots) {
      int hits[32] = {}, most = 0;
      for (int t = first; t < first + slots && t < T; ++t) {
        const int at = (t / L * (L * r + pad) + t % L) % slots;
        most = ++hits[at] > most ? hits[at] : most;
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

template <typename Real, int N> struct SmoothCfg {
  static constexpr SmoothPlan P = smooth_plan(N, kSmoothValues<Real>);
  static constexpr int T = P.T, V = P.V, NST = P.nst;
  // exchanges in real and imaginary halves where whole lines would leave few blocks per CU
  static constexpr bool SPLIT = N * 2 * sizeof(Real) > 4096;
  static constexpr int ELEM = SPLIT ? sizeof(Real) : 2 * sizeof(Real);
  static constexpr int span(int s) {  // product of the radices before stage s
    int L = 1;
    for (int i = 0; i < s; ++i) L *= P.rad[i];
    return L;
  }
  static constexpr int pad(int s) { return s + 1 < NST ? smooth_pad(span(s), P.rad[s], T, ELEM) : 0; }
  static constexpr int ldsn() {
    int most = N + 1;
    for (int s = 0; s + 1 < NST; ++s) {
      const int x = N + (N / span(s + 1) - 1) * pad(s);
      most = x > most ? x : most;
    }
    return most;
  }
  static constexpr int LDSN = ldsn();
  // Lines of a block across the lines, at least: a 128-byte segment of a row
  // (FP32 passes over 24M elements, 8 / 16 lines: 300 points 46 / 43 us, 480
  // 105 / 97, 675 122 / 99), half of it where a block would pass 768 lanes (960
  // points 49 / 56 us).
  static constexpr int LEAST = sizeof(Real) == 4 && 16 * T <= 768 ? 16 : 8;
  static constexpr int LANES = T * LEAST <= 256 ? 256 : T * LEAST <= 512 ? 512 : 1024;  // most lanes of a block
};

// Stage S: lane t carries butterflies beta = t + q T (q < NB); their inputs
// are positions beta + j nr, their outputs (beta / L) L r + beta % L + j L.
template <typename Real, int N, int S> struct SmoothStage {
  using Cfg = SmoothCfg<Real, N>;
  static constexpr int r = Cfg::P.rad[S], T = Cfg::T, nr = N / r, L = Cfg::span(S), ts = N / (L * r);
  static constexpr int NB = cdiv(nr, T);
  static constexpr int out_group = L * r + Cfg::pad(S);
  static constexpr int in_pad = S > 0 ? Cfg::pad(S > 0 ? S - 1 : 0) : 0;
  static constexpr int in_step = nr + nr / L * in_pad;
  static constexpr int NTW = mix_ntw<r, Real>();
  static constexpr bool kShared = T % L == 0;  // every butterfly of the lane has the same twiddles
  __device__ static __forceinline__ bool on(int t, int q) { return (q + 1) * T <= nr || t + q * T < nr; }
  // beta / L (exact for beta < 1024)
  __device__ static __forceinline__ int group(int beta) {
    if constexpr (L == 1) return beta;
    else if constexpr (L >= nr) return 0;
    else if constexpr ((L & (L - 1)) == 0) return static_cast<int>(static_cast<unsigned>(beta) / L);
    else return static_cast<int>(__umul24(static_cast<unsigned>(beta), (1u << 20) / L + 1) >> 20);
  }
  __device__ static __forceinline__ int gather_base(int beta) { return beta + group(beta) * in_pad; }
  __device__ static __forceinline__ int scatter_base(int beta) { return beta + group(beta) * (out_group - L); }

  __device__ static __forceinline__ void load_twiddles(double2* w, int t, const double2* tw) {
    if constexpr (L > 1) {
#pragma unroll
      for (int q = 0; q < (kShared ? 1 : NB); ++q) {
        if (on(t, q)) {
          const int beta = t + q * T;
          const int e = (beta - group(beta) * L) * ts;
#pragma unroll
          for (int i = 0; i < NTW; ++i) w[q * NTW + i] = twiddle_load(tw + (i + 1) * e);
        }
      }
    }
  }
  template <typename C> __device__ static __forceinline__ void compute(C* v, int t, const double2* w) {
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      if (on(t, q)) {
        if constexpr (L > 1) mix_twiddle<r>(v + q * r, w + (kShared ? 0 : q * NTW));
        mix_bfly<r>(v + q * r);
      }
    }
  }
};

// the stages from S on; inputs and outputs in registers.  FRESH: no lane of
// the block reads the line's LDS any more.
template <typename Real, int N, int S, bool FRESH>
__device__ __forceinline__ void smooth_stages(cplx_t<Real>* v, int t, void* buf, const double2* tw, const double2* w) {
  using C = cplx_t<Real>;
  using Cfg = SmoothCfg<Real, N>;
  using St = SmoothStage<Real, N, S>;
  constexpr int T = Cfg::T;
  St::compute(v, t, w);
  if constexpr (S + 1 < Cfg::NST) {
    using Nx = SmoothStage<Real, N, S + 1>;
    double2 wn[Nx::NB * Nx::NTW];
    if constexpr (!FRESH) __syncthreads();
    if constexpr (Cfg::SPLIT) {
      Real* lr = static_cast<Real*>(buf);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (h) __syncthreads();
#pragma unroll
        for (int q = 0; q < St::NB; ++q) {
          if (St::on(t, q)) {
            Real* dst = lr + St::scatter_base(t + q * T);
#pragma unroll
            for (int j = 0; j < St::r; ++j) dst[j * St::L] = h ? v[q * St::r + j].y : v[q * St::r + j].x;
          }
        }
        // the next stage's twiddles are on their way during the exchange
        if (!h) Nx::load_twiddles(wn, t, tw);
        __syncthreads();
#pragma unroll
        for (int q = 0; q < Nx::NB; ++q) {
          if (Nx::on(t, q)) {
            const Real* src = lr + Nx::gather_base(t + q * T);
#pragma unroll
            for (int j = 0; j < Nx::r; ++j) {
              const Real x = src[j * Nx::in_step];
              if (h) {
                v[q * Nx::r + j].y = x;
              } else {
                v[q * Nx::r + j].x = x;
              }
            }
          }
        }
      }
    } else {
      C* lc = static_cast<C*>(buf);
#pragma unroll
      for (int q = 0; q < St::NB; ++q) {
        if (St::on(t, q)) {
          C* dst = lc + St::scatter_base(t + q * T);
#pragma unroll
          for (int j = 0; j < St::r; ++j) dst[j * St::L] = v[q * St::r + j];
        }
      }
      Nx::load_twiddles(wn, t, tw);
      __syncthreads();
#pragma unroll
      for (int q = 0; q < Nx::NB; ++q) {
        if (Nx::on(t, q)) {
          const C* src = lc + Nx::gather_base(t + q * T);
#pragma unroll
          for (int j = 0; j < Nx::r; ++j) v[q * Nx::r + j] = src[j * Nx::in_step];
        }
      }
    }
    smooth_stages<Real, N, S + 1, false>(v, t, buf, tw, wn);
  }
}

// One line per T lanes.  Real lines run one by one: two of them as one complex
// line (as the power-of-two lengths do) take half the arithmetic, but then an
// infinity or a large value of one line reaches the other, which may belong to
// another transform, and the error of a C2R line is up to 1.35 times as large.
// The zero imaginary parts of R2C inputs and the unused ones of C2R outputs
// drop out of the first and the last stage.
// BAND: a pass of a dealiased field's kept modes (LinePass::band): modes beyond
// are neither read (zeros) nor stored.  PROD: a products pass
// (LinePass::products): the field axis is the fastest batch axis.
template <typename Real, int N, bool NT, int KIND, bool PROD = false, bool BAND = false>
__global__ void __launch_bounds__((SmoothCfg<Real, N>::LANES)) fft_smooth(const FastPass p) {
  using C = cplx_t<Real>;
  using Cfg = SmoothCfg<Real, N>;
  using S0 = SmoothStage<Real, N, 0>;
  using Sl = SmoothStage<Real, N, Cfg::NST - 1>;
  constexpr int T = Cfg::T;
  extern __shared__ unsigned char smem_raw[];
  const int tid = threadIdx.x, B = p.lines_per_block;
  int b, t;
  if (p.lines_fast) {
    t = static_cast<int>(p.bdiv.div(static_cast<uint32_t>(tid)));
    b = tid - t * B;
  } else {
    b = tid / T;
    t = tid % T;
  }
  int32_t unit = pass_block(p, blockIdx.x, gridDim.x) * B + b;
  // a wave holds one line: its addresses are worked out on the scalar unit
  if (T % 64 == 0 && !p.lines_fast) unit = __builtin_amdgcn_readfirstlane(unit);
  const double2* tw = reinterpret_cast<const double2*>(p.tw);
  void* buf = smem_raw + b * p.line_bytes;
  C v[Cfg::V];
#pragma unroll
  for (int j = 0; j < Cfg::V; ++j) v[j] = C{Real(0), Real(0)};

  LineIO<Real, NT> io{};
  bool valid = unit < p.nlines;
  if (valid) valid = make_line_io<Real, NT, BAND, PROD>(p, unit, io);
  if constexpr (KIND == kC2C) {
    if (valid) {
#pragma unroll
      for (int q = 0; q < S0::NB; ++q) {
        if (S0::on(t, q)) {
          const C* src = reinterpret_cast<const C*>(io.ib) + (t + q * T) * io.is;
          const int64_t step = S0::nr * io.is;
#pragma unroll
          for (int j = 0; j < S0::r; ++j) {
            if constexpr (BAND) {
              // lanes beyond the band repeat the line's first address
              const int at = t + q * T + j * S0::nr;
              const bool keep = !p.inverse || at <= p.band || at >= N - p.band;
              const C x = gload_c<NT, Real>(keep ? src : reinterpret_cast<const C*>(io.ib));
              v[q * S0::r + j] = keep ? x : C{Real(0), Real(0)};
            } else {
              v[q * S0::r + j] = gload_c<NT, Real>(src);
            }
            src += step;
          }
        }
      }
      if (p.inverse) {
#pragma unroll
        for (int j = 0; j < Cfg::V; ++j) v[j].y = -v[j].y;
      }
    }
    smooth_stages<Real, N, 0, true>(v, t, buf, tw, nullptr);
    if (valid) {
      const Real sy = p.inverse ? -io.scale : io.scale;
#pragma unroll
      for (int q = 0; q < Sl::NB; ++q) {
        if (Sl::on(t, q)) {
          C* dst = reinterpret_cast<C*>(io.ob) + (t + q * T) * io.os;
          const int64_t step = Sl::nr * io.os;
#pragma unroll
          for (int j = 0; j < Sl::r; ++j) {
            const int at = t + q * T + j * Sl::nr;
            if (!BAND || p.inverse || at <= p.band || at >= N - p.band)
              gstore_c<NT, Real>(dst, C{v[q * Sl::r + j].x * io.scale, v[q * Sl::r + j].y * sy});
            dst += step;
          }
        }
      }
    }
  } else if constexpr (KIND == kR2C) {
    if constexpr (PROD) {
      // slots 6m..6m+5 are the product fields of one position: the first three
      // stage its velocity lines, each then forms its product line from LDS
      const int f = b % 6;
      Real* st = reinterpret_cast<Real*>(smem_raw + (b - f) * p.line_bytes);
      if (valid && f < 3) {
#pragma unroll
        for (int q = 0; q < S0::NB; ++q) {
          if (S0::on(t, q)) {
            const Real* src = reinterpret_cast<const Real*>(io.ib) + (t + q * T) * io.is;
            const int64_t step = S0::nr * io.is;
#pragma unroll
            for (int j = 0; j < S0::r; ++j) {
              st[f * N + t + q * T + j * S0::nr] = gload<NT>(src);
              src += step;
            }
          }
        }
      }
      __syncthreads();
      const Real* f0 = st + prod_first(f) * N;
      const Real* f1 = st + prod_second(f) * N;
#pragma unroll
      for (int q = 0; q < S0::NB; ++q) {
        if (S0::on(t, q)) {
#pragma unroll
          for (int j = 0; j < S0::r; ++j) {
            const int at = t + q * T + j * S0::nr;
            v[q * S0::r + j].x = f0[at] * f1[at];
          }
        }
      }
    } else if (valid) {
#pragma unroll
      for (int q = 0; q < S0::NB; ++q) {
        if (S0::on(t, q)) {
          const Real* src = reinterpret_cast<const Real*>(io.ib) + (t + q * T) * io.is;
          const int64_t step = S0::nr * io.is;
#pragma unroll
          for (int j = 0; j < S0::r; ++j) {
            v[q * S0::r + j].x = gload<NT>(src);
            src += step;
          }
        }
      }
    }
    smooth_stages<Real, N, 0, !PROD>(v, t, buf, tw, nullptr);  // the staged lines share LDS with the exchanges
    if (valid) {
      constexpr int LOW = (N + 1) / (2 * Sl::nr);  // outputs j < LOW lie below n/2
      constexpr int TOP = N / 2 / Sl::nr;          // outputs j > TOP above
      const Real hw = io.scale * io.hw;
#pragma unroll
      for (int q = 0; q < Sl::NB; ++q) {
        if (Sl::on(t, q)) {
          const int beta = t + q * T;
          C* dst = reinterpret_cast<C*>(io.ob) + beta * io.os;
          const int64_t step = Sl::nr * io.os;
#pragma unroll
          for (int j = 0; j <= TOP; ++j) {
            const int at = beta + j * Sl::nr;
            const bool self = (j == 0 && q == 0 && t == 0) || (j >= LOW && 2 * at == N);
            const C z = v[q * Sl::r + j];
            const Real h = self ? io.scale : hw;
            if (BAND ? at <= p.band : j < LOW || 2 * at <= N) gstore_c<NT, Real>(dst, C{z.x * h, z.y * h});
            dst += step;
          }
        }
      }
    }
  } else {
    // C2R: the lane that holds position m <= n/2 loads entry m of the half
    // spectrum, takes its conjugate as the input at m and hands the entry over
    // through LDS as the input at n - m
    constexpr int LOW = (N + 1) / (2 * S0::nr), TOP = N / 2 / S0::nr;
    C up[S0::NB * (TOP + 1)];
#pragma unroll
    for (int k = 0; k < S0::NB * (TOP + 1); ++k) up[k] = C{Real(0), Real(0)};
    if (valid) {
#pragma unroll
      for (int q = 0; q < S0::NB; ++q) {
        if (S0::on(t, q)) {
          const int beta = t + q * T;
          const C* src = reinterpret_cast<const C*>(io.ib) + beta * io.is;
          const int64_t step = S0::nr * io.is;
#pragma unroll
          for (int j = 0; j <= TOP; ++j) {
            // above n/2 (only lanes of the middle output): the first entry again, not used
            const bool low = BAND ? beta + j * S0::nr <= p.band : j < LOW || 2 * (beta + j * S0::nr) <= N;
            const C x = gload_c<NT, Real>(low ? src : reinterpret_cast<const C*>(io.ib));
            up[q * (TOP + 1) + j] = BAND && !low ? C{Real(0), Real(0)} : x;
            src += step;
          }
        }
      }
    }
#pragma unroll
    for (int q = 0; q < S0::NB; ++q) {
#pragma unroll
      for (int j = 0; j <= TOP; ++j) {
        const int at = t + q * T + j * S0::nr, k = q * (TOP + 1) + j;
        const bool self = (j == 0 && q == 0 && t == 0) || (j >= LOW && 2 * at == N);
        const Real hw = self ? Real(1) : io.hw;
        up[k].x *= hw;
        up[k].y = self ? Real(0) : up[k].y * hw;
        v[q * S0::r + j] = cconj(up[k]);
      }
    }
    auto hand = [&](auto* lds, auto value, auto take) {
#pragma unroll
      for (int q = 0; q < S0::NB; ++q) {
        if (S0::on(t, q)) {
#pragma unroll
          for (int j = 0; j <= TOP; ++j) {
            const int at = t + q * T + j * S0::nr;
            if ((j > 0 || q > 0 || t > 0) && (j < LOW || 2 * at < N)) lds[N - at] = value(up[q * (TOP + 1) + j]);
          }
        }
      }
      __syncthreads();
#pragma unroll
      for (int q = 0; q < S0::NB; ++q) {
        if (S0::on(t, q)) {
#pragma unroll
          for (int j = LOW; j < S0::r; ++j) {
            const int at = t + q * T + j * S0::nr;
            if (j > TOP || 2 * at > N) take(v[q * S0::r + j], lds[at]);
          }
        }
      }
    };
    if constexpr (Cfg::SPLIT) {
      hand(static_cast<Real*>(buf), [](const C& x) { return x.x; }, [](C& d, Real x) { d.x = x; });
      __syncthreads();
      hand(static_cast<Real*>(buf), [](const C& x) { return x.y; }, [](C& d, Real x) { d.y = x; });
    } else {
      hand(static_cast<C*>(buf), [](const C& x) { return x; }, [](C& d, const C& x) { d = x; });
    }
    smooth_stages<Real, N, 0, false>(v, t, buf, tw, nullptr);
    if (valid) {
#pragma unroll
      for (int q = 0; q < Sl::NB; ++q) {
        if (Sl::on(t, q)) {
          Real* dst = reinterpret_cast<Real*>(io.ob) + (t + q * T) * io.os;
          const int64_t step = Sl::nr * io.os;
#pragma unroll
          for (int j = 0; j < Sl::r; ++j) {
            gstore<NT>(dst, v[q * Sl::r + j].x * io.scale);
            dst += step;
          }
        }
      }
    }
  }
}

namespace {

template <typename Real, int N, bool NT, int KIND>
hipError_t launch_smooth_kernel(const LinePass& p, unsigned grid, unsigned threads, size_t smem, hipStream_t s) {
  static std::atomic<size_t> limit{64 * 1024};
  const hipError_t e = raise_lds_limit(limit, reinterpret_cast<const void*>(&fft_smooth<Real, N, NT, KIND>), smem);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((fft_smooth<Real, N, NT, KIND>), dim3(grid), dim3(threads), smem, s,
                     fast_pass(p, sizeof(Real) == 8));
  return hipGetLastError();
}

template <typename Real, int N>
hipError_t launch_smooth(LinePass p, hipStream_t s) {
  using Cfg = SmoothCfg<Real, N>;
  constexpr int T = Cfg::T;
  const int64_t units = p.nlines;
  if (units <= 0) return hipSuccess;
  int B = p.lines_per_block;
  if constexpr (N == 96 || N == 160) {
    // a caller's block shape beyond a workgroup of the power-of-two kernel,
    // which runs these lengths too, is refused, as it always was
    const bool split = split_available<Real, N>() && p.split_lds != 0;
    const size_t line = split ? line_lds_bytes<Real, N, 8, true>() : line_lds_bytes<Real, N, 8, false>();
    if (!p.fit_block && B > 0 && (B * FastCfg<Real, N, 8>::T > 1024 || B * line > kGenericLdsMax))
      return hipErrorInvalidConfiguration;
  }
  if (B <= 0) {
    if (p.lines_fast) {
      B = 32;
      while (B > Cfg::LEAST && B * T > 256) B /= 2;
    } else {
      // one wave: its barriers cost least (1.1 % over 256 lanes, 39 lengths)
      B = T >= 64 ? 1 : 64 / T;
    }
    while (B > 1 && (units + B - 1) / B < 512 && B * T > 64) B = (B + 1) / 2;
  }
  constexpr size_t kLine = static_cast<size_t>(Cfg::LDSN) * Cfg::ELEM;
  auto stride = [&](int lines) { return line_stride(kLine, Cfg::ELEM, p.lines_fast != 0, lines, T); };
  while (B > 1 && (B * T > Cfg::LANES || static_cast<size_t>(B) * stride(B) > kGenericLdsMax)) B /= 2;
  p.lines_per_block = B;
  p.line_bytes = static_cast<int32_t>(stride(B));
  p.swizzle = 0;
  const size_t smem = Cfg::NST > 1 || p.kind != kC2C ? static_cast<size_t>(B) * p.line_bytes : 0;
  const unsigned grid = static_cast<unsigned>((units + B - 1) / B), threads = static_cast<unsigned>(B * T);
  const bool nt = p.nontemporal != 0;
  switch (p.kind) {
    case kC2C:
      return nt ? launch_smooth_kernel<Real, N, true, kC2C>(p, grid, threads, smem, s)
                : launch_smooth_kernel<Real, N, false, kC2C>(p, grid, threads, smem, s);
    case kR2C:
      return nt ? launch_smooth_kernel<Real, N, true, kR2C>(p, grid, threads, smem, s)
                : launch_smooth_kernel<Real, N, false, kR2C>(p, grid, threads, smem, s);
    default:
      return nt ? launch_smooth_kernel<Real, N, true, kC2R>(p, grid, threads, smem, s)
                : launch_smooth_kernel<Real, N, false, kC2R>(p, grid, threads, smem, s);
  }
}

template <int N, int KIND, bool PROD>
hipError_t launch_smooth_band_kernel(const LinePass& p, unsigned grid, unsigned threads, size_t smem, hipStream_t s) {
  static std::atomic<size_t> limit{64 * 1024};
  const void* fn = reinterpret_cast<const void*>(&fft_smooth<double, N, false, KIND, PROD, true>);
  const hipError_t e = raise_lds_limit(limit, fn, smem);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((fft_smooth<double, N, false, KIND, PROD, true>), dim3(grid), dim3(threads), smem, s,
                     fast_pass(p, true));
  return hipGetLastError();
}

// a kept-mode pass (launch_band_pass)
template <int N>
hipError_t launch_smooth_band(LinePass p, hipStream_t s) {
  using Cfg = SmoothCfg<double, N>;
  constexpr int T = Cfg::T;
  if (p.kind != kC2C && (p.kind == kR2C) == (p.inverse != 0)) return hipErrorInvalidValue;
  if (p.products && (p.kind != kR2C || p.nlines % 6 != 0 || p.line_begin % 6 != 0)) return hipErrorInvalidConfiguration;
  const int64_t units = p.nlines;
  if (units <= 0) return hipSuccess;
  int B;
  if (p.products) {
    B = std::max(1, 256 / (6 * T)) * 6;  // whole positions
  } else if (p.lines_fast) {
    B = 32;
    while (B > Cfg::LEAST && B * T > 256) B /= 2;
  } else {
    B = T >= 64 ? 1 : 64 / T;
  }
  if (!p.products)
    while (B > 1 && (units + B - 1) / B < 512 && B * T > 64) B = (B + 1) / 2;
  constexpr size_t kLine = static_cast<size_t>(Cfg::LDSN) * Cfg::ELEM;
  const size_t stride = line_stride(kLine, Cfg::ELEM, p.lines_fast != 0, B, T);
  if (B * T > Cfg::LANES || B * stride > kGenericLdsMax) return hipErrorInvalidConfiguration;
  p.lines_per_block = B;
  p.line_bytes = static_cast<int32_t>(stride);
  p.swizzle = 0;
  const size_t smem = B * stride;
  const unsigned grid = static_cast<unsigned>((units + B - 1) / B), threads = static_cast<unsigned>(B * T);
  if (p.kind == kC2C) return launch_smooth_band_kernel<N, kC2C, false>(p, grid, threads, smem, s);
  if (p.kind == kC2R) return launch_smooth_band_kernel<N, kC2R, false>(p, grid, threads, smem, s);
  return p.products ? launch_smooth_band_kernel<N, kR2C, true>(p, grid, threads, smem, s)
                    : launch_smooth_band_kernel<N, kR2C, false>(p, grid, threads, smem, s);
}

template <int... Ns>
hipError_t dispatch_smooth_band(const LinePass& p, hipStream_t s) {
  hipError_t e = hipErrorNotSupported;
  static_cast<void>(((p.n == Ns ? (e = launch_smooth_band<Ns>(p, s), true) : false) || ...));
  return e;
}

// runs p on the kernel of its length if it is one of Ns
template <typename Real, int... Ns>
hipError_t dispatch_smooth(const LinePass& p, hipStream_t s) {
  hipError_t e = hipErrorNotSupported;
  static_cast<void>(((p.n == Ns ? (e = launch_smooth<Real, Ns>(p, s), true) : false) || ...));
  return e;
}

}  // namespace
}  // namespace dfft
