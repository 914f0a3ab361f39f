// Line passes of any length n = product of radices 2..13, 15, 16 (every n
// without a prime factor above 13): a Stockham kernel whose radices are read
// from the launch's plan and whose butterflies are straight-line code on
// registers.  It serves the lengths without a compiled kernel
// (fft_line_impl.hpp, fft_smooth_impl.hpp): those with a factor 11 or 13,
// those with a 7 above 256 and those above 1024, e.g. 143, 504, 1155, 1536.
//
// Why this shape: the per-element kernel (fft_line_generic) forms every output
// of a radix-r stage as an r-term sum read from LDS, 4 to 16 LDS reads and
// complex products per element and stage, and moves 0.25 to 0.9 TB/s.  Here a
// lane reads a butterfly's r inputs once, so LDS traffic and arithmetic drop
// by about r; a pass is bound by instruction issue (100 to 160 vector
// instructions per element) at 1.1 to 5.4 TB/s, in the middle 2.6.  An LDS index
// with a shift per element instead of one constant step per exchange cost
// 5-10 % there.  Per-element kernel -> this one over ten lengths from 99 to 2187,
// both precisions, complex and real: 4.8 times as fast (24M elements, us: 1536
// complex FP64 1064 -> 182 along the lines, 1312 -> 277 across; 504 real FP32 639
// -> 83, 392 -> 76).
#pragma once

#include <hip/hip_runtime.h>

#include "fft_kernels.hpp"
#include "fft_line_impl.hpp"

namespace dfft {

constexpr int kMixStages = 8;
// V: complex values a lane holds at most, and with it the radices a kernel
// instance knows.  FP32 lanes hold 16.  FP64 lanes hold 10: with 16 (or with
// radices 12 to 16) the kernel spills registers at the 128 that a block of
// 1024 lanes leaves it; lengths with a factor 11 or 13 run an instance of
// their own with up to 13 (a few spill slots).
template <int V> constexpr bool mix_has(int r) { return r <= V; }
// butterflies of radix r a lane carries through one stage
template <int V> constexpr int mix_nb_max() { return V >= 16 ? 4 : 2; }
template <int V> constexpr int mix_nb(int r) { return V / r < mix_nb_max<V>() ? V / r : mix_nb_max<V>(); }
// half-spectrum entries a lane handles at most (n/2 + 1 entries over at least n / V lanes)
template <int V> constexpr int mix_half() { return (V + 1) / 2 + 1; }

struct MixStage {
  int32_t r;    // radix
  int32_t nr;   // n / r: butterflies of a line
  int32_t L;    // product of the radices before
  int32_t ts;   // n / (L r): twiddle-table step
  // LDS index of position p in the exchange after a stage: p + pad (p / (L r)).
  // Both sides of the exchange walk it with one constant step, as the next
  // stage's n / r is a multiple of L r.
  int32_t out_group;  // L r + pad: groups of the stage's outputs
  int32_t in_pad;     // pad of the exchange before
  int32_t in_step;    // (nr + nr / L * in_pad) * ps: from input j to j + 1
  FastDiv dL;
};

struct MixPlan {
  int32_t nst;
  int32_t T;         // lanes per line
  int32_t log2B;     // lanes across lines: B = 1 << log2B lines per block
  int32_t ps, bs;    // LDS strides (reals) of a position and of a line
  FastDiv dT;
  MixStage st[kMixStages];
};

// ---------------------------------------------------------------------------
// Butterflies beyond 2, 3, 4 and 5 (exponent -2 pi i jk / r).
// ---------------------------------------------------------------------------
template <int r> struct Roots;  // c[k] = cos(2 pi k / r), s[k] = sin(2 pi k / r), k <= r / 2; cl, sl: see Wide
template <> struct Roots<7> {
  static constexpr double c[4] = {1.0, 0.623489801858733530525, -0.222520933956314404289, -0.900968867902419126236};
  static constexpr double cl[4] = {0.0, 4.716100e-17, -1.141249e-17, 1.976265e-17};
  static constexpr double s[4] = {0.0, 0.781831482468029808708, 0.974927912181823607018, 0.433883739117558120475};
  static constexpr double sl[4] = {0.0, 5.074320e-18, -1.232384e-17, 7.407189e-20};
};
template <> struct Roots<9> {
  static constexpr double c[5] = {1.0, 0.766044443118978035202, 0.173648177666930348852, -0.5,
                                  -0.939692620785908384054};
  static constexpr double cl[5] = {0.0, 2.175071e-17, -1.009049e-17, 0.0, 4.385093e-17};
  static constexpr double s[5] = {0.0, 0.642787609686539326323, 0.984807753012208059367, 0.866025403784438646764,
                                  0.342020143325668733044};
  static constexpr double sl[5] = {0.0, -3.659608e-17, 3.905109e-17, 5.017542e-17, 2.013602e-17};
};
template <> struct Roots<11> {
  static constexpr double c[6] = {1.0, 0.841253532831181168862, 0.415415013001886425529, -0.142314838273285140443,
                                  -0.654860733945285064056, -0.959492973614497389891};
  static constexpr double cl[6] = {0.0, -3.664729e-17, -9.555212e-18, 3.133448e-18, 3.655315e-17, -2.123968e-17};
  static constexpr double s[6] = {0.0, 0.540640817455597582108, 0.909631995354518371412, 0.989821441880932732376,
                                  0.755749574354258283774, 0.281732556841429697711};
  static constexpr double sl[6] = {0.0, 2.667779e-17, 4.130148e-17, 4.815530e-17, 1.486952e-17, 2.667630e-17};
};
template <> struct Roots<13> {
  static constexpr double c[7] = {1.0, 0.885456025653209895900, 0.568064746731155775490, 0.12053668025532305335,
                                  -0.354604887042535625970, -0.748510748171101098635, -0.970941817426052027156};
  static constexpr double cl[7] = {0.0, -1.460830e-17, -9.353414e-18, 5.709930e-18, -4.547648e-18, -1.735159e-17,
                                   -1.536013e-17};
  static constexpr double s[7] = {0.0, 0.464723172043768546302, 0.82298386589365639458, 0.992708874098054009100,
                                  0.935016242685414832420, 0.663122658240795206160, 0.23931566428755776715};
  static constexpr double sl[7] = {0.0, -1.637795e-17, 4.233793e-17, 2.007753e-17, -9.984533e-18, 9.324777e-18,
                                   4.947072e-19};
};
template <> struct Roots<16> {
  static constexpr double c[10] = {1.0, 0.923879532511286756128, 0.707106781186547524401, 0.382683432365089771728,
                                   0.0, -0.382683432365089771728, -0.707106781186547524401, -0.923879532511286756128,
                                   -1.0, -0.923879532511286756128};
  static constexpr double s[10] = {0.0, 0.382683432365089771728, 0.707106781186547524401, 0.923879532511286756128,
                                   1.0, 0.923879532511286756128, 0.707106781186547524401, 0.382683432365089771728,
                                   0.0, -0.382683432365089771728};
};
// cos and sin(2 pi k / r), 0 <= k < r
template <int r, typename R> __device__ __forceinline__ constexpr Wide<R> root_cos(int k) {
  const int m = 2 * k <= r ? k : r - k;
  return wide<R>(Roots<r>::c[m], Roots<r>::cl[m]);
}
template <int r, typename R> __device__ __forceinline__ constexpr Wide<R> root_sin(int k) {
  const int m = 2 * k <= r ? k : r - k;
  const Wide<R> w = wide<R>(Roots<r>::s[m], Roots<r>::sl[m]);
  return 2 * k <= r ? w : Wide<R>{-w.high, -w.low};
}

// term m (1 <= m <= r / 2) with the i-th smallest factor (sine or cosine) in
// output k: added in this order, a sum's partial sums and with them its
// rounding errors are smallest
template <int r> constexpr int root_order(int k, int i, bool sine) {
  auto size = [=](int m) {
    const int q = k * m % r, t = 2 * q <= r ? q : r - q;
    const double v = sine ? Roots<r>::s[t] : Roots<r>::c[t];
    return v < 0.0 ? -v : v;
  };
  for (int m = 1; 2 * m < r; ++m) {
    int below = 0;
    for (int o = 1; 2 * o < r; ++o) below += size(o) < size(m) || (size(o) == size(m) && o < m) ? 1 : 0;
    if (below == i) return m;
  }
  return 0;
}

// odd radix: the terms m and r - m share their cosine and sine products.  For 9
// too: as 3 x 3 it takes a third less arithmetic, but the twiddles between the
// two add to the error (729 points FP64 2.2e-16, this way 2.0e-16).
template <int r, typename C> __device__ __forceinline__ void bfly_odd(C* a) {
  using R = decltype(a[0].x);
  constexpr int h = (r - 1) / 2;
  C s[h], d[h];
  C sum = a[0];
#pragma unroll
  for (int m = 0; m < h; ++m) {
    s[m] = cadd(a[m + 1], a[r - 1 - m]);
    d[m] = csub(a[m + 1], a[r - 1 - m]);
    sum = cadd(sum, s[m]);
  }
  const C a0 = a[0];
  a[0] = sum;
#pragma unroll
  for (int k = 1; k <= h; ++k) {
    C A = a0, B{R(0), R(0)};
#pragma unroll
    for (int i = 0; i < h; ++i) {
      const int mc = root_order<r>(k, i, false), ms = root_order<r>(k, i, true);
      const Wide<R> c = root_cos<r, R>(k * mc % r), sn = root_sin<r, R>(k * ms % r);
      const C x = s[mc - 1], y = d[ms - 1];
      A = C{add_wide(A.x, c, x.x), add_wide(A.y, c, x.y)};
      B = i == 0 ? C{mul_wide(sn, y.x), mul_wide(sn, y.y)} : C{add_wide(B.x, sn, y.x), add_wide(B.y, sn, y.y)};
    }
    const C t = cmul_mi(B);
    a[k] = cadd(A, t);
    a[r - k] = csub(A, t);
  }
}

// 8 points as 2 x 4, the two outputs of an odd position by fused products with
// 1/sqrt(2)
template <typename C> __device__ __forceinline__ void bfly8_wide(C* a) {
  using R = decltype(a[0].x);
  constexpr Wide<R> h = wide<R>(0.70710678118654752440, -4.833647e-17);
  C e[4] = {a[0], a[2], a[4], a[6]};
  C o[4] = {a[1], a[3], a[5], a[7]};
  bfly4(e);
  bfly4(o);
  // o[k] *= exp(-2 pi i k / 8), but for h
  const C o1 = C{o[1].x + o[1].y, o[1].y - o[1].x};
  const C o2 = cmul_mi(o[2]);
  const C o3 = C{o[3].y - o[3].x, -(o[3].x + o[3].y)};
  a[0] = cadd(e[0], o[0]);
  a[4] = csub(e[0], o[0]);
  a[1] = C{add_wide(e[1].x, h, o1.x), add_wide(e[1].y, h, o1.y)};
  a[5] = C{sub_wide(e[1].x, h, o1.x), sub_wide(e[1].y, h, o1.y)};
  a[2] = cadd(e[2], o2);
  a[6] = csub(e[2], o2);
  a[3] = C{add_wide(e[3].x, h, o3.x), add_wide(e[3].y, h, o3.y)};
  a[7] = C{sub_wide(e[3].x, h, o3.x), sub_wide(e[3].y, h, o3.y)};
}

// 16 = 4 x 4: sub-transforms of the inputs 4 i + j, a twiddle, 4 across
template <typename C> __device__ __forceinline__ void bfly16(C* a) {
  using R = decltype(a[0].x);
  C g[4][4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
#pragma unroll
    for (int i = 0; i < 4; ++i) g[j][i] = a[4 * i + j];
    bfly4(g[j]);
#pragma unroll
    for (int k = 1; k < 4; ++k) {
      if (j > 0) {
        const R c = static_cast<R>(Roots<16>::c[j * k]), s = static_cast<R>(Roots<16>::s[j * k]);
        const C x = g[j][k];
        g[j][k] = C{x.x * c + x.y * s, x.y * c - x.x * s};
      }
    }
  }
#pragma unroll
  for (int k1 = 0; k1 < 4; ++k1) {
    C t[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) t[j] = g[j][k1];
    bfly4(t);
#pragma unroll
    for (int k2 = 0; k2 < 4; ++k2) a[k1 + 4 * k2] = t[k2];
  }
}

template <int r, typename C> __device__ __forceinline__ void mix_bfly(C* a) {
  if constexpr (r == 8) bfly8_wide(a);
  else if constexpr (r == 16) bfly16(a);
  else if constexpr (r == 7 || r == 9 || r == 11 || r == 13) bfly_odd<r>(a);
  else bfly<r>(a);
}

// Twiddle-table entries a butterfly loads: FP64 all its powers (products of w,
// w^4 and w^8 left the error of a 504-point line 21 % larger), FP32 w alone,
// whose powers are FP64 products.
template <int r, typename Real> constexpr int mix_ntw() { return sizeof(Real) == 8 ? r - 1 : 1; }

// v[j] *= w^j
template <int r, typename C> __device__ __forceinline__ void mix_twiddle(C* v, const double2* ww) {
  if constexpr (sizeof(C) == 16) {
#pragma unroll
    for (int j = 1; j < r; ++j) v[j] = cmul(v[j], ww[j - 1]);
  } else {
    // each power is rounded once to FP32 and used before the next is formed
    const double2 w = ww[0];
    double2 lo[4];
    lo[1] = w;
    if constexpr (r > 2) lo[2] = cmul(w, w);
    if constexpr (r > 3) lo[3] = cmul(lo[2], w);
#pragma unroll
    for (int j = 1; j < 4 && j < r; ++j) v[j] = cmul(v[j], to_prec<C>(lo[j]));
    if constexpr (r > 4) {
      const double2 w4 = cmul(lo[2], lo[2]);
      double2 hi = w4;
#pragma unroll
      for (int g = 4; g < r; g += 4) {
        v[g] = cmul(v[g], to_prec<C>(hi));
#pragma unroll
        for (int j = 1; j < 4; ++j)
          if (g + j < r) v[g + j] = cmul(v[g + j], to_prec<C>(cmul(hi, lo[j])));
        if (g + 4 < r) hi = cmul(hi, w4);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Stage pieces.  Lane t of a line carries butterflies beta = t + q T of a
// stage (q < mix_nb<V>(r)); its inputs are positions beta + j nr, its outputs
// (beta / L) L r + beta % L + j L.
// ---------------------------------------------------------------------------
// Real or imaginary halves of the values of one lane through the line's LDS
// positions (the exchanges always travel in two halves: half the LDS per
// line, so two blocks of long lines stay resident on a CU)
template <int r, int V, typename Real>
__device__ __forceinline__ void mix_gather(Real* v, const MixStage& st, int t, int T, const Real* lds, int ps) {
#pragma unroll
  for (int q = 0; q < mix_nb<V>(r); ++q) {
    const int beta = t + q * T;
    if (beta < st.nr) {
      const int g = static_cast<int>(st.dL.div(static_cast<uint32_t>(beta)));
      const Real* src = lds + (beta + g * st.in_pad) * ps;
#pragma unroll
      for (int j = 0; j < r; ++j) v[q * r + j] = src[j * st.in_step];
    }
  }
}
template <int r, int V, typename Real>
__device__ __forceinline__ void mix_scatter(const Real* v, const MixStage& st, int t, int T, Real* lds, int ps) {
  const int step = st.L * ps;
#pragma unroll
  for (int q = 0; q < mix_nb<V>(r); ++q) {
    const int beta = t + q * T;
    if (beta < st.nr) {
      const int g = static_cast<int>(st.dL.div(static_cast<uint32_t>(beta)));
      Real* dst = lds + (beta + g * (st.out_group - st.L)) * ps;
#pragma unroll
      for (int j = 0; j < r; ++j) dst[j * step] = v[q * r + j];
    }
  }
}
// twiddle-table entries of butterfly beta of a stage
template <int r, typename Real>
__device__ __forceinline__ void mix_tw_entries(double2* w, const MixStage& st, int beta, const double2* tw) {
  const int g = static_cast<int>(st.dL.div(static_cast<uint32_t>(beta)));
  const int e = (beta - g * st.L) * st.ts;
#pragma unroll
  for (int i = 0; i < mix_ntw<r, Real>(); ++i) w[i] = twiddle_load(tw + (i + 1) * e);
}
// FP32: those of the lane's butterflies, ahead of the stage.  FP64 has r - 1 of
// each, too many to hold beside the values: mix_compute loads them.
template <int r, int V, typename Real>
__device__ __forceinline__ void mix_tw_load(double2* w, const MixStage& st, int t, int T, const double2* tw) {
  if constexpr (sizeof(Real) == 4) {
#pragma unroll
    for (int q = 0; q < mix_nb<V>(r); ++q)
      if (t + q * T < st.nr) mix_tw_entries<r, Real>(w + q, st, t + q * T, tw);
  }
}
template <int r, int V, typename Real>
__device__ __forceinline__ void mix_compute(Real* re, Real* im, const MixStage& st, int t, int T, const double2* w,
                                            const double2* tw) {
  using C = cplx_t<Real>;
#pragma unroll
  for (int q = 0; q < mix_nb<V>(r); ++q) {
    if (t + q * T < st.nr) {
      C a[r];
#pragma unroll
      for (int j = 0; j < r; ++j) a[j] = C{re[q * r + j], im[q * r + j]};
      if (st.L > 1) {
        if constexpr (sizeof(Real) == 4) {
          mix_twiddle<r>(a, w + q);
        } else {
          double2 all[mix_ntw<r, Real>()];
          mix_tw_entries<r, Real>(all, st, t + q * T, tw);
          mix_twiddle<r>(a, all);
        }
      }
      mix_bfly<r>(a);
#pragma unroll
      for (int j = 0; j < r; ++j) {
        re[q * r + j] = a[j].x;
        im[q * r + j] = a[j].y;
      }
    }
  }
}

// the radix of a stage is uniform over the launch: a scalar branch
#define DFFT_MIX_SWITCH(radix, CALL) \
  switch (radix) {                   \
    case 2: if constexpr (mix_has<V>(2)) { CALL(2); } break; \
    case 3: if constexpr (mix_has<V>(3)) { CALL(3); } break; \
    case 4: if constexpr (mix_has<V>(4)) { CALL(4); } break; \
    case 5: if constexpr (mix_has<V>(5)) { CALL(5); } break; \
    case 6: if constexpr (mix_has<V>(6)) { CALL(6); } break; \
    case 7: if constexpr (mix_has<V>(7)) { CALL(7); } break; \
    case 8: if constexpr (mix_has<V>(8)) { CALL(8); } break; \
    case 9: if constexpr (mix_has<V>(9)) { CALL(9); } break; \
    case 10: if constexpr (mix_has<V>(10)) { CALL(10); } break; \
    case 11: if constexpr (mix_has<V>(11)) { CALL(11); } break; \
    case 12: if constexpr (mix_has<V>(12)) { CALL(12); } break; \
    case 13: if constexpr (mix_has<V>(13)) { CALL(13); } break; \
    case 15: if constexpr (mix_has<V>(15)) { CALL(15); } break; \
    case 16: if constexpr (mix_has<V>(16)) { CALL(16); } break; \
    default: break;                  \
  }

// global loads of the first stage / stores of the last one
template <int r, int V, bool NT, typename Real>
__device__ __forceinline__ void mix_load_c2c(Real* re, Real* im, const MixStage& st, int t, int T, const char* ib,
                                             int64_t is, bool inverse) {
  using C = cplx_t<Real>;
#pragma unroll
  for (int q = 0; q < mix_nb<V>(r); ++q) {
    const int beta = t + q * T;
    if (beta < st.nr) {
      const C* src = reinterpret_cast<const C*>(ib) + beta * is;
      const int64_t step = st.nr * is;
      C x[r];
#pragma unroll
      for (int j = 0; j < r; ++j) {
        x[j] = gload_c<NT, Real>(src);
        src += step;
      }
#pragma unroll
      for (int j = 0; j < r; ++j) {
        re[q * r + j] = x[j].x;
        im[q * r + j] = inverse ? -x[j].y : x[j].y;
      }
    }
  }
}
template <int r, int V, bool NT, typename Real>
__device__ __forceinline__ void mix_load_real(Real* v, const MixStage& st, int t, int T, const char* ib, int64_t is) {
#pragma unroll
  for (int q = 0; q < mix_nb<V>(r); ++q) {
    const int beta = t + q * T;
    if (beta < st.nr) {
      const Real* src = reinterpret_cast<const Real*>(ib) + beta * is;
      const int64_t step = st.nr * is;
#pragma unroll
      for (int j = 0; j < r; ++j) {
        v[q * r + j] = gload<NT>(src);
        src += step;
      }
    }
  }
}
template <int r, int V, bool NT, typename Real>
__device__ __forceinline__ void mix_store_c2c(const Real* re, const Real* im, const MixStage& st, int t, int T,
                                              char* ob, int64_t os, Real sx, Real sy) {
  using C = cplx_t<Real>;
#pragma unroll
  for (int q = 0; q < mix_nb<V>(r); ++q) {
    const int beta = t + q * T;
    if (beta < st.nr) {
      C* dst = reinterpret_cast<C*>(ob) + beta * os;
      const int64_t step = st.nr * os;
#pragma unroll
      for (int j = 0; j < r; ++j) {
        gstore_c<NT, Real>(dst, C{re[q * r + j] * sx, im[q * r + j] * sy});
        dst += step;
      }
    }
  }
}
// the outputs at positions up to n/2 (R2C)
template <int r, int V, bool NT, typename Real>
__device__ __forceinline__ void mix_store_half(const Real* re, const Real* im, const MixStage& st, int t, int T, int n,
                                               const LineIO<Real, NT>& io) {
  using C = cplx_t<Real>;
  const Real hw = io.scale * io.hw;
#pragma unroll
  for (int q = 0; q < mix_nb<V>(r); ++q) {
    const int beta = t + q * T;
    if (beta < st.nr) {
      C* dst = reinterpret_cast<C*>(io.ob) + beta * io.os;
      const int64_t step = st.nr * io.os;
#pragma unroll
      for (int j = 0; j <= r / 2; ++j) {
        const int at = beta + j * st.nr;
        const Real h = at == 0 || 2 * at == n ? io.scale : hw;
        if (2 * at <= n) gstore_c<NT, Real>(dst, C{re[q * r + j] * h, im[q * r + j] * h});
        dst += step;
      }
    }
  }
}
template <int r, int V, bool NT, typename Real>
__device__ __forceinline__ void mix_store_real(const Real* v, const MixStage& st, int t, int T, char* ob, int64_t os,
                                               Real s) {
#pragma unroll
  for (int q = 0; q < mix_nb<V>(r); ++q) {
    const int beta = t + q * T;
    if (beta < st.nr) {
      Real* dst = reinterpret_cast<Real*>(ob) + beta * os;
      const int64_t step = st.nr * os;
#pragma unroll
      for (int j = 0; j < r; ++j) {
        gstore<NT>(dst, v[q * r + j] * s);
        dst += step;
      }
    }
  }
}

// All radix stages of a line whose stage-0 inputs are in registers; leaves
// the outputs of the last stage there.
template <int V, typename Real>
__device__ __forceinline__ void mix_stages(Real* re, Real* im, const MixPlan& m, int t, Real* lds, const double2* tw) {
  double2 w[mix_nb_max<V>()];
  for (int s = 0;; ++s) {
    const MixStage& st = m.st[s];
#define DFFT_MIX_CALL(r) mix_compute<r, V, Real>(re, im, st, t, m.T, w, tw)
    DFFT_MIX_SWITCH(st.r, DFFT_MIX_CALL)
#undef DFFT_MIX_CALL
    if (s + 1 >= m.nst) break;
    const MixStage& nx = m.st[s + 1];
    __syncthreads();
#define DFFT_MIX_CALL(r) mix_scatter<r, V, Real>(re, st, t, m.T, lds, m.ps)
    DFFT_MIX_SWITCH(st.r, DFFT_MIX_CALL)
#undef DFFT_MIX_CALL
    __syncthreads();
    // the next stage's twiddles are on their way during the second half
#define DFFT_MIX_CALL(r)                             \
  mix_tw_load<r, V, Real>(w, nx, t, m.T, tw);                 \
  mix_gather<r, V, Real>(re, nx, t, m.T, lds, m.ps)
    DFFT_MIX_SWITCH(nx.r, DFFT_MIX_CALL)
#undef DFFT_MIX_CALL
    __syncthreads();
#define DFFT_MIX_CALL(r) mix_scatter<r, V, Real>(im, st, t, m.T, lds, m.ps)
    DFFT_MIX_SWITCH(st.r, DFFT_MIX_CALL)
#undef DFFT_MIX_CALL
    __syncthreads();
#define DFFT_MIX_CALL(r) mix_gather<r, V, Real>(im, nx, t, m.T, lds, m.ps)
    DFFT_MIX_SWITCH(nx.r, DFFT_MIX_CALL)
#undef DFFT_MIX_CALL
  }
}

// One line per T lanes; real lines run one by one (why: fft_smooth).
template <typename Real, int V, bool NT, int KIND>
__global__ void __launch_bounds__(1024) fft_mixed(const FastPass p, const MixPlan m) {
  using C = cplx_t<Real>;
  extern __shared__ unsigned char smem_raw[];
  const int tid = threadIdx.x;
  const int B = p.lines_per_block, T = m.T, n = p.n;
  int b, t;
  if (p.lines_fast) {
    b = tid & (B - 1);
    t = tid >> m.log2B;
  } else {
    b = static_cast<int>(m.dT.div(static_cast<uint32_t>(tid)));
    t = tid - b * T;
  }
  // lanes beyond the block's lines hold no butterfly (beta < nr never holds)
  // and touch neither LDS nor global memory; they reach every barrier
  const bool active = tid < B * T;
  if (!active) {
    b = 0;
    t = 1 << 28;
  }
  Real* lds = reinterpret_cast<Real*>(smem_raw) + b * m.bs;
  const double2* tw = reinterpret_cast<const double2*>(p.tw);
  const int32_t unit = pass_block(p, blockIdx.x, gridDim.x) * B + b;
  const MixStage& s0 = m.st[0];
  const MixStage& sl = m.st[m.nst - 1];
  Real re[V], im[V];
#pragma unroll
  for (int j = 0; j < V; ++j) {
    re[j] = Real(0);
    im[j] = Real(0);
  }

  LineIO<Real, NT> io{};
  bool valid = active && unit < p.nlines;
  if (valid) valid = make_line_io<Real, NT>(p, unit, io);
  if constexpr (KIND == kC2C) {
    if (valid) {
#define DFFT_MIX_CALL(r) mix_load_c2c<r, V, NT, Real>(re, im, s0, t, T, io.ib, io.is, p.inverse != 0)
      DFFT_MIX_SWITCH(s0.r, DFFT_MIX_CALL)
#undef DFFT_MIX_CALL
    }
    mix_stages<V, Real>(re, im, m, t, lds, tw);
    if (valid) {
      const Real sy = p.inverse ? -io.scale : io.scale;
#define DFFT_MIX_CALL(r) mix_store_c2c<r, V, NT, Real>(re, im, sl, t, T, io.ob, io.os, io.scale, sy)
      DFFT_MIX_SWITCH(sl.r, DFFT_MIX_CALL)
#undef DFFT_MIX_CALL
    }
  } else if constexpr (KIND == kR2C) {
    if (valid) {
#define DFFT_MIX_CALL(r) mix_load_real<r, V, NT, Real>(re, s0, t, T, io.ib, io.is)
      DFFT_MIX_SWITCH(s0.r, DFFT_MIX_CALL)
#undef DFFT_MIX_CALL
    }
    mix_stages<V, Real>(re, im, m, t, lds, tw);
    if (valid) {
#define DFFT_MIX_CALL(r) mix_store_half<r, V, NT, Real>(re, im, sl, t, T, n, io)
      DFFT_MIX_SWITCH(sl.r, DFFT_MIX_CALL)
#undef DFFT_MIX_CALL
    }
  } else {
    // C2R: the lane that loads entry k <= n/2 of the half spectrum hands its
    // conjugate out through LDS as the input at k and the entry as that at n - k
    C x[mix_half<V>()];
#pragma unroll
    for (int q = 0; q < mix_half<V>(); ++q) {
      const int k = t + q * T;
      x[q] = C{Real(0), Real(0)};
      if (valid && 2 * k <= n) x[q] = gload_c<NT, Real>(reinterpret_cast<const C*>(io.ib) + static_cast<int64_t>(k) * io.is);
    }
#pragma unroll
    for (int q = 0; q < mix_half<V>(); ++q) {
      const int k = t + q * T;
      const bool self = k == 0 || 2 * k == n;
      x[q].x *= self ? Real(1) : io.hw;
      x[q].y = self ? Real(0) : x[q].y * io.hw;
      if (2 * k <= n) {
        lds[k * m.ps] = x[q].x;
        if (k > 0 && 2 * k < n) lds[(n - k) * m.ps] = x[q].x;
      }
    }
    __syncthreads();
#define DFFT_MIX_CALL(r) mix_gather<r, V, Real>(re, s0, t, T, lds, m.ps)
    DFFT_MIX_SWITCH(s0.r, DFFT_MIX_CALL)
#undef DFFT_MIX_CALL
    __syncthreads();
#pragma unroll
    for (int q = 0; q < mix_half<V>(); ++q) {
      const int k = t + q * T;
      if (2 * k <= n) {
        lds[k * m.ps] = -x[q].y;
        if (k > 0 && 2 * k < n) lds[(n - k) * m.ps] = x[q].y;
      }
    }
    __syncthreads();
#define DFFT_MIX_CALL(r) mix_gather<r, V, Real>(im, s0, t, T, lds, m.ps)
    DFFT_MIX_SWITCH(s0.r, DFFT_MIX_CALL)
#undef DFFT_MIX_CALL
    mix_stages<V, Real>(re, im, m, t, lds, tw);
    if (valid) {
#define DFFT_MIX_CALL(r) mix_store_real<r, V, NT, Real>(re, sl, t, T, io.ob, io.os, io.scale)
      DFFT_MIX_SWITCH(sl.r, DFFT_MIX_CALL)
#undef DFFT_MIX_CALL
    }
  }
}

#undef DFFT_MIX_SWITCH

}  // namespace dfft
