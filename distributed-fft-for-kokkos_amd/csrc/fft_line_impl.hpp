// Templates of the compile-time-length line-pass kernels and their
// launchers, shared by the translation units that instantiate them (one per
// precision and range of lengths, compiled in parallel).
//
// FFT conventions (the ones kokkos-fft exposes to the reference plans,
// KokkosFFT_Distributed_SlabPlan.hpp:978-1081): forward X[k] = sum_j x[j]
// exp(-2 pi i jk/n), backward with +i, both unscaled; scaling is applied by
// the caller-supplied factor at the final store.  Inverse transforms run the
// forward kernel between two conjugations (IDFT(x) = conj(DFT(conj(x)))).
#pragma once

#include <hip/hip_runtime.h>

#include "fft_kernels.hpp"

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <mutex>
#include <type_traits>

namespace dfft {

// ---------------------------------------------------------------------------
// Radix plans of the compile-time kernels.
// ---------------------------------------------------------------------------
struct FPlan {
  int R = 1;    // complex values each thread keeps in registers
  int nst = 0;  // number of stages
  int rad[12] = {};
  bool ok = true;
};

constexpr int cgcd(int a, int b) { return b == 0 ? a : cgcd(b, a % b); }

// Power-of-two stages first, then 3s and 5s, the first of them together with a
// single 2 left over as a radix 6 or 10 (96 = 4*4*6, 160 = 4*4*10: an exchange
// less than 4*4*2*5 at the same values per thread).  R (values per thread) is
// the least common multiple of the radices, doubled while below `rmin` and
// still a divisor of n.  With an odd factor the power-of-two part uses radix 4
// (not 8) so R stays small: 160 holds 20 values per thread, not 40.
constexpr FPlan make_plan(int n, int rmin = 1) {
  FPlan p;
  if (n <= 1) return p;
  int m = n;
  int odd = n;
  while (odd % 2 == 0) odd /= 2;
  if (odd == 1) {
    while (m % 8 == 0) { p.rad[p.nst++] = 8; m /= 8; }
  }
  while (m % 4 == 0) { p.rad[p.nst++] = 4; m /= 4; }
  if (m % 6 == 0) { p.rad[p.nst++] = 6; m /= 6; }
  else if (m % 10 == 0) { p.rad[p.nst++] = 10; m /= 10; }
  else if (m % 2 == 0) { p.rad[p.nst++] = 2; m /= 2; }
  while (m % 3 == 0) { p.rad[p.nst++] = 3; m /= 3; }
  while (m % 5 == 0) { p.rad[p.nst++] = 5; m /= 5; }
  p.ok = (m == 1);
  int R = 1;
  for (int s = 0; s < p.nst; ++s) R = R / cgcd(R, p.rad[s]) * p.rad[s];
  while (R < rmin && n % (2 * R) == 0) R *= 2;
  p.R = R;
  return p;
}

constexpr int span_before(int n, int s) {
  FPlan p = make_plan(n);
  int L = 1;
  for (int i = 0; i < s; ++i) L *= p.rad[i];
  return L;
}

// ---------------------------------------------------------------------------
// Forward DFT butterflies on registers (exponent -2 pi i jk/r).
// ---------------------------------------------------------------------------
template <typename C> __device__ __forceinline__ void bfly2(C* a) {
  C t = a[0];
  a[0] = cadd(t, a[1]);
  a[1] = csub(t, a[1]);
}

template <typename C> __device__ __forceinline__ void bfly4(C* a) {
  C t0 = cadd(a[0], a[2]), t1 = csub(a[0], a[2]);
  C t2 = cadd(a[1], a[3]), t3 = cmul_mi(csub(a[1], a[3]));
  a[0] = cadd(t0, t2);
  a[2] = csub(t0, t2);
  a[1] = cadd(t1, t3);
  a[3] = csub(t1, t3);
}

template <typename C> __device__ __forceinline__ void bfly8(C* a) {
  using R = decltype(a[0].x);
  const R h = static_cast<R>(0.70710678118654752440);  // 1/sqrt(2)
  C e[4] = {a[0], a[2], a[4], a[6]};
  C o[4] = {a[1], a[3], a[5], a[7]};
  bfly4(e);
  bfly4(o);
  // o[k] *= exp(-2 pi i k / 8)
  C o1 = C{h * (o[1].x + o[1].y), h * (o[1].y - o[1].x)};
  C o2 = cmul_mi(o[2]);
  C o3 = C{h * (o[3].y - o[3].x), -h * (o[3].x + o[3].y)};
  a[0] = cadd(e[0], o[0]);
  a[4] = csub(e[0], o[0]);
  a[1] = cadd(e[1], o1);
  a[5] = csub(e[1], o1);
  a[2] = cadd(e[2], o2);
  a[6] = csub(e[2], o2);
  a[3] = cadd(e[3], o3);
  a[7] = csub(e[3], o3);
}

__device__ __forceinline__ double fmadd(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fmadd(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// A constant of a butterfly as the rounded value and what the rounding took
// away.  Every line multiplies by the same few constants, so their rounding
// errors add up over the stages instead of averaging out: with sqrt(3)/2 alone
// (off by half an ulp) a 243-point FP64 line was 2.3e-16 off, with its low part
// 1.95e-16.  low is zero where it is less than a seventh of the ulp below one.
template <typename R> struct Wide {
  R high, low;
};
template <typename R> constexpr Wide<R> wide(double high, double low) {
  const R h = static_cast<R>(high);
  const double l = sizeof(R) == 8 ? low : high - static_cast<double>(h);
  const double least = sizeof(R) == 8 ? 1.5e-17 : 8e-9;
  return Wide<R>{h, l < least && l > -least ? R(0) : static_cast<R>(l)};
}
// a + c b and a - c b, the low part of c first
template <typename R> __device__ __forceinline__ R add_wide(R a, const Wide<R>& c, R b) {
  return fmadd(c.high, b, c.low != R(0) ? fmadd(c.low, b, a) : a);
}
template <typename R> __device__ __forceinline__ R sub_wide(R a, const Wide<R>& c, R b) {
  return add_wide(a, Wide<R>{-c.high, -c.low}, b);
}
template <typename R> __device__ __forceinline__ R mul_wide(const Wide<R>& c, R b) {
  return c.low != R(0) ? fmadd(c.low, b, c.high * b) : c.high * b;
}

template <typename C> __device__ __forceinline__ void bfly3(C* a) {
  using R = decltype(a[0].x);
  constexpr Wide<R> s3 = wide<R>(0.86602540378443864676, 5.017542e-17);  // sin(2 pi / 3)
  const C s = cadd(a[1], a[2]);
  const C d = csub(a[1], a[2]);
  const C m = C{fmadd(R(-0.5), s.x, a[0].x), fmadd(R(-0.5), s.y, a[0].y)};
  a[0] = cadd(a[0], s);
  a[1] = C{add_wide(m.x, s3, d.y), sub_wide(m.y, s3, d.x)};
  a[2] = C{sub_wide(m.x, s3, d.y), add_wide(m.y, s3, d.x)};
}

template <typename C> __device__ __forceinline__ void bfly5(C* a) {
  using R = decltype(a[0].x);
  constexpr Wide<R> c1 = wide<R>(0.30901699437494742410, -2.716058e-17);  // cos(2 pi/5)
  constexpr Wide<R> c2 = wide<R>(-0.80901699437494742410, 2.716058e-17);  // cos(4 pi/5)
  constexpr Wide<R> s1 = wide<R>(0.95105651629515357212, 4.093450e-17);   // sin(2 pi/5)
  constexpr Wide<R> s2 = wide<R>(0.58778525229247312917, -7.934751e-18);  // sin(4 pi/5)
  const C b1 = cadd(a[1], a[4]), b2 = cadd(a[2], a[3]);
  const C d1 = csub(a[1], a[4]), d2 = csub(a[2], a[3]);
  // the smaller term of a sum first: its rounding errors are those of the partial sums
  const C A1 = C{add_wide(add_wide(a[0].x, c1, b1.x), c2, b2.x), add_wide(add_wide(a[0].y, c1, b1.y), c2, b2.y)};
  const C A2 = C{add_wide(add_wide(a[0].x, c1, b2.x), c2, b1.x), add_wide(add_wide(a[0].y, c1, b2.y), c2, b1.y)};
  const C X1 = cmul_mi(C{add_wide(mul_wide(s2, d2.x), s1, d1.x), add_wide(mul_wide(s2, d2.y), s1, d1.y)});
  const C X2 = cmul_mi(C{sub_wide(mul_wide(s2, d1.x), s1, d2.x), sub_wide(mul_wide(s2, d1.y), s1, d2.y)});
  a[0] = cadd(cadd(a[0], b1), b2);
  a[1] = cadd(A1, X1);
  a[4] = csub(A1, X1);
  a[2] = cadd(A2, X2);
  a[3] = csub(A2, X2);
}

template <int r, typename C> __device__ __forceinline__ void bfly(C* a);

// r = r1 * r2, coprime: input r2 i + r1 j and output e1 k1 + e2 k2 (mod r)
// with e1 = 1 (mod r1), 0 (mod r2) and e2 the other way round need no
// twiddles between the two dimensions (Good 1958, Thomas 1963)
template <int r1, int r2, typename C> __device__ __forceinline__ void bfly_coprime(C* a) {
  constexpr int r = r1 * r2;
  constexpr int e1 = [] { for (int v = r2;; v += r2) if (v % r1 == 1) return v; }();
  constexpr int e2 = [] { for (int v = r1;; v += r1) if (v % r2 == 1) return v; }();
  C g[r2][r1];
#pragma unroll
  for (int j = 0; j < r2; ++j) {
#pragma unroll
    for (int i = 0; i < r1; ++i) g[j][i] = a[(r2 * i + r1 * j) % r];
    bfly<r1>(g[j]);
  }
#pragma unroll
  for (int k1 = 0; k1 < r1; ++k1) {
    C t[r2];
#pragma unroll
    for (int j = 0; j < r2; ++j) t[j] = g[j][k1];
    bfly<r2>(t);
#pragma unroll
    for (int k2 = 0; k2 < r2; ++k2) a[(e1 * k1 + e2 * k2) % r] = t[k2];
  }
}

template <int r, typename C> __device__ __forceinline__ void bfly(C* a) {
  if constexpr (r == 2) bfly2(a);
  else if constexpr (r == 3) bfly3(a);
  else if constexpr (r == 4) bfly4(a);
  else if constexpr (r == 5) bfly5(a);
  else if constexpr (r == 8) bfly8(a);
  else if constexpr (r == 6) bfly_coprime<2, 3>(a);
  else if constexpr (r == 10) bfly_coprime<2, 5>(a);
  else if constexpr (r == 12) bfly_coprime<4, 3>(a);
  else if constexpr (r == 15) bfly_coprime<3, 5>(a);
}

// ---------------------------------------------------------------------------
// Element access of a line.
// ---------------------------------------------------------------------------
// Global element access: nontemporal (streaming) or cached, chosen at
// compile time (a runtime choice between the two forms of one access is
// folded into the cached form by the compiler).  The pointer is taken as a
// global-memory one: line addresses read from a table in device memory (the
// grouped kernel) are otherwise generic and compile to flat instructions,
// which also count against the LDS wait counter.
template <typename T> using global_ptr = __attribute__((address_space(1))) T*;
template <bool NT, typename T> __device__ __forceinline__ T gload(const T* p) {
  const global_ptr<const T> g = (global_ptr<const T>)p;
  if constexpr (NT) return __builtin_nontemporal_load(g);
  else return *g;
}
template <bool NT, typename T> __device__ __forceinline__ void gstore(T* p, T v) {
  const global_ptr<T> g = (global_ptr<T>)p;
  if constexpr (NT) __builtin_nontemporal_store(v, g);
  else *g = v;
}
template <bool NT, typename Real> __device__ __forceinline__ cplx_t<Real> gload_c(const cplx_t<Real>* p) {
  typedef Real V2 __attribute__((ext_vector_type(2)));
  const V2 t = gload<NT>(reinterpret_cast<const V2*>(p));
  return cplx_t<Real>{t.x, t.y};
}
template <bool NT, typename Real> __device__ __forceinline__ void gstore_c(cplx_t<Real>* p, cplx_t<Real> v) {
  typedef Real V2 __attribute__((ext_vector_type(2)));
  V2 t;
  t.x = v.x;
  t.y = v.y;
  gstore<NT>(reinterpret_cast<V2*>(p), t);
}

template <typename Real, bool NT = false> struct LineIO {
  using C = cplx_t<Real>;
  const char* ib;
  char* ob;
  int64_t is, os;
  int32_t kind, n, inverse;
  Real scale;
  Real hw;  // interior half-spectrum weight (1: none)

  __device__ __forceinline__ C load(int32_t pos) const {
    if (kind == kC2C) return load_kind<kC2C>(pos);
    if (kind == kR2C) return load_kind<kR2C>(pos);
    return load_kind<kC2R>(pos);
  }
  // the same for a kind known at compile time (a loop over positions then
  // has no per-element branch on the kind)
  template <int KIND> __device__ __forceinline__ C load_kind(int32_t pos) const {
    C v;
    if constexpr (KIND == kC2C) {
      v = gload_c<NT, Real>(reinterpret_cast<const C*>(ib) + pos * is);
    } else if constexpr (KIND == kR2C) {
      v = C{gload<NT>(reinterpret_cast<const Real*>(ib) + pos * is), Real(0)};
    } else {
      // the address is selected, not the load: loads under a branch each
      // would be waited for one by one
      const int32_t nh = n / 2 + 1;
      const bool upper = pos >= nh;
      v = gload_c<NT, Real>(reinterpret_cast<const C*>(ib) + (upper ? n - pos : pos) * is);
      if (upper) v = cconj(v);
      if (pos == 0 || 2 * pos == n) {
        v.y = Real(0);
      } else {
        v.x *= hw;
        v.y *= hw;
      }
    }
    return inverse ? cconj(v) : v;
  }
  __device__ __forceinline__ void store(int32_t pos, C v) const {
    if (inverse) v = cconj(v);
    v.x *= scale;
    v.y *= scale;
    if (kind == kC2C) {
      gstore_c<NT, Real>(reinterpret_cast<C*>(ob) + pos * os, v);
    } else if (kind == kR2C) {
      if (pos != 0 && 2 * pos != n) {
        v.x *= hw;
        v.y *= hw;
      }
      if (2 * pos <= n) gstore_c<NT, Real>(reinterpret_cast<C*>(ob) + pos * os, v);
    } else {
      gstore<NT>(reinterpret_cast<Real*>(ob) + pos * os, v.x);
    }
  }
};

// Two real lines a, b per complex line.  R2C: z = a + i b, and after the
// forward FFT Z the spectra are A_k = (Z_k + conj Z_{n-k}) / 2 and
// B_k = (Z_k - conj Z_{n-k}) / (2i).  C2R: Z = A + i B over the Hermitian
// extensions of both half spectra; the inverse transform of Z is a + i b.
template <typename Real, bool NT = false> struct PairIO {
  using C = cplx_t<Real>;
  const char* ib[2];  // products passes: ib[0] = the velocity line this slot stages
  char* ob[2];
  int64_t is[2], os[2];  // per line: the two lines may lie in different rank blocks
  int32_t kind, n;
  Real scale;
  Real hw;     // interior half-spectrum weight (1: none)
  bool has_b;  // the pair's second line exists

  // C2R input at position pos (C2R lines are conjugated: inverse = conj o
  // FFT o conj) from the loaded half-spectrum entries A = X_a[src], Bv =
  // X_b[src], src = pos below n/2+1 (lo) and n - pos above
  __device__ __forceinline__ C c2r_value(int32_t pos, bool lo, C A, C Bv) const {
    if (!lo) {
      A = cconj(A);
      Bv = cconj(Bv);
    }
    if (pos == 0 || 2 * pos == n) {
      A.y = Real(0);
      Bv.y = Real(0);
    } else {
      A.x *= hw;
      A.y *= hw;
      Bv.x *= hw;
      Bv.y *= hw;
    }
    // conj(A + i B)
    return C{A.x - Bv.y, -(A.y + Bv.x)};
  }
};

// Batch indices of a line (slowest axis first).  BAND: a pass over the kept
// modes of a dealiased field only (FastPass::band).
struct BatchIdx {
  int32_t i0, i1, i2;
};
template <bool BAND = false>
__device__ __forceinline__ BatchIdx batch_index(const FastPass& p, int32_t line) {
  const uint32_t l = static_cast<uint32_t>(line + p.line_begin);
  const uint32_t q2 = p.div[2].div(l);
  const uint32_t q1 = p.div[1].div(q2);
  BatchIdx x;
  x.i2 = static_cast<int32_t>(l - q2 * static_cast<uint32_t>(p.ext[2]));
  x.i1 = static_cast<int32_t>(q2 - q1 * static_cast<uint32_t>(p.ext[1]));
  x.i0 = static_cast<int32_t>(q1);
  if constexpr (BAND) {
    x.i0 += x.i0 > p.band ? p.band_shift[0] : 0;
    x.i1 += x.i1 > p.band ? p.band_shift[1] : 0;
    x.i2 += x.i2 > p.band ? p.band_shift[2] : 0;
  }
  return x;
}

// Address of element 0 of line x on one side of a pass, and the line's
// element stride.  Multi-rank sides: per storage axis, fastest first, the
// owner bin and local index of the index (first rem bins one longer --
// KokkosFFT_Distributed_MPI_Extents.hpp:195-235).  Every choice is a mask or
// an exclusive or with a field: selects between two fields compile to
// per-lane loads of the chosen one, selects on an axis to branches.
__device__ __forceinline__ char* side_line(const Side& s, char* const* tab, const BatchIdx& x, int64_t& line) {
  if (!s.multi) {
    line = s.line;
    return s.ptr + ((x.i0 * s.stride[0] + x.i1 * s.stride[1] + x.i2 * s.stride[2]) << s.shift);
  }
  int64_t acc = 1, off = 0, ls = 0;
  int32_t rank = 0;
#pragma unroll
  for (int k = 0; k < kMaxDim; ++k) {
    const SideAxis& a = s.ax[k];
    const int32_t i = (x.i0 & a.sel0) | (x.i1 & a.sel1) | (x.i2 & a.sel2);
    const int32_t low = i < a.split ? -1 : 0;  // in a rank one longer
    const uint32_t t = static_cast<uint32_t>(i - (a.split & ~low));
    const uint32_t q = (__umulhi(t, a.m_small ^ (a.m_xor & static_cast<uint32_t>(low))) + t) >>
                       (a.l_small ^ (a.l_xor & static_cast<uint32_t>(low)));
    const int32_t len = a.base - low;
    rank += (static_cast<int32_t>(q) + (a.rem & ~low)) * a.rstride;
    ls |= acc & a.line_sel;
    off += (static_cast<int32_t>(t) - static_cast<int32_t>(q) * len) * acc;
    acc *= len | a.line_len;
  }
  line = ls;
  return tab[rank] + (off << s.shift);
}

// The line's addresses; false if it is padding (a pass enumerated over padded
// rows).  PROD (products pass, the field axis the fastest batch axis): product
// fields 0 to 2 read velocity lines 0 to 2; the others' input is not used.
template <typename Real, bool NT = false, bool BAND = false, bool PROD = false>
__device__ __forceinline__ bool make_line_io(const FastPass& p, int32_t line, LineIO<Real, NT>& io) {
  const BatchIdx x = batch_index<BAND>(p, line);
  if (x.i2 >= p.pad_real) return false;
  BatchIdx u = x;
  if constexpr (PROD) u.i2 = x.i2 < 2 ? x.i2 : 2;
  io.ib = side_line(p.in, p.in_ptr, u, io.is);
  io.ob = side_line(p.out, p.out_ptr, x, io.os);
  io.kind = p.kind;
  io.n = p.n;
  io.inverse = p.inverse;
  io.scale = static_cast<Real>(p.scale);
  io.hw = p.herm_weight != 0.0 ? static_cast<Real>(p.herm_weight) : Real(1);
  return true;
}

// true if line `line` is padding
__device__ __forceinline__ bool padding_line(const FastPass& p, int32_t line) {
  const uint32_t l = static_cast<uint32_t>(line + p.line_begin);
  return static_cast<int32_t>(l - p.div[2].div(l) * static_cast<uint32_t>(p.ext[2])) >= p.pad_real;
}

// factors of product field f (0..5) of the divergence-form products
__device__ __forceinline__ int32_t prod_first(int32_t f) { return f < 3 ? 0 : (f < 5 ? 1 : 2); }
__device__ __forceinline__ int32_t prod_second(int32_t f) { return f < 3 ? f : (f < 5 ? f - 2 : 2); }

// PROD (products pass): the field axis is the fastest batch axis, and the
// slot of the pair of fields (f, f + 1) stages velocity line f / 2 of its
// position for the position's three slots.
template <typename Real, bool NT, bool PROD = false, bool BAND = false>
__device__ __forceinline__ PairIO<Real, NT> make_pair_io(const FastPass& p, int32_t pair) {
  PairIO<Real, NT> io;
  const int32_t la = 2 * pair;
  BatchIdx x = batch_index<BAND>(p, la);
  io.ob[0] = side_line(p.out, p.out_ptr, x, io.os[0]);
  if constexpr (PROD) {
    BatchIdx u = x;
    u.i2 >>= 1;
    io.ib[0] = side_line(p.in, p.in_ptr, u, io.is[0]);
  } else {
    io.ib[0] = side_line(p.in, p.in_ptr, x, io.is[0]);
  }
  io.has_b = la + 1 < p.nlines;
  if (io.has_b) {
    x = batch_index<BAND>(p, la + 1);
    if constexpr (PROD) {
      io.ib[1] = io.ib[0];
      io.is[1] = io.is[0];
    } else {
      io.ib[1] = side_line(p.in, p.in_ptr, x, io.is[1]);
    }
    io.ob[1] = side_line(p.out, p.out_ptr, x, io.os[1]);
  } else {
    io.ib[1] = io.ib[0];
    io.ob[1] = io.ob[0];
    io.is[1] = io.is[0];
    io.os[1] = io.os[0];
  }
  io.kind = p.kind;
  io.n = p.n;
  io.scale = static_cast<Real>(p.scale);
  io.hw = p.herm_weight != 0.0 ? static_cast<Real>(p.herm_weight) : Real(1);
  return io;
}

// ---------------------------------------------------------------------------
// Compile-time-length Stockham kernel: each line is processed by T = N/R
// threads holding R values in registers; radix stages exchange through LDS.
// ---------------------------------------------------------------------------
template <typename Real> struct LdsPad;
template <> struct LdsPad<double> { static constexpr int shift = 3; };
template <> struct LdsPad<float> { static constexpr int shift = 4; };

template <typename Real, int N, int RM> struct FastCfg {
  static constexpr FPlan P = make_plan(N, RM);
  static constexpr int R = P.R;
  static constexpr int T = N / R;
  static constexpr int NST = P.nst;
  static constexpr int LDSN = N + (N >> LdsPad<Real>::shift) + 1;
  __device__ static __forceinline__ int lidx(int pos) { return pos + (pos >> LdsPad<Real>::shift); }
};

// Twiddles of a radix-r butterfly are the powers w^j (j = 1..r-1) of one
// table entry w = exp(-2 pi i k / (L r)): one FP64 load, the other powers by
// FP64 products (three multiplications deep, w^9 four), each rounded once to the
// kernel's precision.  FP64 lines of 96 and 160 points read w to w^4 and w^8:
// chains up to w^9, four products deep, left a 160-point line 2.8e-16 off
// instead of 1.7e-16.
template <typename Real, int N> constexpr bool powers_from_table() { return sizeof(Real) == 8 && (N & (N - 1)) != 0; }
template <int r>
__device__ __forceinline__ void twiddle_powers(double2 w, double2* p) {
  p[1] = w;
  if constexpr (r > 2) p[2] = cmul(w, w);
  if constexpr (r > 3) p[3] = cmul(p[2], w);
  if constexpr (r > 4) p[4] = cmul(p[2], p[2]);
  if constexpr (r > 5) p[5] = cmul(p[4], w);
  if constexpr (r > 6) p[6] = cmul(p[3], p[3]);
  if constexpr (r > 7) p[7] = cmul(p[4], p[3]);
  if constexpr (r > 8) p[8] = cmul(p[4], p[4]);
  if constexpr (r > 9) p[9] = cmul(p[5], p[4]);
}

template <typename C> __device__ __forceinline__ C to_prec(double2 w);
template <> __device__ __forceinline__ double2 to_prec<double2>(double2 w) { return w; }
template <> __device__ __forceinline__ float2 to_prec<float2>(double2 w) {
  return float2{static_cast<float>(w.x), static_cast<float>(w.y)};
}

// One twiddle-table entry, read as a native vector from global memory (a
// double2 is a class: copying it through a global pointer would pass a
// generic reference and compile to a flat load).
__device__ __forceinline__ double2 twiddle_load(const double2* p) {
  typedef double D2 __attribute__((ext_vector_type(2)));
  const D2 w = gload<false>(reinterpret_cast<const D2*>(p));
  return double2{w.x, w.y};
}

// The twiddle-table entries radix stage S of lane t multiplies by.  When a
// lane needs at most four (a few registers), they are loaded ahead: the
// stage loop issues them before the LDS exchange that precedes the stage, so
// their latency passes under the exchange's barriers instead of stalling
// every wave of the block right after them.
template <typename Real, int N, int RM, int S> struct StageTwiddles {
  using Cfg = FastCfg<Real, N, RM>;
  static constexpr int r = Cfg::P.rad[S];
  static constexpr int L = span_before(N, S);
  static constexpr int T = Cfg::T;
  static constexpr int NB = Cfg::R / r;
  static constexpr int ts = N / (L * r);
  // butterfly q of lane t is beta = t + q*T and needs entry beta mod L: where L
  // divides T that is the same one for every q
  static constexpr bool kShared = L > 1 && T % L == 0;
  static constexpr bool kAhead = L > 1 && !kShared && NB <= 4;
  // more entries per lane (the last radix-2 stage of 16-value lanes): where T
  // divides L, entry (t + q*T) mod L is entry t times entry q*T mod L, the
  // same for every lane (a scalar load): one entry per lane is loaded ahead
  static constexpr bool kBase = L > 1 && !kShared && NB > 4 && L % T == 0;
  double2 w[kAhead ? NB : 1];
  __device__ __forceinline__ void load(int t, const double2* tw) {
    if constexpr (powers_from_table<Real, N>()) {
      // stage_twiddle loads them
    } else if constexpr (kAhead) {
#pragma unroll
      for (int q = 0; q < NB; ++q) w[q] = twiddle_load(tw + entry(t, q) * ts);
    } else if constexpr (kBase || kShared) {
      w[0] = twiddle_load(tw + entry(t, 0) * ts);
    }
  }
  // (t + q*T) mod L: T divides L or L divides T
  __device__ static __forceinline__ unsigned entry(int t, int q) {
    return T % L == 0 ? static_cast<unsigned>(t) % L : static_cast<unsigned>(t) + q * T % L;
  }
  __device__ __forceinline__ double2 get(int t, const double2* tw, int q) const {
    if constexpr (kAhead) return w[q];
    else if constexpr (kShared) return w[0];
    else if constexpr (kBase) return q * T % L == 0 ? w[0] : cmul(w[0], twiddle_load(tw + (q * T % L) * ts));
    else return twiddle_load(tw + entry(t, q) * ts);
  }
};

// Multiplies the lane's values by the stage's twiddles; `sets` register sets
// of the same positions.  Where every butterfly of the lane has the same
// twiddles each power is formed once and used up before the next (all powers
// held over the lane's butterflies spilled the two-line kernel of 16 values).
template <typename Real, int N, int RM, int S, int SETS>
__device__ __forceinline__ void stage_twiddle(cplx_t<Real>* const (&v)[SETS], int t, const double2* tw,
                                              const StageTwiddles<Real, N, RM, S>& pre) {
  using C = cplx_t<Real>;
  using Tw = StageTwiddles<Real, N, RM, S>;
  constexpr int r = Tw::r, NB = Tw::NB;
  if constexpr (Tw::L > 1) {
    if constexpr (powers_from_table<Real, N>()) {
#pragma unroll
      for (int q = 0; q < NB; ++q) {
        const unsigned e = Tw::entry(t, q) * Tw::ts;
        double2 lo[5], hi;
#pragma unroll
        for (int j = 1; j < 5 && j < r; ++j) lo[j] = twiddle_load(tw + j * e);
        if constexpr (r > 8) hi = twiddle_load(tw + 8 * e);
#pragma unroll
        for (int j = 1; j < r; ++j) {
          const double2 w = j < 5 ? lo[j] : j == 8 ? hi : cmul(j < 8 ? lo[4] : hi, lo[j % 4]);
#pragma unroll
          for (int k = 0; k < SETS; ++k) v[k][q * r + j] = cmul(v[k][q * r + j], w);
        }
      }
    } else if constexpr (Tw::kShared) {
      double2 pw[10];
      twiddle_powers<r>(pre.get(t, tw, 0), pw);
#pragma unroll
      for (int j = 1; j < r; ++j) {
        const C w = to_prec<C>(pw[j]);
#pragma unroll
        for (int q = 0; q < NB; ++q) {
#pragma unroll
          for (int k = 0; k < SETS; ++k) v[k][q * r + j] = cmul(v[k][q * r + j], w);
        }
      }
    } else {
#pragma unroll
      for (int q = 0; q < NB; ++q) {
        double2 pw[10];
        twiddle_powers<r>(pre.get(t, tw, q), pw);
#pragma unroll
        for (int j = 1; j < r; ++j) {
          const C w = to_prec<C>(pw[j]);
#pragma unroll
          for (int k = 0; k < SETS; ++k) v[k][q * r + j] = cmul(v[k][q * r + j], w);
        }
      }
    }
  }
}

template <typename Real, int N, int RM, int S>
__device__ __forceinline__ void stage_compute(cplx_t<Real>* v, int t, const double2* tw,
                                              const StageTwiddles<Real, N, RM, S>& pre) {
  using Cfg = FastCfg<Real, N, RM>;
  constexpr int r = Cfg::P.rad[S];
  cplx_t<Real>* const set[1] = {v};
  stage_twiddle<Real, N, RM, S, 1>(set, t, tw, pre);
#pragma unroll
  for (int q = 0; q < Cfg::R / r; ++q) bfly<r>(v + q * r);
}

// Bytes of one line's LDS buffer: LDSN complex values, or LDSN reals when
// the exchanges travel in two halves (SPLIT).
template <typename Real, int N, int RM, bool SPLIT> constexpr size_t line_lds_bytes() {
  return static_cast<size_t>(FastCfg<Real, N, RM>::LDSN) * (SPLIT ? sizeof(Real) : sizeof(cplx_t<Real>));
}

template <typename Real, int N, int RM> constexpr size_t dual_line_bytes() {
  return static_cast<size_t>(FastCfg<Real, N, RM>::LDSN) * sizeof(Real);
}

// LDS bytes from one line buffer to the next.  A cycle serves 128 bytes, 16
// lanes of 8 or 32 of 4: lanes that access one position of `across`
// neighbouring buffers together should lie 128 / across bytes apart (mod
// `cycle`).  Buffers of n + n/8 + 1 reals alone left 61 % of the LDS cycles of
// a strided 256-point FP64 pass in bank conflicts.  Lines below 256 bytes stay
// as they are.
inline size_t bank_stride(size_t bytes, int elem, int across, int cycle = 128) {
  if (bytes < 256 || across <= 1) return bytes;
  const size_t want = static_cast<size_t>(std::max(elem, 128 / across / elem * elem) % cycle);
  while (bytes % static_cast<size_t>(cycle) != want) bytes += static_cast<size_t>(elem);
  return bytes;
}
// lanes across the lines: B buffers share a position; along them: a line's T
// lanes cover T elements of the 128 bytes
inline size_t line_stride(size_t bytes, int elem, bool lanes_across, int B, int T) {
  return bank_stride(bytes, elem, lanes_across ? B : 128 / std::min(128, T * elem));
}
// two lines per lane: neighbouring lanes access every second buffer
inline size_t dual_stride(size_t bytes, int B) { return bank_stride(bytes, 4, B, 64); }

// LDS positions of the exchange after stage S.  Lane t writes the outputs of
// its butterflies t + q*T, (beta / L) L r + beta % L + j L, and reads the inputs
// t + q*T + j*(N/r2) of stage S + 1.  T divides L or L divides T, so each is a
// position of the lane plus a constant of (q, j), and the padding of the two
// adds up (the constant never carries into the lane's part): one index per
// lane and immediate offsets.
template <typename Real, int N, int RM, int S> struct Exchange {
  using Cfg = FastCfg<Real, N, RM>;
  static constexpr int R = Cfg::R, T = Cfg::T;
  static constexpr int r = Cfg::P.rad[S], L = span_before(N, S), NB = R / r;
  static constexpr int r2 = Cfg::P.rad[S + 1], NB2 = R / r2;
  static_assert(T % L == 0 || L % T == 0, "butterflies of a lane");
  static constexpr int padded(int c) { return c + (c >> LdsPad<Real>::shift); }
  __device__ static __forceinline__ int write_base(unsigned t) {
    return Cfg::lidx(static_cast<int>(T % L == 0 ? t / L * (L * r) + t % L : t));
  }
  static constexpr int write_at(int q, int j) {
    return padded((T % L == 0 ? q * T * r : q * T / L * (L * r) + q * T % L) + j * L);
  }
  __device__ static __forceinline__ int read_base(unsigned t) { return Cfg::lidx(static_cast<int>(t)); }
  static constexpr int read_at(int q, int j) { return padded(q * T + j * (N / r2)); }
};

// Write the outputs of stage S, read the inputs of stage S+1.  SPLIT moves the
// real parts first and the imaginary parts second through a buffer of reals:
// after the first half a lane's old real parts are in LDS and can be
// overwritten, its old imaginary parts are still in registers for the second
// half.
template <typename Real, int N, int RM, bool SPLIT, int S>
__device__ __forceinline__ void stage_exchange(cplx_t<Real>* v, int t, void* line) {
  using X = Exchange<Real, N, RM, S>;
  const int wb = X::write_base(static_cast<unsigned>(t)), rb = X::read_base(static_cast<unsigned>(t));
  if constexpr (SPLIT) {
    Real* lw = static_cast<Real*>(line) + wb;
    const Real* lr = static_cast<const Real*>(line) + rb;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      __syncthreads();
#pragma unroll
      for (int q = 0; q < X::NB; ++q) {
#pragma unroll
        for (int j = 0; j < X::r; ++j) lw[X::write_at(q, j)] = h ? v[q * X::r + j].y : v[q * X::r + j].x;
      }
      __syncthreads();
#pragma unroll
      for (int q = 0; q < X::NB2; ++q) {
#pragma unroll
        for (int j = 0; j < X::r2; ++j) {
          const Real x = lr[X::read_at(q, j)];
          if (h) {
            v[q * X::r2 + j].y = x;
          } else {
            v[q * X::r2 + j].x = x;
          }
        }
      }
    }
  } else {
    cplx_t<Real>* lw = static_cast<cplx_t<Real>*>(line) + wb;
    const cplx_t<Real>* lr = static_cast<const cplx_t<Real>*>(line) + rb;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < X::NB; ++q) {
#pragma unroll
      for (int j = 0; j < X::r; ++j) lw[X::write_at(q, j)] = v[q * X::r + j];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < X::NB2; ++q) {
#pragma unroll
      for (int j = 0; j < X::r2; ++j) v[q * X::r2 + j] = lr[X::read_at(q, j)];
    }
  }
}

// After the last stage, of radix rl with NBl butterflies per lane, value
// q*rl + j is output t + q*T + j*(N/rl) = t + (q + j*NBl)*T: reordered, value
// k of lane t is output t + k*T.  (With consecutive butterflies t*NBl + q
// this took one more exchange through LDS, a third of all for 256 points.)
template <typename Real, int N, int RM> __device__ __forceinline__ void final_order(cplx_t<Real>* v) {
  using Cfg = FastCfg<Real, N, RM>;
  constexpr int R = Cfg::R;
  constexpr int rl = Cfg::P.rad[Cfg::NST - 1];
  if constexpr (rl != R) {
    constexpr int NBl = R / rl;
    cplx_t<Real> u[R];
#pragma unroll
    for (int k = 0; k < R; ++k) u[k] = v[(k % NBl) * rl + k / NBl];
#pragma unroll
    for (int k = 0; k < R; ++k) v[k] = u[k];
  }
}

template <typename Real, int N, int RM, bool SPLIT, int S> struct StageLoop {
  __device__ static __forceinline__ void run(cplx_t<Real>* v, int t, const double2* tw, void* line,
                                             const StageTwiddles<Real, N, RM, S>& pre) {
    stage_compute<Real, N, RM, S>(v, t, tw, pre);
    if constexpr (S + 1 < FastCfg<Real, N, RM>::NST) {
      StageTwiddles<Real, N, RM, S + 1> next;
      next.load(t, tw);
      stage_exchange<Real, N, RM, SPLIT, S>(v, t, line);
      StageLoop<Real, N, RM, SPLIT, S + 1>::run(v, t, tw, line, next);
    }
  }
  __device__ static __forceinline__ void run(cplx_t<Real>* v, int t, const double2* tw, void* line) {
    StageTwiddles<Real, N, RM, S> pre;
    pre.load(t, tw);
    run(v, t, tw, line, pre);
  }
};

// ---------------------------------------------------------------------------
// Two lines per lane (FP32 lanes-across-lines passes whose consecutive lines
// are adjacent elements of one row): lane b of a block holds lines 2b and
// 2b+1, one 16-byte access moves element k of both, and the two register
// sets share twiddles and barriers.  B = 32 lines per block reads 256-byte
// row segments with 16 lanes across the lines; the LDS exchanges always move
// real and imaginary halves (2 lines x N + N/16 + 1 floats per lane pair).
// ---------------------------------------------------------------------------
template <typename Real, int N, int RM, int S>
__device__ __forceinline__ void stage_compute2(cplx_t<Real>* va, cplx_t<Real>* vb, int t, const double2* tw,
                                               const StageTwiddles<Real, N, RM, S>& pre) {
  using Cfg = FastCfg<Real, N, RM>;
  constexpr int r = Cfg::P.rad[S];
  cplx_t<Real>* const set[2] = {va, vb};
  stage_twiddle<Real, N, RM, S, 2>(set, t, tw, pre);
#pragma unroll
  for (int q = 0; q < Cfg::R / r; ++q) {
    bfly<r>(va + q * r);
    bfly<r>(vb + q * r);
  }
}

// stage_exchange for the two register sets of a lane (buffers la, lb of reals)
template <typename Real, int N, int RM, int S>
__device__ __forceinline__ void stage_exchange2(cplx_t<Real>* va, cplx_t<Real>* vb, int t, Real* la, Real* lb) {
  using X = Exchange<Real, N, RM, S>;
  const int wb = X::write_base(static_cast<unsigned>(t)), rb = X::read_base(static_cast<unsigned>(t));
  Real *wa = la + wb, *wl = lb + wb;
  const Real *ra = la + rb, *rl = lb + rb;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    __syncthreads();
#pragma unroll
    for (int q = 0; q < X::NB; ++q) {
#pragma unroll
      for (int j = 0; j < X::r; ++j) {
        wa[X::write_at(q, j)] = h ? va[q * X::r + j].y : va[q * X::r + j].x;
        wl[X::write_at(q, j)] = h ? vb[q * X::r + j].y : vb[q * X::r + j].x;
      }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < X::NB2; ++q) {
#pragma unroll
      for (int j = 0; j < X::r2; ++j) {
        const Real xa = ra[X::read_at(q, j)], xb = rl[X::read_at(q, j)];
        if (h) {
          va[q * X::r2 + j].y = xa;
          vb[q * X::r2 + j].y = xb;
        } else {
          va[q * X::r2 + j].x = xa;
          vb[q * X::r2 + j].x = xb;
        }
      }
    }
  }
}

template <typename Real, int N, int RM, int S> struct StageLoop2 {
  __device__ static __forceinline__ void run(cplx_t<Real>* va, cplx_t<Real>* vb, int t, const double2* tw, Real* la,
                                             Real* lb) {
    StageTwiddles<Real, N, RM, S> pre;
    pre.load(t, tw);
    run(va, vb, t, tw, la, lb, pre);
  }
  __device__ static __forceinline__ void run(cplx_t<Real>* va, cplx_t<Real>* vb, int t, const double2* tw, Real* la,
                                             Real* lb, const StageTwiddles<Real, N, RM, S>& pre) {
    stage_compute2<Real, N, RM, S>(va, vb, t, tw, pre);
    if constexpr (S + 1 < FastCfg<Real, N, RM>::NST) {
      StageTwiddles<Real, N, RM, S + 1> next;
      next.load(t, tw);
      stage_exchange2<Real, N, RM, S>(va, vb, t, la, lb);
      StageLoop2<Real, N, RM, S + 1>::run(va, vb, t, tw, la, lb, next);
    }
  }
};

// SPLIT_IN: the input side has odd rows under a padded enumeration; its
// line pairs are loaded as two 8-byte elements, and the second element of a
// pair whose second line is padding (the next row's first element there, or
// past the end of the rank's array) is not loaded.
template <typename Real, int N, int RM, bool NT, int SPLIT_IN = 0>
__device__ __forceinline__ void fast_line2_body(const FastPass& p, int32_t blk, int B, unsigned char* lds) {
  using C = cplx_t<Real>;
  using Cfg = FastCfg<Real, N, RM>;
  typedef Real V4 __attribute__((ext_vector_type(4)));
  constexpr int R = Cfg::R, T = Cfg::T;
  const size_t LB = static_cast<size_t>(p.line_bytes);
  const int P2 = B >> 1;
  const int tid = threadIdx.x;
  // lanes beyond P2*T (grouped launches of 256 lanes) run the stages on zeros
  // in two spare LDS slots (2*P2, 2*P2 + 1) and load and store nothing
  const bool active = tid < P2 * T;
  int t = static_cast<int>(p.bdiv.div(static_cast<uint32_t>(2 * tid)));  // tid / (B / 2): B is even
  const int b = active ? tid - t * P2 : P2;
  if (!active) t = 0;
  const int32_t la = blk * B + 2 * b;  // lines la, la + 1 (nlines is even)
  const double2* tw = reinterpret_cast<const double2*>(p.tw);
  Real* ba = reinterpret_cast<Real*>(lds + (2 * b) * LB);
  Real* bb = reinterpret_cast<Real*>(lds + (2 * b + 1) * LB);
  LineIO<Real, NT> io;
  bool valid = active && la < p.nlines;
  if (valid) valid = make_line_io<Real, NT>(p, la, io);

  bool second = false;
  if constexpr (SPLIT_IN == 1) second = valid && !padding_line(p, la + 1);
  // SPLIT_IN == 2: line la + 1 has addresses of its own on both sides
  [[maybe_unused]] LineIO<Real, NT> io2 = io;
  if constexpr (SPLIT_IN == 2) {
    second = valid && la + 1 < p.nlines;
    if (second) second = make_line_io<Real, NT>(p, la + 1, io2);
  }
  C va[R], vb[R];
  constexpr int r0 = Cfg::P.rad[0];
  constexpr int NB0 = R / r0;
#pragma unroll
  for (int q = 0; q < NB0; ++q) {
    const C* src = reinterpret_cast<const C*>(io.ib) + static_cast<int64_t>(t + q * T) * io.is;
    const int64_t step = static_cast<int64_t>(N / r0) * io.is;
    [[maybe_unused]] const C* src2 = nullptr;
    [[maybe_unused]] int64_t step2 = 0;
    if constexpr (SPLIT_IN == 2) {
      src2 = reinterpret_cast<const C*>(io2.ib) + static_cast<int64_t>(t + q * T) * io2.is;
      step2 = static_cast<int64_t>(N / r0) * io2.is;
    }
#pragma unroll
    for (int j = 0; j < r0; ++j) {
      C a, c;
      if constexpr (SPLIT_IN == 2) {
        a = valid ? gload_c<NT, Real>(src) : C{Real(0), Real(0)};
        c = second ? gload_c<NT, Real>(src2) : C{Real(0), Real(0)};
        src2 += step2;
      } else if constexpr (SPLIT_IN == 1) {
        a = valid ? gload_c<NT, Real>(src) : C{Real(0), Real(0)};
        c = second ? gload_c<NT, Real>(src + 1) : C{Real(0), Real(0)};
      } else {
        const V4 x = valid ? gload<NT>(reinterpret_cast<const V4*>(src)) : V4{Real(0), Real(0), Real(0), Real(0)};
        a = C{x.x, x.y};
        c = C{x.z, x.w};
      }
      va[q * r0 + j] = p.inverse ? cconj(a) : a;
      vb[q * r0 + j] = p.inverse ? cconj(c) : c;
      src += step;
    }
  }
  StageLoop2<Real, N, RM, 0>::run(va, vb, t, tw, ba, bb);
  final_order<Real, N, RM>(va);
  final_order<Real, N, RM>(vb);
  // SPLIT_IN == 2: the pair is stored as one 16-byte element pair where the
  // second line's output follows the first's on a 16-byte boundary at every
  // position (even element stride), else as two elements
  bool pair_out = true;
  if constexpr (SPLIT_IN == 2)
    pair_out = second && io2.ob == io.ob + sizeof(C) && io2.os == io.os && (io.os & 1) == 0 &&
               (reinterpret_cast<uintptr_t>(io.ob) & 15) == 0;
  if (valid && pair_out) {
    C* dst = reinterpret_cast<C*>(io.ob) + static_cast<int64_t>(t) * io.os;
    const int64_t step = static_cast<int64_t>(T) * io.os;
#pragma unroll
    for (int j = 0; j < R; ++j) {
      C a = p.inverse ? cconj(va[j]) : va[j];
      C c = p.inverse ? cconj(vb[j]) : vb[j];
      V4 x;
      x.x = a.x * io.scale;
      x.y = a.y * io.scale;
      x.z = c.x * io.scale;
      x.w = c.y * io.scale;
      gstore<NT>(reinterpret_cast<V4*>(dst), x);
      dst += step;
    }
  } else if constexpr (SPLIT_IN == 2) {
    if (valid) {
      C* dst = reinterpret_cast<C*>(io.ob) + static_cast<int64_t>(t) * io.os;
      const int64_t step = static_cast<int64_t>(T) * io.os;
      [[maybe_unused]] C* dst2 = nullptr;
      [[maybe_unused]] int64_t stepb = 0;
      if (second) {
        dst2 = reinterpret_cast<C*>(io2.ob) + static_cast<int64_t>(t) * io2.os;
        stepb = static_cast<int64_t>(T) * io2.os;
      }
#pragma unroll
      for (int j = 0; j < R; ++j) {
        C a = p.inverse ? cconj(va[j]) : va[j];
        gstore_c<NT, Real>(dst, C{a.x * io.scale, a.y * io.scale});
        dst += step;
        if (second) {
          C c = p.inverse ? cconj(vb[j]) : vb[j];
          gstore_c<NT, Real>(dst2, C{c.x * io.scale, c.y * io.scale});
          dst2 += stepb;
        }
      }
    }
  }
}

// One block's share of a line pass: lines [blk*B, blk*B + B) of p, T = N/R
// lanes per line.  Lanes beyond B*T (a block shape shared by several line
// lengths) run the stages on zeros in a spare LDS slot (index B) so every
// lane reaches every barrier; they load and store nothing.  STAGE (complex64
// grouped passes) moves contiguous lines 16 bytes per lane through LDS.
// BAND: a C2C pass over kept modes: inverse lines read positions outside the
// band as zeros, forward lines store only the band.
template <typename Real, int N, int RM, bool NT, bool SPLIT, bool STAGE = false, bool BAND = false>
__device__ __forceinline__ void fast_line_body(const FastPass& p, int32_t blk, int B, unsigned char* lds) {
  using C = cplx_t<Real>;
  using Cfg = FastCfg<Real, N, RM>;
  constexpr int R = Cfg::R, T = Cfg::T;
  const int tid = threadIdx.x;
  int b, t;
  if (p.lines_fast) {
    t = static_cast<int>(p.bdiv.div(static_cast<uint32_t>(tid)));
    b = tid - t * B;
  } else {
    t = tid % T;
    b = tid / T;
  }
  const bool active = tid < B * T;
  if (!active) {
    b = B;
    t = 0;
  }
  const int32_t line = blk * B + b;
  const double2* tw = reinterpret_cast<const double2*>(p.tw);
  void* buf = lds + b * p.line_bytes;

  bool valid;
  LineIO<Real, NT> io;
  if (T >= 64 && !p.lines_fast) {
    // lanes along the line with T >= 64: each wave holds one line (or only
    // spare lanes), so the line index is wave-uniform and the descriptor
    // arithmetic of make_line_io runs once per wave on the scalar unit
    const int32_t wl = __builtin_amdgcn_readfirstlane(line);
    valid = active && wl < p.nlines;
    if (valid) valid = make_line_io<Real, NT, BAND>(p, wl, io);
  } else {
    valid = active && line < p.nlines;
    if (valid) valid = make_line_io<Real, NT, BAND>(p, line, io);
  }

  C v[R];
  constexpr int r0 = Cfg::P.rad[0];
  constexpr int NB0 = R / r0;
  typedef Real V4 __attribute__((ext_vector_type(4)));
  static_assert(!STAGE || (std::is_same<Real, float>::value && !SPLIT && R % 2 == 0),
                "staged lines are complex64 with complex LDS exchanges");
  bool vin = false;
  if constexpr (STAGE) {
    // contiguous C2C lines that start on a 16-byte boundary are read as
    // element pairs (lane t takes pairs t, t + T, ...: T lanes cover 16*T
    // adjacent bytes per access) and regrouped through the line's LDS buffer
    C* lc = static_cast<C*>(buf);
    vin = valid && p.kind == kC2C && io.is == 1 && (reinterpret_cast<uintptr_t>(io.ib) & 15) == 0;
    if (vin) {
      const V4* src = reinterpret_cast<const V4*>(io.ib) + t;
#pragma unroll
      for (int k = 0; k < R / 2; ++k) {
        const V4 x = gload<NT>(src + k * T);
        const int e = 2 * (t + k * T);
        lc[Cfg::lidx(e)] = C{x.x, x.y};
        lc[Cfg::lidx(e + 1)] = C{x.z, x.w};
      }
    }
    if (p.kind == kC2C) __syncthreads();  // p is the same member for the whole block
    if (vin) {
#pragma unroll
      for (int q = 0; q < NB0; ++q) {
#pragma unroll
        for (int j = 0; j < r0; ++j) {
          const C x = lc[Cfg::lidx(t + q * T + j * (N / r0))];
          v[q * r0 + j] = p.inverse ? cconj(x) : x;
        }
      }
    }
  }
  if (vin) {
    // loaded above, through LDS
  } else if (BAND && p.inverse) {
    // positions p.band < pos < N - p.band are zeros: runs of S positions that
    // lie in there whole are not loaded (a branch on scalars), lanes of the
    // two runs at its ends repeat the address of the band's edge
    constexpr int S = N / r0;
#pragma unroll
    for (int j = 0; j < R; ++j) v[j] = C{Real(0), Real(0)};
    if (valid) {
#pragma unroll
      for (int j = 0; j < r0; ++j) {
        if (j * S > p.band && (j + 1) * S - 1 < N - p.band) continue;
#pragma unroll
        for (int q = 0; q < NB0; ++q) {
          const int pos = t + q * T + j * S;
          const bool keep = pos <= p.band || pos >= N - p.band;
          const C x = gload_c<NT, Real>(reinterpret_cast<const C*>(io.ib) +
                                        static_cast<int64_t>(keep ? pos : p.band) * io.is);
          v[q * r0 + j] = keep ? cconj(x) : C{Real(0), Real(0)};
        }
      }
    }
  } else if (p.kind == kC2C) {
    // C2C lines are walked with pointer increments (no 64-bit product per
    // element).  One branch around all the loads: a select per load puts
    // each load under its own exec mask, and the zeroing moves between them
    // made the compiler wait for the loads in flight halfway through.
    if (valid) {
#pragma unroll
      for (int q = 0; q < NB0; ++q) {
        const C* src = reinterpret_cast<const C*>(io.ib) + static_cast<int64_t>(t + q * T) * io.is;
        const int64_t step = static_cast<int64_t>(N / r0) * io.is;
#pragma unroll
        for (int j = 0; j < r0; ++j) {
          v[q * r0 + j] = gload_c<NT, Real>(src);
          src += step;
        }
      }
      if (p.inverse) {
#pragma unroll
        for (int j = 0; j < R; ++j) v[j] = cconj(v[j]);
      }
    } else {
#pragma unroll
      for (int j = 0; j < R; ++j) v[j] = C{Real(0), Real(0)};
    }
  } else if (valid) {
    // R2C / C2R lines (one branch around the loads, as for C2C, and one per kind)
    if (p.kind == kR2C) {
#pragma unroll
      for (int q = 0; q < NB0; ++q) {
#pragma unroll
        for (int j = 0; j < r0; ++j) v[q * r0 + j] = io.template load_kind<kR2C>(t + q * T + j * (N / r0));
      }
    } else {
#pragma unroll
      for (int q = 0; q < NB0; ++q) {
#pragma unroll
        for (int j = 0; j < r0; ++j) v[q * r0 + j] = io.template load_kind<kC2R>(t + q * T + j * (N / r0));
      }
    }
  } else {
#pragma unroll
    for (int j = 0; j < R; ++j) v[j] = C{Real(0), Real(0)};
  }
  StageLoop<Real, N, RM, SPLIT, 0>::run(v, t, tw, buf);
  bool vout = false;
  if constexpr (STAGE) {
    // the last stage's outputs go to LDS in natural order (this replaces
    // final_order); contiguous aligned C2C outputs are stored as element
    // pairs, any other line reads back positions t + j*T
    constexpr int rl = Cfg::P.rad[Cfg::NST - 1];
    constexpr int NBl = R / rl;
    C* lc = static_cast<C*>(buf);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NBl; ++q) {
#pragma unroll
      for (int j = 0; j < rl; ++j) lc[Cfg::lidx(t + q * T + j * (N / rl))] = v[q * rl + j];
    }
    __syncthreads();
    vout = valid && p.kind == kC2C && io.os == 1 && (reinterpret_cast<uintptr_t>(io.ob) & 15) == 0;
    if (vout) {
      V4* dst = reinterpret_cast<V4*>(io.ob) + t;
#pragma unroll
      for (int k = 0; k < R / 2; ++k) {
        const int e = 2 * (t + k * T);
        C a = lc[Cfg::lidx(e)], c = lc[Cfg::lidx(e + 1)];
        if (p.inverse) {
          a = cconj(a);
          c = cconj(c);
        }
        V4 x;
        x.x = a.x * io.scale;
        x.y = a.y * io.scale;
        x.z = c.x * io.scale;
        x.w = c.y * io.scale;
        gstore<NT>(dst + k * T, x);
      }
    } else {
#pragma unroll
      for (int j = 0; j < R; ++j) v[j] = lc[Cfg::lidx(t + j * T)];
    }
  } else {
    final_order<Real, N, RM>(v);
  }

  if (valid && !vout) {
    if (BAND && !p.inverse) {
#pragma unroll
      for (int j = 0; j < R; ++j) {
        const int pos = t + j * T;
        if (j * T > p.band && (j + 1) * T - 1 < N - p.band) continue;
        if (pos <= p.band || pos >= N - p.band)
          gstore_c<NT, Real>(reinterpret_cast<C*>(io.ob) + static_cast<int64_t>(pos) * io.os,
                             C{v[j].x * io.scale, v[j].y * io.scale});
      }
    } else if (p.kind == kC2C) {
      C* dst = reinterpret_cast<C*>(io.ob) + static_cast<int64_t>(t) * io.os;
      const int64_t step = static_cast<int64_t>(T) * io.os;
#pragma unroll
      for (int j = 0; j < R; ++j) {
        C x = p.inverse ? cconj(v[j]) : v[j];
        x.x *= io.scale;
        x.y *= io.scale;
        gstore_c<NT, Real>(dst, x);
        dst += step;
      }
    } else {
#pragma unroll
      for (int j = 0; j < R; ++j) io.store(t + j * T, v[j]);
    }
  }
}

// Paired R2C / C2R (KIND): slot b of the block transforms lines 2q and 2q+1
// (q = blk*B + b) as one complex line; same stage code as fast_line_body.
// Lane t holds positions t + k*T throughout.
// PROD: a products pass (LinePass::products): each loaded real value is the
// product of the two factor lines' values at that position.
// BAND: half-spectrum entries above p.band are neither read (zeros) nor stored.
template <typename Real, int N, int RM, bool NT, bool SPLIT, int KIND, bool PROD = false, bool BAND = false>
__device__ __forceinline__ void fast_pair_body(const FastPass& p, int32_t blk, int B, unsigned char* lds) {
  using C = cplx_t<Real>;
  using Cfg = FastCfg<Real, N, RM>;
  constexpr int R = Cfg::R, T = Cfg::T, H = R / 2;
  static_assert(R % 2 == 0 && (KIND == kR2C || KIND == kC2R), "real lines");
  const int tid = threadIdx.x;
  int b, t;
  if (p.lines_fast) {
    t = static_cast<int>(p.bdiv.div(static_cast<uint32_t>(tid)));
    b = tid - t * B;
  } else {
    t = tid % T;
    b = tid / T;
  }
  const bool active = tid < B * T;
  if (!active) {
    b = B;
    t = 0;
  }
  const int32_t pair = blk * B + b;
  const bool valid = active && 2 * pair < p.nlines;  // paired passes never enumerate padding
  const double2* tw = reinterpret_cast<const double2*>(p.tw);
  void* buf = lds + b * p.line_bytes;

  PairIO<Real, NT> io{};
  if (T >= 64 && !p.lines_fast) {
    // lanes along the pair with T >= 64: each wave holds one pair (or only
    // spare lanes), so the pair index is wave-uniform and the descriptor
    // arithmetic of make_pair_io runs once per wave on the scalar unit
    const int32_t wp = __builtin_amdgcn_readfirstlane(pair);
    if (valid) io = make_pair_io<Real, NT, PROD, BAND>(p, wp);
  } else {
    if (valid) io = make_pair_io<Real, NT, PROD, BAND>(p, pair);
  }
  const bool vb = valid && io.has_b;

  // LDS index of position t + k*T, and of the mirrored N - t - k*T: both a
  // lane part and a constant where the padding interval divides T
  constexpr bool kLinear = T % (1 << LdsPad<Real>::shift) == 0;
  const int at0 = Cfg::lidx(t), mir0 = Cfg::lidx(N - t);
  auto at = [&](int k) { return kLinear ? at0 + k * T + (k * T >> LdsPad<Real>::shift) : Cfg::lidx(t + k * T); };
  auto mir = [&](int k) { return kLinear ? mir0 - k * T - (k * T >> LdsPad<Real>::shift) : Cfg::lidx(N - t - k * T); };

  // input k of lane t (position t + k*T) is value (k % NB0)*r0 + k / NB0 of
  // the first stage
  constexpr int r0 = Cfg::P.rad[0];
  constexpr int NB0 = R / r0;
  C v[R];
  auto in = [](int k) { return (k % NB0) * r0 + k / NB0; };
  if constexpr (PROD) {
    // Products pass: the block holds whole positions (B is a multiple of 3 and
    // the field axis is enumerated fastest, so slots 3m..3m+2 are the pairs
    // (0,1), (2,3), (4,5) of one position).  Slot 3m+q stages velocity line q
    // of the position into the LDS of the position's three slots; each slot
    // then forms its two product lines from LDS.  Global loads: 3 lines per
    // position instead of 2 per product line.
    const int pq = b % 3;
    Real* st = reinterpret_cast<Real*>(lds + (b - pq) * p.line_bytes);
    if (valid) {
      const Real* src = reinterpret_cast<const Real*>(io.ib[0]) + static_cast<int64_t>(t) * io.is[0];
      const int64_t step = static_cast<int64_t>(T) * io.is[0];
#pragma unroll
      for (int k = 0; k < R; ++k) {
        st[pq * N + t + k * T] = gload<NT>(src);
        src += step;
      }
    }
    __syncthreads();
    // pair q = fields 2q, 2q + 1: (0,0) (0,1) | (0,2) (1,1) | (1,2) (2,2)
    const Real* fa0 = st + prod_first(2 * pq) * N + t;
    const Real* fa1 = st + prod_second(2 * pq) * N + t;
    const Real* fb0 = st + prod_first(2 * pq + 1) * N + t;
    const Real* fb1 = st + prod_second(2 * pq + 1) * N + t;
#pragma unroll
    for (int k = 0; k < R; ++k) v[in(k)] = C{fa0[k * T] * fa1[k * T], fb0[k * T] * fb1[k * T]};
    __syncthreads();  // the staged lines share LDS with the exchanges
  } else if constexpr (KIND == kR2C) {
#pragma unroll
    for (int k = 0; k < R; ++k) v[k] = C{Real(0), Real(0)};
    if (valid) {
      const Real* pa = reinterpret_cast<const Real*>(io.ib[0]) + static_cast<int64_t>(t) * io.is[0];
      const int64_t sa = static_cast<int64_t>(T) * io.is[0];
#pragma unroll
      for (int k = 0; k < R; ++k) {
        v[in(k)].x = gload<NT>(pa);
        pa += sa;
      }
    }
    if (vb) {
      const Real* pb = reinterpret_cast<const Real*>(io.ib[1]) + static_cast<int64_t>(t) * io.is[1];
      const int64_t sb = static_cast<int64_t>(T) * io.is[1];
#pragma unroll
      for (int k = 0; k < R; ++k) {
        v[in(k)].y = gload<NT>(pb);
        pb += sb;
      }
    }
  } else {
    // C2R: each half-spectrum entry X[m], m <= n/2, is loaded once, by the
    // lane holding position m; that lane also forms the input at the mirrored
    // position n - m (from conj X[m]) and hands it over through LDS.  The
    // positions of k < R/2 are below n/2, the one of k = R/2 reaches n/2 only
    // for t = 0; the loads sit under one branch per line (a branch per load
    // would wait for each pair of loads before the next).
    C A[H + 1], Bv[H + 1];
#pragma unroll
    for (int k = 0; k <= H; ++k) {
      A[k] = C{Real(0), Real(0)};
      Bv[k] = C{Real(0), Real(0)};
    }
    const C* la = reinterpret_cast<const C*>(io.ib[0]) + static_cast<int64_t>(t) * io.is[0];
    const C* lb = reinterpret_cast<const C*>(io.ib[1]) + static_cast<int64_t>(t) * io.is[1];
    const int64_t sa = static_cast<int64_t>(T) * io.is[0], sb = static_cast<int64_t>(T) * io.is[1];
    if constexpr (BAND) {
      // as in fast_line_body: whole runs above the band are skipped, lanes
      // beyond its edge repeat the edge's address
      const C* ea = reinterpret_cast<const C*>(io.ib[0]) + p.band * io.is[0];
      const C* eb = reinterpret_cast<const C*>(io.ib[1]) + p.band * io.is[1];
#pragma unroll
      for (int k = 0; k < H; ++k) {
        if (k * T > p.band) continue;
        const bool keep = t + k * T <= p.band;
        if (valid) {
          const C x = gload_c<NT, Real>(keep ? la + k * sa : ea);
          A[k] = keep ? x : C{Real(0), Real(0)};
        }
        if (vb) {
          const C x = gload_c<NT, Real>(keep ? lb + k * sb : eb);
          Bv[k] = keep ? x : C{Real(0), Real(0)};
        }
      }
    } else {
      if (valid) {
#pragma unroll
        for (int k = 0; k < H; ++k) A[k] = gload_c<NT, Real>(la + k * sa);
        if (t == 0) A[H] = gload_c<NT, Real>(la + H * sa);
      }
      if (vb) {
#pragma unroll
        for (int k = 0; k < H; ++k) Bv[k] = gload_c<NT, Real>(lb + k * sb);
        if (t == 0) Bv[H] = gload_c<NT, Real>(lb + H * sb);
      }
    }
    C mirror[H];
#pragma unroll
    for (int k = 0; k <= H; ++k) {
      v[in(k)] = io.c2r_value(t + k * T, true, A[k], Bv[k]);
      if (k < H) mirror[k] = io.c2r_value(N - t - k * T, false, A[k], Bv[k]);
    }
    // positions above n/2 receive the value formed by the lane holding n - pos
    if constexpr (SPLIT) {
      Real* lr = static_cast<Real*>(buf);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (h) __syncthreads();
#pragma unroll
        for (int k = 0; k < H; ++k)
          if (k > 0 || t > 0) lr[mir(k)] = h ? mirror[k].y : mirror[k].x;
        __syncthreads();
#pragma unroll
        for (int k = H; k < R; ++k) {
          if (k > H || t > 0) {
            const Real x = lr[at(k)];
            if (h) {
              v[in(k)].y = x;
            } else {
              v[in(k)].x = x;
            }
          }
        }
      }
    } else {
      C* lc = static_cast<C*>(buf);
#pragma unroll
      for (int k = 0; k < H; ++k)
        if (k > 0 || t > 0) lc[mir(k)] = mirror[k];
      __syncthreads();
#pragma unroll
      for (int k = H; k < R; ++k)
        if (k > H || t > 0) v[in(k)] = lc[at(k)];
    }
  }
  StageLoop<Real, N, RM, SPLIT, 0>::run(v, t, tw, buf);
  final_order<Real, N, RM>(v);
  const int64_t ta = static_cast<int64_t>(T) * io.os[0], tb = static_cast<int64_t>(T) * io.os[1];
  if constexpr (KIND == kC2R) {
    // w = FFT(conj Z) at each position, so a + i b = conj(w)
    if (valid) {
      Real* pa = reinterpret_cast<Real*>(io.ob[0]) + static_cast<int64_t>(t) * io.os[0];
#pragma unroll
      for (int k = 0; k < R; ++k) {
        gstore<NT>(pa, v[k].x * io.scale);
        pa += ta;
      }
    }
    if (vb) {
      Real* pb = reinterpret_cast<Real*>(io.ob[1]) + static_cast<int64_t>(t) * io.os[1];
#pragma unroll
      for (int k = 0; k < R; ++k) {
        gstore<NT>(pb, -v[k].y * io.scale);
        pb += tb;
      }
    }
  } else {
    // R2C: entry m = t + k*T <= n/2 of both spectra from Z_m and Z_{n-m}.  The
    // lanes hand out the upper half of Z; Z_0 and Z_{n/2} are their own
    // mirrors.
    C A[H + 1], Bv[H + 1];
    const bool own = t == 0;
    if constexpr (SPLIT) {
      Real* lr = static_cast<Real*>(buf);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        __syncthreads();
#pragma unroll
        for (int k = H; k < R; ++k) lr[at(k)] = h ? v[k].y : v[k].x;
        __syncthreads();
#pragma unroll
        for (int k = 0; k <= H; ++k) {
          const Real z = h ? v[k].y : v[k].x;
          Real m = z;
          if (k < H) {
            m = lr[mir(k)];
            if (k == 0 && own) m = z;
          }
          if (h) {
            A[k].y = z - m;
            Bv[k].x = z + m;
          } else {
            A[k].x = z + m;
            Bv[k].y = m - z;
          }
        }
      }
    } else {
      C* lc = static_cast<C*>(buf);
      __syncthreads();
#pragma unroll
      for (int k = H; k < R; ++k) lc[at(k)] = v[k];
      __syncthreads();
#pragma unroll
      for (int k = 0; k <= H; ++k) {
        C m = v[k];
        if (k < H) {
          m = lc[mir(k)];
          if (k == 0 && own) m = v[0];
        }
        A[k] = C{v[k].x + m.x, v[k].y - m.y};
        Bv[k] = C{v[k].y + m.y, m.x - v[k].x};
      }
    }
    const Real h0 = Real(0.5) * io.scale, hw = h0 * io.hw;
    if (valid) {
      C* pa = reinterpret_cast<C*>(io.ob[0]) + static_cast<int64_t>(t) * io.os[0];
#pragma unroll
      for (int k = 0; k <= H; ++k) {
        const Real h = k == H || (k == 0 && own) ? h0 : hw;
        if (BAND ? k < H && t + k * T <= p.band : k < H || own) gstore_c<NT, Real>(pa, C{A[k].x * h, A[k].y * h});
        pa += ta;
      }
    }
    if (vb) {
      C* pb = reinterpret_cast<C*>(io.ob[1]) + static_cast<int64_t>(t) * io.os[1];
#pragma unroll
      for (int k = 0; k <= H; ++k) {
        const Real h = k == H || (k == 0 && own) ? h0 : hw;
        if (BAND ? k < H && t + k * T <= p.band : k < H || own) gstore_c<NT, Real>(pb, C{Bv[k].x * h, Bv[k].y * h});
        pb += tb;
      }
    }
  }
}

// Workgroups go to the 8 XCDs round-robin; renumber them so XCD x owns the
// x-th contiguous range of blocks (a bijection for any grid size).
__device__ __forceinline__ int32_t xcd_block(int32_t b, int32_t nb) {
  constexpr int32_t kXcds = 8;
  const int32_t q = nb / kXcds, r = nb % kXcds;
  const int32_t x = b % kXcds, i = b / kXcds;
  return x < r ? x * (q + 1) + i : r * (q + 1) + (x - r) * q + i;
}

// Block of the pass for hardware block b: optional XCD-contiguous numbering,
// then an optional column-major walk of the (nb / C) x C block grid, where C
// blocks cover one row of the fastest batch axis (p.swizzle = C; the launcher
// sets it only when it divides the grid).
__device__ __forceinline__ int32_t pass_block(const FastPass& p, int32_t b, int32_t nb) {
  if (p.xcd_remap) b = xcd_block(b, nb);
  if (p.swizzle > 1) {
    const int32_t rows = nb / p.swizzle;
    b = (b % rows) * p.swizzle + b / rows;
  }
  return b;
}

template <typename Real, int N, int RM, bool NT, bool SPLIT, int KIND, bool PROD = false, bool BAND = false>
__global__ void __launch_bounds__(1024) fft_pair_fast(const FastPass p) {
  extern __shared__ unsigned char smem_raw[];
  const int32_t blk = pass_block(p, blockIdx.x, gridDim.x);
  fast_pair_body<Real, N, RM, NT, SPLIT, KIND, PROD, BAND>(p, blk, p.lines_per_block, smem_raw);
}

template <typename Real, int N, int RM, bool NT, bool SPLIT, bool BAND = false>
__global__ void __launch_bounds__(1024) fft_line_fast(const FastPass p) {
  extern __shared__ unsigned char smem_raw[];
  const int32_t blk = pass_block(p, blockIdx.x, gridDim.x);
  fast_line_body<Real, N, RM, NT, SPLIT, false, BAND>(p, blk, p.lines_per_block, smem_raw);
}

template <typename Real, int N, int RM, bool NT, int SPLIT_IN>
__global__ void __launch_bounds__(1024) fft_line2_fast(const FastPass p) {
  extern __shared__ unsigned char smem_raw[];
  const int32_t blk = pass_block(p, blockIdx.x, gridDim.x);
  fast_line2_body<Real, N, RM, NT, SPLIT_IN>(p, blk, p.lines_per_block, smem_raw);
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
namespace {

// Raises kernel fn's dynamic-LDS limit to at least `bytes` (the cached
// limit belongs to that one kernel; updates only grow it and are serialised,
// so concurrent launches from several host threads never lower it).  Never
// called inside a stream capture that follows an eager launch of the same
// shape: the limit is then already raised.
inline hipError_t raise_lds_limit(std::atomic<size_t>& limit, const void* fn, size_t bytes) {
  if (bytes <= limit.load(std::memory_order_acquire)) return hipSuccess;
  static std::mutex m;
  std::lock_guard<std::mutex> lock(m);
  if (bytes <= limit.load(std::memory_order_relaxed)) return hipSuccess;
  const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes));
  if (e != hipSuccess) return e;
  limit.store(bytes, std::memory_order_release);
  return hipSuccess;
}

// One compile-time variant of the fast kernels: paired or single lines,
// nontemporal or cached accesses, split or complex LDS exchanges.
template <typename Real, int N, int RM, bool NT, bool SPLIT> struct FastVariant {
  static constexpr bool kPairs = !(std::is_same<Real, double>::value && (N % 3 == 0 || N % 5 == 0));
  // pair: 0 single lines, else kR2C or kC2R
  static const void* fn(int pair) {
    if constexpr (kPairs) {
      if (pair == kR2C) return reinterpret_cast<const void*>(&fft_pair_fast<Real, N, 8, NT, SPLIT, kR2C>);
      if (pair == kC2R) return reinterpret_cast<const void*>(&fft_pair_fast<Real, N, 8, NT, SPLIT, kC2R>);
    }
    return reinterpret_cast<const void*>(&fft_line_fast<Real, N, RM, NT, SPLIT>);
  }
  static void launch(int pair, unsigned grid, unsigned threads, size_t smem, hipStream_t s, const FastPass& f) {
    if constexpr (kPairs) {
      if (pair == kR2C) {
        hipLaunchKernelGGL((fft_pair_fast<Real, N, 8, NT, SPLIT, kR2C>), dim3(grid), dim3(threads), smem, s, f);
        return;
      }
      if (pair == kC2R) {
        hipLaunchKernelGGL((fft_pair_fast<Real, N, 8, NT, SPLIT, kC2R>), dim3(grid), dim3(threads), smem, s, f);
        return;
      }
    }
    hipLaunchKernelGGL((fft_line_fast<Real, N, RM, NT, SPLIT>), dim3(grid), dim3(threads), smem, s, f);
  }
};

// split exchanges exist for FP64, and for FP32 lines of 1024 points and more
// (shorter FP32 lines are small in LDS already and ran slower split)
template <typename Real, int N> constexpr bool split_available() {
  return std::is_same<Real, double>::value || N >= 1024;
}

template <typename Real, int N, int RM, bool NT>
void launch_fast_variant(bool split, int pair, unsigned grid, unsigned threads, size_t smem, hipStream_t s,
                         const FastPass& p) {
  if constexpr (split_available<Real, N>()) {
    if (split) {
      FastVariant<Real, N, RM, NT, true>::launch(pair, grid, threads, smem, s, p);
      return;
    }
  }
  FastVariant<Real, N, RM, NT, false>::launch(pair, grid, threads, smem, s, p);
}

template <typename Real, int N, int RM>
const void* fast_variant_fn(bool split, int pair, bool nt) {
  if constexpr (split_available<Real, N>()) {
    if (split) return nt ? FastVariant<Real, N, RM, true, true>::fn(pair) : FastVariant<Real, N, RM, false, true>::fn(pair);
  }
  return nt ? FastVariant<Real, N, RM, true, false>::fn(pair) : FastVariant<Real, N, RM, false, false>::fn(pair);
}

// Two lines per lane applies to FP32 C2C lanes-across-lines passes of
// power-of-two lengths >= 128 whose consecutive lines are adjacent elements
// of one row on both sides (the fastest batch axis is the innermost storage
// axis, not split over ranks, with even row lengths (pitches) and 16-byte
// aligned rank buffers, so every line pair is one aligned 16-byte element
// pair), with an even number of lines per block, of lines and of the first
// line.
template <typename Real, int N> constexpr bool dual_kernel_exists() {
  return std::is_same<Real, float>::value && N >= 128 && (N & (N - 1)) == 0;
}

// Returns -1 where two lines per lane do not apply, else the dual_split
// mask of the pass.  An input side whose rows are odd is accepted when the
// lines are enumerated over a padded extent of even pitch along the row axis
// (pairs then never straddle two rows): its pairs are loaded as two 8-byte
// elements and the padding half of a row's last pair is skipped.  (Storing
// such a side as two 8-byte elements measured slower than the one-line
// kernel on the 1024^3 x pass, so odd output rows keep one line per lane.)
inline int dual_lines_mode(const LinePass& p, int B) {
  if (!p.dual_lines || p.kind != kC2C || !p.lines_fast || p.nbatch < 1 || B < 2 || B % 2) return -1;
  const int j = p.nbatch - 1, fa = p.batch_axis[j];
  // an odd unpadded row length of a padded array is fine: the pair at the
  // end of a row then covers one padding element, which lies inside the row
  // pitch and is never read by any pass
  if (p.batch_ext[j] % 2 || p.line_begin % 2 || p.nlines % 2) return -1;
  const bool padded_rows = p.pad_real > 0 && p.pad_axis == fa;
  int mask = 0, bit = 1;
  for (const DDesc* d : {&p.in, &p.out}) {
    const int inner = d->layout_left ? d->map[0] : d->map[d->ndim - 1];
    if (inner != fa || d->ntopo[fa] != 1) return -1;
    const int32_t row = (!d->layout_left && d->pitch > 0) ? d->pitch : d->ext[fa];
    int ranks = 1;
    for (int a = 0; a < d->ndim; ++a) ranks *= d->ntopo[a];
    bool aligned = true;
    for (int r = 0; r < ranks && r < kMaxRanks; ++r)
      if (reinterpret_cast<uintptr_t>(d->ptr[r]) % 16 != 0) aligned = false;
    if (row % 2) {
      if (!padded_rows || bit != 1) return -1;
      mask |= bit;
    } else if (!aligned) {
      return -1;
    }
    bit <<= 1;
  }
  return mask;
}

inline bool dual_lines_apply_impl(const LinePass& p, int B) { return dual_lines_mode(p, B) == 0; }

// Where dual_lines_mode refuses odd output rows: an unpadded output whose
// rows run along the fastest batch axis, both sides with that axis innermost
// and undistributed.  Enumerated over the real elements, lines 2b and 2b+1
// are consecutive output elements, also across a row end; the kernel then
// takes each line's addresses on their own (two-lines mode 2) and pairs the
// stores where they are adjacent and 16-byte aligned.  Returns false or
// p in that mode.
inline bool dual_lines_linear(const LinePass& p, int B, LinePass& q) {
  if (!p.dual_lines || p.kind != kC2C || !p.lines_fast || p.nbatch < 1 || B < 2 || B % 2) return false;
  if (p.line_begin != 0) return false;
  const int j = p.nbatch - 1, fa = p.batch_axis[j];
  for (const DDesc* d : {&p.in, &p.out}) {
    if (d->layout_left) return false;
    if (d->map[d->ndim - 1] != fa || d->ntopo[fa] != 1) return false;
  }
  if (p.out.pitch > 0 || p.out.ext[fa] % 2 == 0) return false;
  if (p.pad_real > 0) return false;
  q = p;
  q.dual_split = 2;
  return true;
}

template <typename Real, int N, int RM>
hipError_t launch_dual(LinePass p, int B, hipStream_t s) {
  if constexpr (!dual_kernel_exists<Real, N>()) {
    return hipErrorInvalidConfiguration;
  } else {
    using Cfg = FastCfg<Real, N, RM>;
    constexpr int T = Cfg::T;
    const int P2 = B / 2;
    size_t line = dual_stride(dual_line_bytes<Real, N, RM>(), B);
    if (B * line > 160 * 1024) line = dual_line_bytes<Real, N, RM>();
    p.line_bytes = static_cast<int32_t>(line);
    const size_t smem = B * line;
    if (P2 * T > 1024 || smem > 160 * 1024) return hipErrorInvalidConfiguration;
    p.lines_per_block = B;
    static std::atomic<size_t> lds_limit[6] = {64 * 1024, 64 * 1024, 64 * 1024, 64 * 1024, 64 * 1024, 64 * 1024};
    const int nt = p.nontemporal ? 1 : 0;
    // 0: paired 16-byte loads, 1: adjacent input lines as two 8-byte loads,
    // 2: every line with its own addresses
    const int mode = p.dual_split & 2 ? 2 : (p.dual_split & 1);
    const void* fns[2][3] = {
        {reinterpret_cast<const void*>(&fft_line2_fast<Real, N, RM, false, 0>),
         reinterpret_cast<const void*>(&fft_line2_fast<Real, N, RM, false, 1>),
         reinterpret_cast<const void*>(&fft_line2_fast<Real, N, RM, false, 2>)},
        {reinterpret_cast<const void*>(&fft_line2_fast<Real, N, RM, true, 0>),
         reinterpret_cast<const void*>(&fft_line2_fast<Real, N, RM, true, 1>),
         reinterpret_cast<const void*>(&fft_line2_fast<Real, N, RM, true, 2>)}};
    const hipError_t e = raise_lds_limit(lds_limit[3 * nt + mode], fns[nt][mode], smem);
    if (e != hipSuccess) return e;
    const unsigned grid = static_cast<unsigned>((static_cast<int64_t>(p.nlines) + B - 1) / B);
    if (grid == 0) return hipSuccess;
    if (p.swizzle) {
      const int32_t inner = p.batch_ext[p.nbatch - 1];
      const int32_t C = (inner > 0 && inner % B == 0) ? inner / B : 0;
      p.swizzle = (C > 1 && grid % static_cast<unsigned>(C) == 0 && grid / C > 1) ? C : 0;
    }
    const dim3 g(grid), b(P2 * T);
    if (nt) {
      if (mode == 2) hipLaunchKernelGGL((fft_line2_fast<Real, N, RM, true, 2>), g, b, smem, s, fast_pass(p, sizeof(Real) == 8));
      else if (mode == 1) hipLaunchKernelGGL((fft_line2_fast<Real, N, RM, true, 1>), g, b, smem, s, fast_pass(p, sizeof(Real) == 8));
      else hipLaunchKernelGGL((fft_line2_fast<Real, N, RM, true, 0>), g, b, smem, s, fast_pass(p, sizeof(Real) == 8));
    } else {
      if (mode == 2) hipLaunchKernelGGL((fft_line2_fast<Real, N, RM, false, 2>), g, b, smem, s, fast_pass(p, sizeof(Real) == 8));
      else if (mode == 1) hipLaunchKernelGGL((fft_line2_fast<Real, N, RM, false, 1>), g, b, smem, s, fast_pass(p, sizeof(Real) == 8));
      else hipLaunchKernelGGL((fft_line2_fast<Real, N, RM, false, 0>), g, b, smem, s, fast_pass(p, sizeof(Real) == 8));
    }
    return hipGetLastError();
  }
}

template <typename Real, int N, int RM>
hipError_t launch_fast(LinePass p, hipStream_t s) {
  using Cfg = FastCfg<Real, N, RM>;
  using C = cplx_t<Real>;
  constexpr int T = Cfg::T;
  if constexpr (dual_kernel_exists<Real, N>()) {
    // default: 32 lines (256-byte row segments) or as many as 1024 lanes hold
    int Bd = p.lines_per_block > 0 ? p.lines_per_block : (T <= 64 ? 32 : 2 * (1024 / T));
    if (p.fit_block)
      while (Bd > 2 && Bd / 2 * T > 1024) Bd /= 2;
    const int mode = dual_lines_mode(p, Bd);
    if (mode >= 0) {
      p.dual_split = mode;
      return launch_dual<Real, N, RM>(p, Bd, s);
    }
    LinePass q;
    if (dual_lines_linear(p, Bd, q)) return launch_dual<Real, N, RM>(q, Bd, s);
  }
  const bool split = split_available<Real, N>() && p.split_lds != 0;
  const size_t line_bytes = split ? line_lds_bytes<Real, N, RM, true>() : line_lds_bytes<Real, N, RM, false>();
  const int elem = static_cast<int>(split ? sizeof(Real) : sizeof(C));
  int B = p.lines_per_block;
  if (B <= 0) {
    if (p.lines_fast) {
      B = 128 / static_cast<int>(sizeof(C));  // lines per 128-byte row segment
      while (B * T > 1024 && B > 1) B /= 2;
    } else {
      B = T >= 256 ? 1 : 256 / T;
    }
    while (B > 1 && static_cast<size_t>(B) * line_bytes > 160 * 1024) B /= 2;
  }
  if (p.fit_block)  // at least two blocks resident on a CU, two blocks per CU in the grid
    while (B > 1 && (B * T > 1024 || static_cast<size_t>(B) * line_bytes > 80 * 1024 ||
                     (B > 4 && B * T > 64 && p.nlines / B < 512)))
      B /= 2;
  size_t line = line_stride(line_bytes, elem, p.lines_fast != 0, B, T);
  if (B * line > 160 * 1024) line = line_bytes;
  p.line_bytes = static_cast<int32_t>(line);
  const size_t smem = B * line;
  if (B * T > 1024 || smem > 160 * 1024) return hipErrorInvalidConfiguration;
  p.lines_per_block = B;
  // two real lines per complex FFT for forward R2C and inverse C2R passes
  // (kernels for 8 values per thread)
  // (FP64 lines of 96 and 160 points run one by one)
  const bool pair = FastVariant<Real, N, RM, false, false>::kPairs && RM == 8 && p.paired &&
                    ((p.kind == kR2C && !p.inverse) || (p.kind == kC2R && p.inverse));
  const bool nt = p.nontemporal != 0;
  const int kind = pair ? p.kind : 0;
  const int v = 6 * (split ? 1 : 0) + 2 * kind + (nt ? 1 : 0);
  // raise the dynamic-LDS limit once per kernel instance
  static std::atomic<size_t> lds_limit[12] = {64 * 1024, 64 * 1024, 64 * 1024, 64 * 1024, 64 * 1024, 64 * 1024,
                                              64 * 1024, 64 * 1024, 64 * 1024, 64 * 1024, 64 * 1024, 64 * 1024};
  {
    const hipError_t e = raise_lds_limit(lds_limit[v], fast_variant_fn<Real, N, RM>(split, kind, nt), smem);
    if (e != hipSuccess) return e;
  }
  const int64_t units = pair ? (static_cast<int64_t>(p.nlines) + 1) / 2 : p.nlines;
  const unsigned grid = static_cast<unsigned>((units + B - 1) / B);
  if (grid == 0) return hipSuccess;
  if (p.swizzle) {
    // C = blocks per row of the fastest batch axis; the walk needs whole rows
    const int32_t inner = p.nbatch > 0 ? p.batch_ext[p.nbatch - 1] : 0;
    const int32_t per = pair ? 2 * B : B;
    const int32_t C = (inner > 0 && inner % per == 0) ? inner / per : 0;
    p.swizzle = (C > 1 && grid % static_cast<unsigned>(C) == 0 && grid / C > 1) ? C : 0;
  }
  const FastPass f = fast_pass(p, sizeof(Real) == 8);
  if (nt) {
    launch_fast_variant<Real, N, RM, true>(split, kind, grid, static_cast<unsigned>(T * B), smem, s, f);
  } else {
    launch_fast_variant<Real, N, RM, false>(split, kind, grid, static_cast<unsigned>(T * B), smem, s, f);
  }
  return hipGetLastError();
}

template <typename Real, int N>
hipError_t launch_fast_r(const LinePass& p, hipStream_t s) {
  switch (p.values_per_thread) {
    case 4: return launch_fast<Real, N, 4>(p, s);
    case 16: return launch_fast<Real, N, 16>(p, s);
    default: return launch_fast<Real, N, 8>(p, s);
  }
}

// FP64 products pass: the paired R2C kernel (8 values per thread) with the
// products formed at the loads; block shape as launch_fast's pair path.
template <int N>
hipError_t launch_products(LinePass p, hipStream_t s) {
  using Real = double;
  using Cfg = FastCfg<Real, N, 8>;
  constexpr int T = Cfg::T;
  if (!p.products || p.kind != kR2C || p.inverse) return hipErrorInvalidValue;
  const bool split = p.split_lds != 0;
  const size_t line_bytes = split ? line_lds_bytes<Real, N, 8, true>() : line_lds_bytes<Real, N, 8, false>();
  // pairs per block: whole positions (3 pairs each) filling at least three
  // full waves (192 lanes; the 256^3 NS step took 8.01 ms with it, 8.23 ms
  // with the R2C pass's own 3 pairs of 32 lanes, 8.36-8.49 ms with 6 or 12
  // waves), cut to what this shape can hold
  int B = 3;
  while (B * T < 192 || (B * T) % 64) B += 3;
  while (B > 3 && (B * T > 1024 || static_cast<size_t>(B) * line_bytes > 160 * 1024)) B -= 3;
  p.line_bytes = static_cast<int32_t>(line_bytes);
  const size_t smem = static_cast<size_t>(B) * line_bytes;
  if (B * T > 1024 || smem > 160 * 1024 || p.nlines % 6 != 0 || p.line_begin % 6 != 0)
    return hipErrorInvalidConfiguration;
  // the staged velocity lines (3 per position) fit in the three slots' LDS
  static_assert(3 * sizeof(Real) * N <= 3 * line_lds_bytes<Real, N, 8, true>(), "staging area");
  p.lines_per_block = B;
  p.swizzle = 0;
  const bool nt = p.nontemporal != 0;
  static std::atomic<size_t> lds_limit[4] = {64 * 1024, 64 * 1024, 64 * 1024, 64 * 1024};
  const void* fn = split ? (nt ? reinterpret_cast<const void*>(&fft_pair_fast<Real, N, 8, true, true, kR2C, true>)
                               : reinterpret_cast<const void*>(&fft_pair_fast<Real, N, 8, false, true, kR2C, true>))
                         : (nt ? reinterpret_cast<const void*>(&fft_pair_fast<Real, N, 8, true, false, kR2C, true>)
                               : reinterpret_cast<const void*>(&fft_pair_fast<Real, N, 8, false, false, kR2C, true>));
  const hipError_t e = raise_lds_limit(lds_limit[2 * (split ? 1 : 0) + (nt ? 1 : 0)], fn, smem);
  if (e != hipSuccess) return e;
  const int64_t units = (static_cast<int64_t>(p.nlines) + 1) / 2;
  const unsigned grid = static_cast<unsigned>((units + B - 1) / B);
  if (grid == 0) return hipSuccess;
  const dim3 g(grid), b(static_cast<unsigned>(T * B));
  if (split) {
    if (nt) hipLaunchKernelGGL((fft_pair_fast<Real, N, 8, true, true, kR2C, true>), g, b, smem, s, fast_pass(p, sizeof(Real) == 8));
    else hipLaunchKernelGGL((fft_pair_fast<Real, N, 8, false, true, kR2C, true>), g, b, smem, s, fast_pass(p, sizeof(Real) == 8));
  } else {
    if (nt) hipLaunchKernelGGL((fft_pair_fast<Real, N, 8, true, false, kR2C, true>), g, b, smem, s, fast_pass(p, sizeof(Real) == 8));
    else hipLaunchKernelGGL((fft_pair_fast<Real, N, 8, false, false, kR2C, true>), g, b, smem, s, fast_pass(p, sizeof(Real) == 8));
  }
  return hipGetLastError();
}

// FP64 passes over kept modes (LinePass::band): 8 values per lane, exchanges
// in halves; C2C lines, R2C / C2R lines in pairs, products formed at the loads.
template <int N, bool NT>
hipError_t launch_band(LinePass p, hipStream_t s) {
  using Real = double;
  using Cfg = FastCfg<Real, N, 8>;
  constexpr int T = Cfg::T;
  constexpr size_t line_bytes = line_lds_bytes<Real, N, 8, true>();
  const bool pair = p.kind != kC2C;
  if (pair && (p.kind == kR2C) == (p.inverse != 0)) return hipErrorInvalidValue;
  int B = p.lines_per_block;
  if (p.products) {
    // whole positions of three pairs each, as launch_products
    B = 3;
    while (B * T < 192 || (B * T) % 64) B += 3;
    while (B > 3 && (B * T > 1024 || static_cast<size_t>(B) * line_bytes > 160 * 1024)) B -= 3;
    if (p.kind != kR2C || p.nlines % 6 != 0 || p.line_begin % 6 != 0) return hipErrorInvalidConfiguration;
  } else if (B <= 0) {
    B = p.lines_fast ? 8 : (T >= 256 ? 1 : 256 / T);
    while (B * T > 1024) B /= 2;
  }
  if (p.fit_block && !p.products)  // as launch_fast
    while (B > 1 && (B * T > 1024 || (B > 4 && B * T > 64 && p.nlines / B < 512))) B /= 2;
  size_t line = p.products ? line_bytes : line_stride(line_bytes, sizeof(Real), p.lines_fast != 0, B, T);
  if (B * line > 160 * 1024) line = line_bytes;
  p.line_bytes = static_cast<int32_t>(line);
  const size_t smem = B * line;
  if (B * T > 1024 || smem > 160 * 1024) return hipErrorInvalidConfiguration;
  p.lines_per_block = B;
  p.swizzle = 0;
  const int64_t units = pair ? (static_cast<int64_t>(p.nlines) + 1) / 2 : p.nlines;
  const dim3 grid(static_cast<unsigned>((units + B - 1) / B)), block(static_cast<unsigned>(T * B));
  static std::atomic<size_t> limit[4] = {64 * 1024, 64 * 1024, 64 * 1024, 64 * 1024};
  const void* fns[4] = {reinterpret_cast<const void*>(&fft_line_fast<Real, N, 8, NT, true, true>),
                        reinterpret_cast<const void*>(&fft_pair_fast<Real, N, 8, NT, true, kR2C, false, true>),
                        reinterpret_cast<const void*>(&fft_pair_fast<Real, N, 8, NT, true, kC2R, false, true>),
                        reinterpret_cast<const void*>(&fft_pair_fast<Real, N, 8, NT, true, kR2C, true, true>)};
  const int k = p.products ? 3 : p.kind == kC2R ? 2 : pair ? 1 : 0;
  const hipError_t e = raise_lds_limit(limit[k], fns[k], smem);
  if (e != hipSuccess) return e;
  const FastPass f = fast_pass(p, true);
  if (k == 3) hipLaunchKernelGGL((fft_pair_fast<Real, N, 8, NT, true, kR2C, true, true>), grid, block, smem, s, f);
  else if (k == 2) hipLaunchKernelGGL((fft_pair_fast<Real, N, 8, NT, true, kC2R, false, true>), grid, block, smem, s, f);
  else if (k == 1) hipLaunchKernelGGL((fft_pair_fast<Real, N, 8, NT, true, kR2C, false, true>), grid, block, smem, s, f);
  else hipLaunchKernelGGL((fft_line_fast<Real, N, 8, NT, true, true>), grid, block, smem, s, f);
  return hipGetLastError();
}

}  // namespace

// fast-kernel dispatch for one precision and a range of lengths (defined in
// fft_lines_*.hip); hipErrorNotSupported for lengths outside the range
hipError_t dispatch_fast_f64_short(const LinePass& p, hipStream_t s);
hipError_t dispatch_fast_f64_long(const LinePass& p, hipStream_t s);
hipError_t dispatch_fast_f32_short(const LinePass& p, hipStream_t s);
hipError_t dispatch_fast_f32_long(const LinePass& p, hipStream_t s);
hipError_t dispatch_fast_f64_xl(const LinePass& p, hipStream_t s);
hipError_t dispatch_fast_f32_xl(const LinePass& p, hipStream_t s);
hipError_t dispatch_products_f64(const LinePass& p, hipStream_t s);
hipError_t dispatch_band_f64(const LinePass& p, hipStream_t s);

}  // namespace dfft
