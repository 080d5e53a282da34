// In-register / LDS line FFT engine for gfx950 (CDNA4, wave64).
//
// A "line" of N complex values is owned by TPL consecutive threads of a
// workgroup.  Thread t holds v[q] = x[t + TPL*q] for q < E = N/TPL (the
// "stride-TPL" layout).  A mixed-radix Stockham autosort transform with the
// compile-time radix list Rs... runs the butterflies of every pass in
// registers; passes exchange through the line's LDS slice.  The last pass
// writes its outputs straight back into registers, and because the Stockham
// autosort output of the final pass lands at j + r*N/R, the output layout is
// the same stride-TPL layout as the input.  Forward and inverse transforms
// therefore chain without any reordering, which is what lets the pass
// kernels do  FFT -> pointwise multiply -> IFFT  with one LDS exchange per
// transform for N = R0*R1.
//
// Forward uses W = exp(-2 pi i / N); the inverse is unnormalised (callers
// fold 1/N into their spectral multipliers).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace kw {

template <typename T>
struct Cx {
  T x, y;
};

template <typename T>
__device__ __forceinline__ Cx<T> cadd(Cx<T> a, Cx<T> b) { return {a.x + b.x, a.y + b.y}; }
template <typename T>
__device__ __forceinline__ Cx<T> csub(Cx<T> a, Cx<T> b) { return {a.x - b.x, a.y - b.y}; }
template <typename T>
__device__ __forceinline__ Cx<T> cmul(Cx<T> a, Cx<T> b) {
  return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}
// a * conj(b)
template <typename T>
__device__ __forceinline__ Cx<T> cmulc(Cx<T> a, Cx<T> b) {
  return {a.x * b.x + a.y * b.y, a.y * b.x - a.x * b.y};
}
template <typename T>
__device__ __forceinline__ Cx<T> cscale(Cx<T> a, T s) { return {a.x * s, a.y * s}; }
// multiply by -i (forward) or +i (inverse)
template <typename T, bool INV>
__device__ __forceinline__ Cx<T> rot90(Cx<T> a) {
  return INV ? Cx<T>{-a.y, a.x} : Cx<T>{a.y, -a.x};
}

// ---------------------------------------------------------------------------
// Compile-time trigonometry for the in-register butterfly constants.
// ---------------------------------------------------------------------------
constexpr double kPi = 3.14159265358979323846264338327950288;

constexpr double ce_sin_red(double x) {  // |x| <= pi/4, Taylor to 1e-20
  double term = x, sum = x, x2 = x * x;
  for (int n = 1; n < 14; ++n) {
    term *= -x2 / ((2 * n) * (2 * n + 1));
    sum += term;
  }
  return sum;
}
constexpr double ce_cos_red(double x) {
  double term = 1.0, sum = 1.0, x2 = x * x;
  for (int n = 1; n < 14; ++n) {
    term *= -x2 / ((2 * n - 1) * (2 * n));
    sum += term;
  }
  return sum;
}
// cos/sin of 2*pi*num/den with exact octant reduction on the rational angle
constexpr void ce_sincos_frac(long num, long den, double& s, double& c) {
  num %= den;
  if (num < 0) num += den;
  // angle = 2 pi num/den; octant = floor(8 num / den)
  long o = (8 * num) / den;
  // remainder angle in [0, pi/4): r = 2pi*num/den - o*pi/4
  double r = 2.0 * kPi * (double)(8 * num - o * den) / (8.0 * (double)den);
  double sr = ce_sin_red(r), cr = ce_cos_red(r);
  // rotate by o*pi/4 using exact octant identities
  const double h = 0.70710678118654752440084436210484904;
  double c8[8] = {1, h, 0, -h, -1, -h, 0, h};
  double s8[8] = {0, h, 1, h, 0, -h, -1, -h};
  c = cr * c8[o] - sr * s8[o];
  s = sr * c8[o] + cr * s8[o];
}

template <int R>
struct RootTable {
  double c[R > 0 ? R : 1];
  double s[R > 0 ? R : 1];
  constexpr RootTable() : c(), s() {
    for (int k = 0; k < R; ++k) {
      double sv = 0, cv = 0;
      ce_sincos_frac(k, R, sv, cv);
      c[k] = cv;
      s[k] = sv;
    }
  }
};

// W_R^m = exp(-2 pi i m / R) (forward), conjugate for the inverse.
template <typename T, int R, bool INV>
__device__ __forceinline__ Cx<T> root(int m) {
  constexpr RootTable<R> tab{};
  m %= R;
  return Cx<T>{(T)tab.c[m], INV ? (T)tab.s[m] : (T)(-tab.s[m])};
}

// ---------------------------------------------------------------------------
// Small DFTs in registers (natural order in, natural order out).
// ---------------------------------------------------------------------------
template <int R>
struct SmallestFactor {
  static constexpr int f() {
    for (int p = 2; p * p <= R; ++p)
      if (R % p == 0) return (p == 2 && R % 4 == 0 && R > 4) ? 4 : p;
    return R;
  }
  static constexpr int value = f();
};

template <typename T, int R, bool INV>
struct DFT {
  static constexpr int A = SmallestFactor<R>::value;  // outer radix
  static constexpr int B = R / A;
  __device__ __forceinline__ static void run(Cx<T> (&x)[R]) {
    if constexpr (A == R) {
      // prime radix > 5: direct O(R^2) evaluation with folded constants
      Cx<T> y[R];
#pragma unroll
      for (int k = 0; k < R; ++k) {
        Cx<T> acc = x[0];
#pragma unroll
        for (int n = 1; n < R; ++n) acc = cadd(acc, cmul(x[n], root<T, R, INV>(n * k)));
        y[k] = acc;
      }
#pragma unroll
      for (int k = 0; k < R; ++k) x[k] = y[k];
    } else {
      // Cooley-Tukey: n = n1 + A*n2, k = k2 + B*k1
      Cx<T> y[A][B];
#pragma unroll
      for (int n1 = 0; n1 < A; ++n1) {
        Cx<T> col[B];
#pragma unroll
        for (int n2 = 0; n2 < B; ++n2) col[n2] = x[n1 + A * n2];
        DFT<T, B, INV>::run(col);
#pragma unroll
        for (int k2 = 0; k2 < B; ++k2)
          y[n1][k2] = (n1 * k2 == 0) ? col[k2] : cmul(col[k2], root<T, R, INV>(n1 * k2));
      }
#pragma unroll
      for (int k2 = 0; k2 < B; ++k2) {
        Cx<T> row[A];
#pragma unroll
        for (int n1 = 0; n1 < A; ++n1) row[n1] = y[n1][k2];
        DFT<T, A, INV>::run(row);
#pragma unroll
        for (int k1 = 0; k1 < A; ++k1) x[k2 + B * k1] = row[k1];
      }
    }
  }
};

template <typename T, bool INV>
struct DFT<T, 1, INV> {
  __device__ __forceinline__ static void run(Cx<T> (&)[1]) {}
};
template <typename T, bool INV>
struct DFT<T, 2, INV> {
  __device__ __forceinline__ static void run(Cx<T> (&x)[2]) {
    Cx<T> a = x[0], b = x[1];
    x[0] = cadd(a, b);
    x[1] = csub(a, b);
  }
};
template <typename T, bool INV>
struct DFT<T, 3, INV> {
  __device__ __forceinline__ static void run(Cx<T> (&x)[3]) {
    const T c1 = (T)-0.5;
    const T s1 = (T)(INV ? 0.86602540378443864676372317075294 : -0.86602540378443864676372317075294);
    Cx<T> t1 = cadd(x[1], x[2]);
    Cx<T> t2 = csub(x[1], x[2]);
    Cx<T> m = {x[0].x + c1 * t1.x, x[0].y + c1 * t1.y};
    // s1 * i * t2
    Cx<T> r = {-s1 * t2.y, s1 * t2.x};
    x[0] = cadd(x[0], t1);
    x[1] = cadd(m, r);
    x[2] = csub(m, r);
  }
};
template <typename T, bool INV>
struct DFT<T, 4, INV> {
  __device__ __forceinline__ static void run(Cx<T> (&x)[4]) {
    Cx<T> a0 = cadd(x[0], x[2]), a1 = csub(x[0], x[2]);
    Cx<T> b0 = cadd(x[1], x[3]), b1 = rot90<T, INV>(csub(x[1], x[3]));
    x[0] = cadd(a0, b0);
    x[2] = csub(a0, b0);
    x[1] = cadd(a1, b1);
    x[3] = csub(a1, b1);
  }
};
template <typename T, bool INV>
struct DFT<T, 5, INV> {
  __device__ __forceinline__ static void run(Cx<T> (&x)[5]) {
    const T c1 = (T)0.30901699437494742410229341718282;   // cos(2pi/5)
    const T c2 = (T)-0.80901699437494742410229341718282;  // cos(4pi/5)
    const T sg = INV ? (T)1 : (T)-1;
    const T s1 = sg * (T)0.95105651629515357211643933337938;  // sin(2pi/5)
    const T s2 = sg * (T)0.58778525229247312916870595463907;  // sin(4pi/5)
    Cx<T> a1 = cadd(x[1], x[4]), b1 = csub(x[1], x[4]);
    Cx<T> a2 = cadd(x[2], x[3]), b2 = csub(x[2], x[3]);
    Cx<T> m1 = {x[0].x + c1 * a1.x + c2 * a2.x, x[0].y + c1 * a1.y + c2 * a2.y};
    Cx<T> m2 = {x[0].x + c2 * a1.x + c1 * a2.x, x[0].y + c2 * a1.y + c1 * a2.y};
    // i*(s1*b1 + s2*b2), i*(s2*b1 - s1*b2)
    Cx<T> n1 = {-(s1 * b1.y + s2 * b2.y), s1 * b1.x + s2 * b2.x};
    Cx<T> n2 = {-(s2 * b1.y - s1 * b2.y), s2 * b1.x - s1 * b2.x};
    x[0] = cadd(x[0], cadd(a1, a2));
    x[1] = cadd(m1, n1);
    x[4] = csub(m1, n1);
    x[2] = cadd(m2, n2);
    x[3] = csub(m2, n2);
  }
};

// ---------------------------------------------------------------------------
// Line plans: threads per line and the radix list for each supported N.
// ---------------------------------------------------------------------------
template <int... Rs>
struct Radices {};

// A plan is a thread count per line and a radix list.  Families (V), each the
// default of one kind of pass in one precision (default_family):
//   0 / 3  strided and spectral passes in FP32 / FP64,
//   1 / 6  contiguous directional x passes in FP32 / FP64,
//   2 / 7  complex-to-real x pass, the adjoint's r2c stage, contiguous elastic
//          and operator passes in FP32 / FP64,
//   4      complex-to-real chirp-z lines in FP32,
//   8      wide rows: strided and spectral passes in FP32 on grids larger than
//          the last-level cache (kWideFamily below),
//   9      strided and spectral chirp-z lines in FP32,
//   5      lines of the fused y-inverse / complex-to-real plane kernel.
// What bounds the passes is memory, reached with enough waves in flight: the
// directional passes carry three to five arrays of E elements per thread, so
// E <= 8 (FP64) ... 10 leaves FP32 at four waves per SIMD (159 of 222 kernels,
// three in 53) and FP64 at two or three (147 and 58) with little or no scratch.
// With 16 elements the FP64 128-point x pass spilled 796 bytes per lane and took
// 85 us on 128^3 (now 31), its strided pass 42 (20); with 8 threads per line
// (32-byte pieces of a row per load) the FP32 128-point x pass took 25 us (now
// 17).  Lengths with several primes take an uneven pass (StockhamPass) rather
// than more elements: 240 = 5 x 8 x 6 on 48 threads.  Both columns of the table
// were taken from timed sweeps of radix lists and thread counts at 8 M (FP32)
// and 4 M (FP64) voxels.
template <int N, int V = 0>
struct Plan;
#define KW_PLAN(V_, N_, TPL_, ...)                 \
  template <>                                      \
  struct Plan<N_, V_> {                            \
    static constexpr int N = N_;                   \
    static constexpr int TPL = TPL_;               \
    static constexpr int E = N_ / TPL_;            \
    using R = Radices<__VA_ARGS__>;                \
  };
// inherited families (specialised below where another plan is faster)
template <int N>
struct Plan<N, 1> : Plan<N, 0> {};
template <int N>
struct Plan<N, 2> : Plan<N, 0> {};
template <int N>
struct Plan<N, 3> : Plan<N, 0> {};
template <int N>
struct Plan<N, 4> : Plan<N, 1> {};
template <int N>
struct Plan<N, 5> : Plan<N, 2> {};
template <int N>
struct Plan<N, 6> : Plan<N, 1> {};
template <int N>
struct Plan<N, 7> : Plan<N, 3> {};
template <int N>
struct Plan<N, 8> : Plan<N, 0> {};
template <int N>
struct Plan<N, 9> : Plan<N, 0> {};

// strided and spectral passes
KW_PLAN(0, 8, 1, 8)
KW_PLAN(0, 9, 1, 9)
KW_PLAN(0, 10, 1, 10)
KW_PLAN(0, 12, 1, 12)
KW_PLAN(0, 15, 1, 15)
KW_PLAN(0, 16, 1, 16)
KW_PLAN(0, 20, 2, 10, 2)
KW_PLAN(0, 24, 2, 12, 2)
KW_PLAN(0, 25, 5, 5, 5)
KW_PLAN(0, 27, 3, 9, 3)
KW_PLAN(0, 32, 4, 8, 4)
KW_PLAN(0, 36, 3, 12, 3)
KW_PLAN(0, 40, 8, 5, 8)
KW_PLAN(0, 45, 9, 5, 9)
KW_PLAN(0, 48, 4, 12, 4)
KW_PLAN(0, 60, 12, 5, 12)
KW_PLAN(0, 64, 16, 4, 4, 4)
KW_PLAN(0, 72, 6, 12, 6)
KW_PLAN(0, 75, 15, 5, 15)
KW_PLAN(0, 80, 20, 4, 5, 4)
KW_PLAN(0, 81, 9, 9, 9)
KW_PLAN(0, 90, 18, 5, 6, 3)
KW_PLAN(0, 96, 24, 4, 6, 4)
KW_PLAN(0, 100, 10, 10, 10)
KW_PLAN(0, 108, 18, 6, 6, 3)
KW_PLAN(0, 120, 24, 5, 6, 4)
KW_PLAN(0, 125, 25, 5, 5, 5)
KW_PLAN(0, 128, 16, 8, 8, 2)
KW_PLAN(0, 135, 27, 5, 9, 3)
KW_PLAN(0, 144, 12, 12, 12)
KW_PLAN(0, 150, 30, 5, 6, 5)
KW_PLAN(0, 160, 20, 8, 5, 4)
KW_PLAN(0, 162, 27, 6, 9, 3)
KW_PLAN(0, 180, 30, 6, 6, 5)
KW_PLAN(0, 192, 24, 8, 6, 4)
KW_PLAN(0, 200, 40, 5, 8, 5)
KW_PLAN(0, 216, 36, 6, 6, 6)
KW_PLAN(0, 225, 45, 5, 9, 5)
KW_PLAN(0, 240, 48, 5, 8, 6)
KW_PLAN(0, 243, 27, 9, 9, 3)
KW_PLAN(0, 250, 50, 5, 10, 5)
KW_PLAN(0, 256, 32, 8, 8, 4)
KW_PLAN(0, 270, 45, 6, 9, 5)
KW_PLAN(0, 288, 48, 6, 8, 6)
KW_PLAN(0, 300, 60, 5, 10, 6)
KW_PLAN(0, 320, 64, 5, 8, 8)
KW_PLAN(0, 324, 54, 6, 9, 6)
KW_PLAN(0, 360, 60, 6, 10, 6)
KW_PLAN(0, 375, 25, 15, 5, 5)
KW_PLAN(0, 384, 64, 6, 8, 8)
KW_PLAN(0, 400, 50, 8, 10, 5)
KW_PLAN(0, 432, 54, 8, 9, 6)
KW_PLAN(0, 450, 50, 9, 10, 5)
KW_PLAN(0, 480, 60, 8, 10, 6)
KW_PLAN(0, 486, 54, 9, 9, 6)
KW_PLAN(0, 500, 50, 10, 10, 5)
KW_PLAN(0, 512, 64, 8, 8, 8)
KW_PLAN(0, 540, 60, 9, 10, 6)
KW_PLAN(0, 576, 48, 12, 12, 4)
KW_PLAN(0, 600, 60, 10, 10, 6)
KW_PLAN(0, 640, 80, 8, 10, 8)
KW_PLAN(0, 648, 54, 12, 9, 6)
KW_PLAN(0, 720, 60, 12, 10, 6)
KW_PLAN(0, 750, 50, 15, 10, 5)
KW_PLAN(0, 768, 64, 12, 4, 4, 4)
KW_PLAN(0, 800, 100, 8, 10, 10)
KW_PLAN(0, 864, 108, 8, 12, 9)
KW_PLAN(0, 900, 100, 9, 10, 10)
KW_PLAN(0, 960, 64, 15, 8, 8)
KW_PLAN(0, 972, 108, 9, 12, 9)
KW_PLAN(0, 1000, 100, 10, 10, 10)
KW_PLAN(0, 1024, 64, 16, 8, 8)
KW_PLAN(0, 2048, 128, 16, 16, 8)
KW_PLAN(0, 4096, 256, 16, 16, 16)
// contiguous directional passes (FP32)
KW_PLAN(1, 16, 4, 4, 4)
KW_PLAN(1, 20, 5, 4, 5)
KW_PLAN(1, 24, 6, 4, 6)
KW_PLAN(1, 32, 8, 4, 8)
KW_PLAN(1, 36, 6, 6, 6)
KW_PLAN(1, 48, 8, 6, 8)
KW_PLAN(1, 72, 12, 6, 12)
KW_PLAN(1, 90, 15, 6, 15)
KW_PLAN(1, 100, 20, 5, 5, 4)
KW_PLAN(1, 108, 12, 9, 12)
KW_PLAN(1, 120, 30, 4, 6, 5)
KW_PLAN(1, 128, 32, 4, 4, 4, 2)
KW_PLAN(1, 144, 24, 6, 6, 4)
KW_PLAN(1, 160, 32, 5, 8, 4)
KW_PLAN(1, 192, 32, 6, 8, 4)
KW_PLAN(1, 256, 64, 4, 4, 4, 4)
KW_PLAN(1, 270, 30, 9, 6, 5)
KW_PLAN(1, 500, 125, 4, 5, 5, 5)
KW_PLAN(1, 576, 72, 8, 9, 8)
KW_PLAN(1, 648, 81, 8, 9, 9)
KW_PLAN(1, 720, 90, 8, 10, 9)
KW_PLAN(1, 750, 75, 10, 15, 5)
KW_PLAN(1, 768, 96, 8, 12, 8)
KW_PLAN(1, 960, 120, 8, 12, 10)
KW_PLAN(1, 1024, 256, 4, 4, 4, 4, 4)
KW_PLAN(1, 2048, 256, 8, 8, 8, 4)
KW_PLAN(1, 4096, 512, 8, 8, 8, 8)
// wide rows
KW_PLAN(8, 256, 16, 16, 16)
KW_PLAN(8, 320, 16, 20, 4, 4)
KW_PLAN(8, 512, 32, 16, 8, 4)
KW_PLAN(8, 1024, 64, 16, 16, 4)
// strided and spectral passes (FP64)
KW_PLAN(3, 12, 4, 3, 4)
KW_PLAN(3, 15, 5, 3, 5)
KW_PLAN(3, 16, 4, 4, 4)
KW_PLAN(3, 20, 5, 4, 5)
KW_PLAN(3, 24, 6, 4, 6)
KW_PLAN(3, 32, 8, 4, 8)
KW_PLAN(3, 36, 6, 6, 6)
KW_PLAN(3, 48, 8, 6, 8)
KW_PLAN(3, 72, 12, 6, 12)
KW_PLAN(3, 108, 18, 6, 6, 3)
KW_PLAN(3, 128, 32, 4, 4, 4, 2)
KW_PLAN(3, 160, 32, 5, 8, 4)
KW_PLAN(3, 256, 64, 4, 4, 4, 4)
KW_PLAN(3, 270, 30, 9, 6, 5)
KW_PLAN(3, 300, 30, 10, 6, 5)
KW_PLAN(3, 360, 30, 12, 6, 5)
KW_PLAN(3, 375, 25, 15, 5, 5)
KW_PLAN(3, 384, 32, 12, 8, 4)
KW_PLAN(3, 432, 36, 12, 6, 6)
KW_PLAN(3, 640, 64, 10, 8, 8)
KW_PLAN(3, 720, 80, 9, 10, 8)
KW_PLAN(3, 750, 75, 10, 15, 5)
KW_PLAN(3, 768, 96, 8, 12, 8)
KW_PLAN(3, 960, 96, 10, 12, 8)
KW_PLAN(3, 1024, 128, 8, 8, 8, 2)
KW_PLAN(3, 2048, 256, 8, 8, 8, 4)
KW_PLAN(3, 4096, 512, 8, 8, 8, 8)
// contiguous directional passes (FP64)
KW_PLAN(6, 100, 25, 4, 5, 5)
KW_PLAN(6, 108, 27, 4, 9, 3)
KW_PLAN(6, 200, 50, 4, 10, 5)
KW_PLAN(6, 216, 54, 4, 9, 6)
KW_PLAN(6, 240, 30, 8, 6, 5)
KW_PLAN(6, 300, 30, 10, 6, 5)
KW_PLAN(6, 375, 75, 5, 15, 5)
KW_PLAN(6, 512, 128, 4, 4, 4, 4, 2)
KW_PLAN(6, 540, 90, 6, 10, 9)
KW_PLAN(6, 576, 64, 9, 8, 8)
KW_PLAN(6, 600, 100, 6, 10, 10)
KW_PLAN(6, 640, 64, 10, 8, 8)
KW_PLAN(6, 648, 108, 6, 12, 9)
KW_PLAN(6, 750, 125, 6, 5, 5, 5)
// contiguous elastic passes (FP32): 1024 x 256 x 64, x derivative 48.7 us on 16 x 8
// x 8, 43.6 on this chain; the complex-to-real pass the same on either (20.2, 20.0)
KW_PLAN(2, 1024, 64, 16, 16, 4)
// complex-to-real (FP64): at most 256 threads
KW_PLAN(7, 4096, 256, 16, 16, 16)
// complex-to-real chirp-z lines, which carry the chirp and filter arrays too
KW_PLAN(4, 1024, 128, 8, 8, 4, 4)
KW_PLAN(4, 2048, 256, 8, 8, 8, 4)
KW_PLAN(4, 4096, 256, 16, 16, 16)
// strided and spectral chirp-z lines (FP32): 16 elements a thread spilled 92
// registers with the chirp beside the fields (256 x 700 FP32 66.9 us a step, 53.1
// on this plan; 97 x 1013 x 64 640 and 514).  At 4096 points 16 elements stay the
// faster: 8 leave one line, rows of 8 bytes, to a workgroup of 512 threads (64 x
// 1500 x 64 512 us, 575).
KW_PLAN(9, 2048, 256, 8, 8, 8, 4)
#undef KW_PLAN

// Threads per line and radix list of a plan in one number.
template <int... Rs>
constexpr long long radix_signature(Radices<Rs...>) {
  long long s = 0;
  for (int r : {Rs...}) s = 32 * s + r;
  return s;
}
template <int N, int V>
constexpr long long plan_signature() {
  return 1024 * radix_signature(typename Plan<N, V>::R{}) + Plan<N, V>::TPL;
}

enum PassKind { kStrided, kContig, kC2R };
template <typename T>
constexpr int default_family(PassKind k, bool chirp = false) {
  if (sizeof(T) == 8) return k == kStrided ? 3 : (k == kContig ? 6 : 7);
  return k == kStrided ? (chirp ? 9 : 0) : (k == kContig ? 1 : (chirp ? 4 : 2));
}

// Line pairs per workgroup of a strided pass: the largest power of two that
// keeps the workgroup at 256 threads, but rows of at least 32 bytes where 512
// threads allow it.  Workgroups of at most 256 threads leave several of them
// on a CU, so one computes while others wait for memory or for a barrier; the
// narrow rows this gives long lines cost no bandwidth as long as neighbouring
// tiles share an L2 (xcd_wg).  Measured at 8 M FP32 voxels, strided pass: 192
// points 38 us with 8 pairs (52 with 16), 320 points 48 us with 4 (57 with 8),
// 256 points 38 us with 8 (41 us with 16 x 16 plans and 16 pairs).
//
// Grids larger than the last-level cache (large) stream every field from HBM,
// where wider rows count more than a fuller CU: rows of 128 bytes where 512
// threads allow them (512 x 512 x 256 FP32 with FP16 maps, 512-point y pass:
// 426 us with 4 pairs, 406 with 8; 256-point z pass 429 with 8, 389 with 16,
// 370 on the 16 x 16 plan of kWideFamily).  Not for lines that do not fill
// whole waves, which lose more to the barriers of larger workgroups (150-point
// z pass of 240 x 216 x 150: 53 us with 8 pairs, 62 with 16).
constexpr int strided_lines(int tpl, int elem_bytes, bool large = false) {
  int l = 1;
  while (2 * l * tpl <= 256) l *= 2;
  while (2 * l * elem_bytes < 32 && 2 * l * tpl <= 512) l *= 2;
  if (large && 64 % tpl == 0)
    while (2 * l * elem_bytes < 128 && 2 * l * tpl <= 512) l *= 2;
  return l;
}
// A grid whose `fields` arrays of n elements do not fit the last-level cache.
constexpr bool beyond_cache(int fields, long long n, int elem_bytes) {
  return (long long)fields * n * elem_bytes > (256LL << 20);
}
// On such grids the FP32 256-point strided passes and the 256-, 512- and
// 1024-point spectral passes take 16 elements per thread, which gives 128-byte
// rows to workgroups of 256 or 512 threads: 512 x 512 x 256, spectral y / z
// passes 125 / 145 us with 8 elements and 110 / 133 with 16; 256^3 35.6 / 37.5
// and 32.9 / 35.1.  The 512-point directional pass keeps 8 (406 us; 433).  The
// family's 320-point plan is for elastic passes (wide_elastic).
constexpr int kWideFamily = 8;
constexpr bool wide_strided(int n) { return n == 256; }
constexpr bool wide_spectral(int n) { return n == 256 || n == 512 || n == 1024; }
// Lines per workgroup of a contiguous pass: 256 threads where several lines
// share a wave, one line where it fills waves of its own (256^3 x pass: 120 us
// with 1, 123 with 4; 512 x 512 x 256: 490 and 506), else about 192 threads
// (240 points on 48 threads, 8 M FP32 voxels: 68 us with 4 pairs, 92 with 8).
constexpr int contig_lines(int tpl) {
  const int th = 64 % tpl == 0 ? (tpl == 64 ? 64 : 256) : (tpl % 64 == 0 ? tpl : 192);
  return th / tpl > 0 ? th / tpl : 1;
}

// LDS slice of one line: one complex of padding per 16 keeps the
// stride-16/32 Stockham writes off a single bank group, and an odd pitch keeps
// the lines of a strided pass, whose lanes run across them, on different banks
// (240 + 15 + 1 = 256 put all of them on one: strided pass 97 us instead of
// 58).  The 4096 plan is left unpadded so a double-precision line still fits a
// 64 KiB workgroup.
template <int N>
struct LdsLayout {
  static constexpr bool PAD = N >= 16 && N < 4096;
  static constexpr int PITCH = PAD ? (N + N / 16) | 1 : N;
  __device__ __forceinline__ static int at(int i) { return PAD ? i + (i >> 4) : i; }
};

// Twiddles of the passes after the first, W_N^((j mod Ns) r N/(Ns R)),
// depend only on the thread's position in the line.  For small plans they
// are loaded once per kernel into registers (all four transforms of a pass
// kernel reuse them, conjugated for the inverse); larger plans read the
// table, which stays L1-resident.
template <int... Rs>
struct RadixArray {
  static constexpr int n = sizeof...(Rs);
  static constexpr int r[n] = {Rs...};
};
template <int... Rs>
constexpr int RadixArray<Rs...>::r[];

// Butterflies of radix r that a thread of a line of n points on tpl threads
// computes: the line's n / r butterflies are dealt to the threads in turn.
constexpr int butterflies_per_thread(int n, int tpl, int r) { return (n / r + tpl - 1) / tpl; }

template <int N, int V, typename RL>
struct TwCount;
template <int N, int V, int... Rs>
struct TwCount<N, V, Radices<Rs...>> {
  static constexpr int f() {
    constexpr int rr[] = {Rs...};
    int Ns = 1, tot = 0;
    for (int i = 0; i < (int)sizeof...(Rs); ++i) {
      if (Ns > 1) tot += butterflies_per_thread(N, Plan<N, V>::TPL, rr[i]) * (rr[i] - 1);
      Ns *= rr[i];
    }
    return tot;
  }
  static constexpr int value = f();
};

template <typename T, int N, int V = 0>
struct Twiddles {
  static constexpr int TOT = TwCount<N, V, typename Plan<N, V>::R>::value;
  static constexpr bool REG = V != 5 && TOT > 0 && TOT <= 16;
  Cx<T> w[REG ? TOT : 1];
  const Cx<T>* g;
};

template <typename T, int N, int V, int TPL, int Ns, int OFF, int R, int... Rest>
struct TwLoad {
  __device__ __forceinline__ static void run(Twiddles<T, N, V>& tw, const Cx<T>* __restrict__ table, int t) {
    constexpr int NB = butterflies_per_thread(N, TPL, R);
    if constexpr (Ns > 1) {
#pragma unroll
      for (int m = 0; m < NB; ++m) {
        const int jm = (t + TPL * m) % Ns;   // in the table also for a butterfly that no thread computes
#pragma unroll
        for (int r = 1; r < R; ++r) tw.w[OFF + m * (R - 1) + (r - 1)] = table[jm * r * (N / (Ns * R))];
      }
    }
    if constexpr (sizeof...(Rest) > 0)
      TwLoad<T, N, V, TPL, Ns * R, (Ns > 1 ? OFF + NB * (R - 1) : OFF), Rest...>::run(tw, table, t);
  }
};
template <typename T, int N, int V, typename RL>
struct TwLoadImpl;
template <typename T, int N, int V, int... Rs>
struct TwLoadImpl<T, N, V, Radices<Rs...>> {
  __device__ __forceinline__ static void run(Twiddles<T, N, V>& tw, const Cx<T>* __restrict__ table, int t) {
    TwLoad<T, N, V, Plan<N, V>::TPL, 1, 0, Rs...>::run(tw, table, t);
  }
};

// Prepare the twiddles of a line of length N for thread t of the line.
template <typename T, int N, int V = 0>
__device__ __forceinline__ Twiddles<T, N, V> load_twiddles(const Cx<T>* __restrict__ table, int t) {
  Twiddles<T, N, V> tw;
  tw.g = table;
  if constexpr (Twiddles<T, N, V>::REG) TwLoadImpl<T, N, V, typename Plan<N, V>::R>::run(tw, table, t);
  return tw;
}

// LDS exchange synchronisation.  WAVE: every line of the workgroup lies within
// one wavefront (contiguous lines of TPL threads, TPL dividing 64), so the
// exchange needs only an ordering fence for the compiler and the wave's own
// in-order LDS queue, not a workgroup barrier.
template <bool WAVE>
__device__ __forceinline__ void lds_sync() {
  if constexpr (WAVE) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  } else {
    __syncthreads();
  }
}

template <typename T, int N, int V, int TPL, bool INV, int Ns, int OFF, bool WAVE, int R, int... Rest>
struct StockhamPass;
// the pass after one (void after the last)
template <typename T, int N, int V, int TPL, bool INV, int Ns, int OFF, bool WAVE, int... Rs>
struct StockhamNext {
  using type = StockhamPass<T, N, V, TPL, INV, Ns, OFF, WAVE, Rs...>;
};
template <typename T, int N, int V, int TPL, bool INV, int Ns, int OFF, bool WAVE>
struct StockhamNext<T, N, V, TPL, INV, Ns, OFF, WAVE> {
  using type = void;
};

template <typename T, int N, int V, int TPL, bool INV, int Ns, int OFF, bool WAVE, int R, int... Rest>
struct StockhamPass {
  static constexpr int E = N / TPL;
  // A radix that divides E keeps the stride-TPL layout: butterfly j of thread
  // t = j % TPL finds its inputs in the thread's registers.  Any other radix
  // (an uneven pass, never the first) takes its inputs from the exchange
  // instead, its butterflies dealt to the threads in turn, the last round not
  // full: lengths such as 240 = 15 x 16 then need 15 elements per thread and
  // two exchanges, where a radix list that divides E would need 30 or 60.
  static constexpr bool EVEN = E % R == 0;
  static constexpr int NB = butterflies_per_thread(N, TPL, R);
  static constexpr bool FULL = (N / R) % TPL == 0;   // every thread has NB butterflies
  static_assert(EVEN || Ns > 1, "the first radix must divide the per-thread element count");
  // this pass reads its twiddles from the table (plans too large to keep
  // them in registers); NW of them per thread
  static constexpr bool TAB = !Twiddles<T, N, V>::REG && Ns > 1;
  static constexpr int NW = TAB ? NB * (R - 1) : 1;
  static constexpr bool LAST = sizeof...(Rest) == 0;
  static_assert(!LAST || Ns * R == N, "radix product must equal N");
  using Next =
      typename StockhamNext<T, N, V, TPL, INV, Ns * R, (Ns > 1 ? OFF + NB * (R - 1) : OFF), WAVE, Rest...>::type;

  __device__ __forceinline__ static void fetch(Cx<T> (&w)[NW], const Twiddles<T, N, V>& tw, int t) {
    if constexpr (TAB) {
#pragma unroll
      for (int m = 0; m < NB; ++m) {
        const int jm = (t + TPL * m) % Ns;
#pragma unroll
        for (int r = 1; r < R; ++r) w[m * (R - 1) + (r - 1)] = tw.g[jm * r * (N / (Ns * R))];
      }
    }
  }
  __device__ __forceinline__ static void run(Cx<T> (&v)[E], Cx<T>* lds, const Twiddles<T, N, V>& tw, int t) {
    Cx<T> w[NW];
    fetch(w, tw, t);
    body(v, lds, tw, t, w);
  }
  // w: this pass's table twiddles, fetched by the caller.  EVEN: v holds the
  // line in the stride-TPL layout; else the line is in LDS, in order.
  __device__ __forceinline__ static void body(Cx<T> (&v)[E], Cx<T>* lds, const Twiddles<T, N, V>& tw, int t,
                                              const Cx<T> (&w)[NW]) {
    if constexpr (EVEN) {
#pragma unroll
      for (int m = 0; m < NB; ++m) {
        Cx<T> x[R];
#pragma unroll
        for (int r = 0; r < R; ++r) x[r] = v[m + r * NB];
        const int j = t + TPL * m;
        if constexpr (Ns > 1) {
#pragma unroll
          for (int r = 1; r < R; ++r) {
            Cx<T> wr;
            if constexpr (Twiddles<T, N, V>::REG)
              wr = tw.w[OFF + m * (R - 1) + (r - 1)];
            else
              wr = w[m * (R - 1) + (r - 1)];
            x[r] = INV ? cmulc(x[r], wr) : cmul(x[r], wr);
          }
        }
        DFT<T, R, INV>::run(x);
        if constexpr (LAST) {
#pragma unroll
          for (int r = 0; r < R; ++r) v[m + r * NB] = x[r];
        } else {
          const int base = (j / Ns) * Ns * R + (j % Ns);
#pragma unroll
          for (int r = 0; r < R; ++r) lds[LdsLayout<N>::at(base + r * Ns)] = x[r];
        }
      }
    } else {
      Cx<T> x[NB][R];
#pragma unroll
      for (int m = 0; m < NB; ++m) {
        const int j = t + TPL * m;
        if (FULL || j < N / R) {
#pragma unroll
          for (int r = 0; r < R; ++r) x[m][r] = lds[LdsLayout<N>::at(j + r * (N / R))];
        }
      }
      lds_sync<WAVE>();   // every input is read before the outputs replace it
#pragma unroll
      for (int m = 0; m < NB; ++m) {
        const int j = t + TPL * m;
        if (FULL || j < N / R) {
#pragma unroll
          for (int r = 1; r < R; ++r) {
            Cx<T> wr;
            if constexpr (Twiddles<T, N, V>::REG)
              wr = tw.w[OFF + m * (R - 1) + (r - 1)];
            else
              wr = w[m * (R - 1) + (r - 1)];
            x[m][r] = INV ? cmulc(x[m][r], wr) : cmul(x[m][r], wr);
          }
          DFT<T, R, INV>::run(x[m]);
          const int base = (j / Ns) * Ns * R + (j % Ns);
#pragma unroll
          for (int r = 0; r < R; ++r) lds[LdsLayout<N>::at(base + r * Ns)] = x[m][r];
        }
      }
    }
    if constexpr (!LAST) {
      // the next pass's table twiddles are requested before the exchange so
      // their latency overlaps the barrier and the LDS reads
      Cx<T> wn[Next::NW];
      Next::fetch(wn, tw, t);
      lds_sync<WAVE>();
      if constexpr (Next::EVEN) {
#pragma unroll
        for (int q = 0; q < E; ++q) v[q] = lds[LdsLayout<N>::at(t + TPL * q)];
        lds_sync<WAVE>();
      }
      Next::body(v, lds, tw, t, wn);
    } else if constexpr (!EVEN) {
      lds_sync<WAVE>();
#pragma unroll
      for (int q = 0; q < E; ++q) v[q] = lds[LdsLayout<N>::at(t + TPL * q)];
      lds_sync<WAVE>();
    }
  }
};

template <typename T, int N, int V, bool INV, bool WAVE, bool OPQ, typename RL>
struct LineFFTImpl;
template <typename T, int N, int V, bool INV, bool WAVE, bool OPQ, int... Rs>
struct LineFFTImpl<T, N, V, INV, WAVE, OPQ, Radices<Rs...>> {
  static constexpr int TPL = Plan<N, V>::TPL;
  static constexpr int E = Plan<N, V>::E;
  __device__ __forceinline__ static void run(Cx<T> (&v)[E], Cx<T>* lds, const Twiddles<T, N, V>& tw, int t) {
    // OPQ: an opaque copy of the thread index, so the address arithmetic of
    // this transform is not merged with that of the kernel's other
    // transforms (which keeps every LDS and twiddle address live across all
    // of them: fewer registers and more waves per SIMD for some kernels, more
    // address arithmetic for all).
    int tt = t;
    if constexpr (OPQ) asm volatile("" : "+v"(tt));
    StockhamPass<T, N, V, TPL, INV, 1, 0, WAVE, Rs...>::run(v, lds, tw, tt);
  }
};

// Lines of plan family V whose threads are consecutive (contiguous-line
// passes) lie inside one wavefront when TPL divides 64.
template <int N, int V>
constexpr bool wave_local_lines() {
  return 64 % Plan<N, V>::TPL == 0;
}

// Public entry: forward (INV=false) or unnormalised inverse transform of the
// line held in v (stride-TPL layout), using the line's LDS slice `lds`.
// Every thread of the workgroup must call it (it contains barriers).  WAVE:
// the caller's lines are wave-local (consecutive threads, TPL dividing 64),
// so the exchanges synchronise the wavefront only.
template <typename T, int N, bool INV, int V = 0, bool WAVE = false, bool OPQ = false>
__device__ __forceinline__ void line_fft(Cx<T> (&v)[(Plan<N, V>::E)], Cx<T>* lds, const Twiddles<T, N, V>& tw,
                                         int t) {
  static_assert(!WAVE || Plan<N, V>::TPL <= 64, "wave-local lines have at most 64 threads");
  LineFFTImpl<T, N, V, INV, WAVE, OPQ, typename Plan<N, V>::R>::run(v, lds, tw, t);
}

// ---------------------------------------------------------------------------
// Lines of any length n (Bluestein / chirp-z): the DFT of length n as a
// circular convolution on a compiled plan of length N >= 2n - 1.
//   X_k = c_k sum_j (x_j c_j) d_(k-j),  c_j = exp(-i pi j^2 / n),  d = conj(c)
//       = c_k IFFT_N( G . FFT_N(c . x) ),  G = FFT_N(g) / N
// with g_m = d_m (0 <= m < n), g_(N-m) = d_m (0 < m < n), 0 elsewhere; the
// unnormalised inverse uses conj(c) and the filter of c.  The tables are
// generated in FP64 on the host.
// ---------------------------------------------------------------------------
template <typename T>
struct Chirp {
  int n;               // logical line length
  const Cx<T>* c;      // c_j, j < n
  const Cx<T>* gf;     // N values: forward filter spectrum, 1/N folded in
  const Cx<T>* gb;     // N values: inverse filter spectrum, 1/N folded in
};

// Forward (INV=false) or unnormalised inverse DFT of a line of length ch.n held
// in v (stride-TPL layout of the N-point plan; slots j >= n hold zero on exit
// and are ignored on entry).  BS=false is the plain N-point line_fft.
template <typename T, int N, bool INV, int V = 0, bool WAVE = false, bool BS = false, bool OPQ = false>
__device__ __forceinline__ void line_dft(Cx<T> (&v)[(Plan<N, V>::E)], Cx<T>* lds, const Twiddles<T, N, V>& tw, int t,
                                         const Chirp<T>& ch) {
  if constexpr (!BS) {
    line_fft<T, N, INV, V, WAVE, OPQ>(v, lds, tw, t);
  } else {
    constexpr int TPL = Plan<N, V>::TPL, E = Plan<N, V>::E;
    const int n = ch.n;
#pragma unroll
    for (int q = 0; q < E; ++q) {
      const int j = t + TPL * q;
      v[q] = j < n ? (INV ? cmulc(v[q], ch.c[j]) : cmul(v[q], ch.c[j])) : Cx<T>{0, 0};
    }
    line_fft<T, N, false, V, WAVE, OPQ>(v, lds, tw, t);
    const Cx<T>* g = INV ? ch.gb : ch.gf;
#pragma unroll
    for (int q = 0; q < E; ++q) v[q] = cmul(v[q], g[t + TPL * q]);
    line_fft<T, N, true, V, WAVE, OPQ>(v, lds, tw, t);
#pragma unroll
    for (int q = 0; q < E; ++q) {
      const int j = t + TPL * q;
      v[q] = j < n ? (INV ? cmulc(v[q], ch.c[j]) : cmul(v[q], ch.c[j])) : Cx<T>{0, 0};
    }
  }
}

}  // namespace kw
