// The whole time loop of a 1-D simulation in one workgroup.
//
// A 1-D step is one line: as separate launches (x pass, complex-to-real pass,
// sensor gather) it took 14.2 us for 512 FP64 points, nearly all of it launch
// latency and reloading a few kilobytes.  Here one workgroup of one line's
// threads keeps p, u, rho and the medium in registers and runs many steps per
// launch; per step only the derivative and equation-of-state tables, the source
// values and the recorded samples touch memory: 6.9 us.  What bounds it is the
// serial chain of six line transforms on one CU; lines take the contiguous
// passes' plans (with the strided passes' 64 x 8 plan, whose line is one wave's
// and needs no barrier: 7.1 us).  The equation of state runs as a full complex
// transform of the real line: M is real and even in k, so the result is the
// half-spectrum one.
#pragma once

#include "kw_kernels.hpp"

namespace kw {

template <typename T>
struct Line1dArgs {
  PassArgs<T> x;           // the x pass's arguments (fields, medium, tables, sources)
  T* p;
  const T* M1;             // equation-of-state multipliers, index |k| (1/N folded in)
  const T* M2;             // second spectrum (:stokes) or null
  RecArgs<T> rec;          // rec.n = 0: nothing recorded
  const long long* tr_idx; // time reversal: rho[tr_idx[j]] = tr_vals[tr_n (Nt - t) + j] before a step
  const T* tr_vals;
  int tr_n;
  int Nt;
  int t0;                  // 1-based index of the first step of this launch
  int nsteps;
};

// LDS: the line's exchange slice, then p and u of the line for the recorder.
template <typename T, int N>
constexpr size_t line1d_lds() {
  return (size_t)LdsLayout<N>::PITCH * sizeof(Cx<T>) + 2 * (size_t)N * sizeof(T);
}
template <typename T>
constexpr int kLineFamily = default_family<T>(kContig);
constexpr bool line1d_wave(int tpl) { return tpl <= 64; }

// values written at the line positions pos[e] & 0xFFFFF, e < count (added to, or
// in place of, what r holds), through the exchange slice
template <typename T, int N, int V, bool BS, bool WAVE, typename F>
__device__ __forceinline__ void line1d_scatter(T (&r)[(Plan<N, V>::E)], T* buf, int t, int nl, int count, F put) {
  constexpr int TPL = Plan<N, V>::TPL, E = Plan<N, V>::E;
#pragma unroll
  for (int q = 0; q < E; ++q)
    if (!BS || t + TPL * q < nl) buf[t + TPL * q] = r[q];
  lds_sync<WAVE>();
  for (int e = t; e < count; e += TPL) put(buf, e);
  lds_sync<WAVE>();
#pragma unroll
  for (int q = 0; q < E; ++q)
    if (!BS || t + TPL * q < nl) r[q] = buf[t + TPL * q];
  lds_sync<WAVE>();
}

template <typename T, int N, bool BS>
__global__ void __launch_bounds__((Plan<N, kLineFamily<T>>::TPL)) k_line1d(Line1dArgs<T> a) {
  constexpr int V = kLineFamily<T>;
  constexpr int TPL = Plan<N, V>::TPL, E = Plan<N, V>::E;
  constexpr bool WAVE = line1d_wave(TPL);
  extern __shared__ __align__(16) unsigned char smem_raw[];
  Cx<T>* lds = reinterpret_cast<Cx<T>*>(smem_raw);
  T* buf = reinterpret_cast<T*>(smem_raw);                       // scatter: the exchange slice
  T* lp = reinterpret_cast<T*>(lds + LdsLayout<N>::PITCH);       // recorder: p and u of the line
  T* lu = lp + N;
  const int t = threadIdx.x;
  const int nl = BS ? a.x.nl : N;
  const PassArgs<T>& x = a.x;
  const Twiddles<T, N, V> tw = load_twiddles<T, N, V>(x.tw, t);
  auto ok = [&](int q) { return !BS || t + TPL * q < nl; };

  T p[E], u[E], rho[E], prev[E], r0[E], rdt[E], c2[E], ba[E], sg[E], pl[E];
#pragma unroll
  for (int q = 0; q < E; ++q) {
    const int n = t + TPL * q, nn = n + 1 == nl ? 0 : n + 1;
    p[q] = u[q] = rho[q] = prev[q] = ba[q] = sg[q] = pl[q] = (T)0;
    r0[q] = rdt[q] = c2[q] = (T)1;
    if (!ok(q)) continue;
    p[q] = a.p[n];
    u[q] = x.u[n];
    rho[q] = x.rho[n];
    if (a.M2) prev[q] = x.rho_prev[n];
    auto map = [&](const void* f, int i, T off) {
      return x.maps_f16 ? off + (T)__half2float(reinterpret_cast<const __half*>(f)[i]) : reinterpret_cast<const T*>(f)[i];
    };
    r0[q] = x.rho0 ? map(x.rho0, n, x.rho0_off) : x.rho0_s;
    rdt[q] = x.rho0 ? fdiv(x.dt, (r0[q] + map(x.rho0, nn, x.rho0_off)) * (T)0.5) : x.dt / x.rho0_s;
    if (x.c0sq) {
      c2[q] = map(x.c0sq, n, x.c0_off);
      if (x.maps_f16) c2[q] *= c2[q];
    }
    ba[q] = x.bona ? x.bona[n] : x.bona_s;
    sg[q] = x.pml_sg[n];
    pl[q] = x.pml[n];
  }
  const bool two = a.M2 != nullptr, nonlinear = x.nonlinear != 0;
  const bool rec_u = records_u(a.rec.rec);
  auto eff = [&](T r, int q) { return nonlinear ? r * ((T)1 + ba[q] / (T)2 * fdiv(r, r0[q])) : r; };
  auto source = [&](const SrcList& s, T (&r)[E], int step) {
    if (s.off == nullptr) return;
    const int e0 = s.off[0], col = (step < s.ncols ? step : s.ncols) - 1;
    const T* vals = reinterpret_cast<const T*>(s.val) + (long long)col * s.n_src;
    line1d_scatter<T, N, V, BS, WAVE>(r, buf, t, nl, s.off[1] - e0, [&](T* b, int e) {
      const int n = s.pos[e0 + e] & 0xFFFFF;
      const T val = vals[s.row[e0 + e]];
      b[n] = s.dirichlet ? val : b[n] + val;
    });
  };

#pragma unroll 1
  for (int k = 0; k < a.nsteps; ++k) {
    const int step = a.t0 + k;
    if (a.tr_n > 0) {
      const T* vals = a.tr_vals + (long long)(a.Nt - step) * a.tr_n;
      line1d_scatter<T, N, V, BS, WAVE>(rho, buf, t, nl, a.tr_n, [&](T* b, int e) { b[a.tr_idx[e]] = vals[e]; });
    }
    Cx<T> v[E];
    T acc[E];   // pressure of the first spectrum
#pragma unroll
    for (int q = 0; q < E; ++q) v[q] = Cx<T>{ok(q) ? p[q] : (T)0, (T)0};
    // phase 0: dp/dx -> u;  1: du/dx -> rho, equation-of-state input;
    // 2: M1 spectrum -> p;  3 (:stokes): M2 spectrum added to p
#pragma unroll 1
    for (int ph = 0; ph < (two ? 4 : 3); ++ph) {
      // the phase's multipliers arrive under the forward transform
      Cx<T> m[E];
      if (ph < 2) {
        const Cx<T>* __restrict__ D = ph == 0 ? x.Dp : x.Dm;
#pragma unroll
        for (int q = 0; q < E; ++q) m[q] = ok(q) ? D[t + TPL * q] : Cx<T>{(T)0, (T)0};
      } else {
        const T* __restrict__ M = ph == 2 ? a.M1 : a.M2;
#pragma unroll
        for (int q = 0; q < E; ++q) {
          const int n = t + TPL * q, kk = n > nl - n ? nl - n : n;
          m[q] = Cx<T>{ok(q) ? M[kk] : (T)0, (T)0};
        }
      }
      line_dft<T, N, false, V, WAVE, BS, true>(v, lds, tw, t, x.ch);
      if (ph < 2) {
#pragma unroll
        for (int q = 0; q < E; ++q) v[q] = cmul(v[q], m[q]);
      } else {
#pragma unroll
        for (int q = 0; q < E; ++q) v[q] = cscale(v[q], m[q].x);
      }
      line_dft<T, N, true, V, WAVE, BS, true>(v, lds, tw, t, x.ch);
      if (ph == 0) {
#pragma unroll
        for (int q = 0; q < E; ++q) u[q] = sg[q] * (sg[q] * u[q] - rdt[q] * v[q].x);
        source(x.usrc, u, step);
#pragma unroll
        for (int q = 0; q < E; ++q) v[q] = Cx<T>{ok(q) ? u[q] : (T)0, (T)0};
      } else if (ph == 1) {
#pragma unroll
        for (int q = 0; q < E; ++q) rho[q] = pl[q] * (pl[q] * rho[q] - x.dt * r0[q] * v[q].x);
        source(x.psrc, rho, step);
#pragma unroll
        for (int q = 0; q < E; ++q) v[q] = Cx<T>{ok(q) ? eff(rho[q], q) * c2[q] : (T)0, (T)0};
      } else if (ph == 2) {
#pragma unroll
        for (int q = 0; q < E; ++q) {
          acc[q] = v[q].x;
          if (two) {
            v[q] = Cx<T>{ok(q) ? (eff(rho[q], q) - eff(prev[q], q)) * x.inv_dt : (T)0, (T)0};
            prev[q] = rho[q];
          }
        }
      } else {
#pragma unroll
        for (int q = 0; q < E; ++q) acc[q] += v[q].x;
      }
    }
#pragma unroll
    for (int q = 0; q < E; ++q) p[q] = ok(q) ? acc[q] : (T)0;
    if (a.rec.n > 0) {
#pragma unroll
      for (int q = 0; q < E; ++q)
        if (ok(q)) {
          lp[t + TPL * q] = p[q];
          if (rec_u) lu[t + TPL * q] = u[q];
        }
      lds_sync<WAVE>();
      for (int j = t; j < a.rec.n; j += TPL) {
        const long long i = a.rec.idx ? a.rec.idx[j] : (long long)j;   // null: every voxel, in order
        const T uv[3] = {rec_u ? lu[i] : (T)0, (T)0, (T)0};
        record_values<T>(a.rec, j, step, lp[i], uv, 1);
      }
      lds_sync<WAVE>();
    }
  }
#pragma unroll
  for (int q = 0; q < E; ++q) {
    const int n = t + TPL * q;
    if (!ok(q)) continue;
    a.p[n] = p[q];
    x.u[n] = u[q];
    x.rho[n] = rho[q];
    if (a.M2) x.rho_prev[n] = prev[q];
  }
}

// n: a length of its own plan, or (bs) the chirp-z plan length
template <typename T>
hipError_t launch_line1d(int n, bool bs, hipStream_t s, const Line1dArgs<T>& a);
// LDS that launch needs; 0 where n has no plan
template <typename T>
size_t line1d_lds_bytes(int n);

}  // namespace kw
