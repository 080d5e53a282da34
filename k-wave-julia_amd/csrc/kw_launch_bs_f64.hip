// Launchers of the any-length (Bluestein) line passes for double: a line of
// length n runs on the plan n_plan >= 2n - 1 (kw_fft.hpp line_dft).
#include "kw_launch.hpp"

namespace kw {

template <>
hipError_t launch_dir_bs<double>(int n_plan, bool contig, dim3 g, dim3 b, size_t sh, hipStream_t s,
                               const PassArgs<double>& a, const RecArgs<double>* rec) {
  const unsigned tiles = g.x;
  const RecArgs<double> r = rec ? *rec : RecArgs<double>{};
  if (rec && !contig) g.x += ((unsigned)r.n + b.x - 1) / b.x;
  switch (n_plan) {
#define X(n_)                                                                          \
  case n_:                                                                             \
    if (contig && a.S2)                                                                \
      hipLaunchKernelGGL((k_dir_pass<double, n_, true, true, true>), g, b, sh, s, a, r, tiles);      \
    else if (contig)                                                                   \
      hipLaunchKernelGGL((k_dir_pass<double, n_, true, false, true>), g, b, sh, s, a, r, tiles);     \
    else                                                                               \
      hipLaunchKernelGGL((k_dir_pass<double, n_, false, false, true>), g, b, sh, s, a, r, tiles);    \
    return hipGetLastError();
    KW_BS_SIZES(X)
#undef X
  }
  return hipErrorInvalidValue;
}

template <int N>
static hipError_t spec_mode_bs(int mode, dim3 g, dim3 b, size_t sh, hipStream_t s, const SpecArgs<double>& a) {
  switch (mode) {
    case 0:
      if (a.S2)
        hipLaunchKernelGGL((k_spec_pass<double, N, 6, true>), g, b, sh, s, a);
      else
        hipLaunchKernelGGL((k_spec_pass<double, N, 0, true>), g, b, sh, s, a);
      break;
    case 1:
      hipLaunchKernelGGL((k_spec_pass<double, N, 1, true>), g, b, sh, s, a);
      break;
    case 2:
      if (a.S2)
        hipLaunchKernelGGL((k_spec_pass<double, N, 4, true>), g, b, sh, s, a);
      else
        hipLaunchKernelGGL((k_spec_pass<double, N, 2, true>), g, b, sh, s, a);
      break;
    case 3:
      hipLaunchKernelGGL((k_spec_pass<double, N, 3, true>), g, b, sh, s, a);
      break;
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <>
hipError_t launch_spec_bs<double>(int n_plan, dim3 g, dim3 b, size_t sh, hipStream_t s, const SpecArgs<double>& a) {
  switch (n_plan) {
#define X(n_)   \
  case n_:      \
    return spec_mode_bs<n_>(a.mode, g, b, sh, s, a);
    KW_BS_SIZES(X)
#undef X
  }
  return hipErrorInvalidValue;
}

template <>
hipError_t launch_c2r_bs<double>(int n_plan, dim3 g, dim3 b, size_t sh, hipStream_t s, const C2RArgs<double>& a) {
  switch (n_plan) {
#define X(n_)                                                       \
  case n_:                                                          \
    hipLaunchKernelGGL((k_c2r_x<double, n_, true>), g, b, sh, s, a);    \
    return hipGetLastError();
    KW_BS_SIZES(X)
#undef X
  }
  return hipErrorInvalidValue;
}

}  // namespace kw
