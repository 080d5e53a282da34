// Spectral-pass launchers for float.
#include "kw_launch.hpp"

namespace kw {

template <int N, typename T>
static hipError_t spec_mode(int mode, dim3 g, dim3 b, size_t sh, hipStream_t s, const SpecArgs<T>& a) {
  switch (mode) {
    case 0:
      if (a.S2)
        hipLaunchKernelGGL((k_spec_pass<T, N, 6>), g, b, sh, s, a);
      else
        hipLaunchKernelGGL((k_spec_pass<T, N, 0>), g, b, sh, s, a);
      break;
    case 1:
      hipLaunchKernelGGL((k_spec_pass<T, N, 1>), g, b, sh, s, a);
      break;
    case 2:
      if (a.S2)
        hipLaunchKernelGGL((k_spec_pass<T, N, 4>), g, b, sh, s, a);
      else
        hipLaunchKernelGGL((k_spec_pass<T, N, 2>), g, b, sh, s, a);
      break;
    case 3:
      hipLaunchKernelGGL((k_spec_pass<T, N, 3>), g, b, sh, s, a);
      break;
    case 5:
      hipLaunchKernelGGL((k_spec_pass<T, N, 5>), g, b, sh, s, a);
      break;
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// spectral passes on another plan than the default
template <int N, int PV>
static hipError_t spec_alt(dim3 g, dim3 b, size_t sh, hipStream_t s, const SpecArgs<float>& a) {
  switch (a.mode) {
    case 0:
      if (a.S2)
        hipLaunchKernelGGL((k_spec_pass<float, N, 6, false, PV>), g, b, sh, s, a);
      else
        hipLaunchKernelGGL((k_spec_pass<float, N, 0, false, PV>), g, b, sh, s, a);
      break;
    case 1:
      hipLaunchKernelGGL((k_spec_pass<float, N, 1, false, PV>), g, b, sh, s, a);
      break;
    case 2:
      if (a.S2)
        hipLaunchKernelGGL((k_spec_pass<float, N, 4, false, PV>), g, b, sh, s, a);
      else
        hipLaunchKernelGGL((k_spec_pass<float, N, 2, false, PV>), g, b, sh, s, a);
      break;
    case 3:
      hipLaunchKernelGGL((k_spec_pass<float, N, 3, false, PV>), g, b, sh, s, a);
      break;
    case 5:
      hipLaunchKernelGGL((k_spec_pass<float, N, 5, false, PV>), g, b, sh, s, a);
      break;
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
template <int N>
static hipError_t spec_alt(int pv, dim3 g, dim3 b, size_t sh, hipStream_t s, const SpecArgs<float>& a) {
  constexpr int D = default_family<float>(kStrided);
  switch (pv) {
    case 0:
      if constexpr (alternative_kernel<N, 0, D>()) return spec_alt<N, 0>(g, b, sh, s, a);
      break;
    case 1:
      if constexpr (alternative_kernel<N, 1, D>()) return spec_alt<N, 1>(g, b, sh, s, a);
      break;
    case kWideFamily: return spec_alt<N, kWideFamily>(g, b, sh, s, a);
  }
  return hipErrorInvalidValue;
}

template <>
hipError_t launch_spec<float>(int n, dim3 g, dim3 b, size_t sh, hipStream_t s, const SpecArgs<float>& a, int pv) {
  if (pv >= 0) {
    if (n == 256) return spec_alt<256>(pv, g, b, sh, s, a);
    if (n == 1024 && pv == kWideFamily) return spec_alt<1024, kWideFamily>(g, b, sh, s, a);
    return n == 512 ? spec_alt<512>(pv, g, b, sh, s, a) : hipErrorInvalidValue;
  }
  switch (n) {
#define X(n_)   \
  case n_:      \
    return spec_mode<n_, float>(a.mode, g, b, sh, s, a);
    KW_SIZES(X)
    KW_DIRECT_SIZES(X)
#undef X
  }
  return hipErrorInvalidValue;
}

}  // namespace kw
