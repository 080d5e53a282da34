// Complex-to-real launchers for double.
#include "kw_launch.hpp"

namespace kw {

// the 256- and 512-point pass on another plan than the default
template <int N, int PV>
static hipError_t c2r_one(dim3 g, dim3 b, size_t sh, hipStream_t s, const C2RArgs<double>& a) {
  if constexpr (alternative_kernel<N, PV, default_family<double>(kC2R)>()) {
    hipLaunchKernelGGL((k_c2r_x<double, N, false, PV>), g, b, sh, s, a);
    return hipGetLastError();
  }
  return hipErrorInvalidValue;
}
template <int N>
static hipError_t c2r_alt(int pv, dim3 g, dim3 b, size_t sh, hipStream_t s, const C2RArgs<double>& a) {
  switch (pv) {
    case 0: return c2r_one<N, 0>(g, b, sh, s, a);
    case 1: return c2r_one<N, 1>(g, b, sh, s, a);
    case kWideFamily: return c2r_one<N, kWideFamily>(g, b, sh, s, a);
  }
  return hipErrorInvalidValue;
}

template <>
hipError_t launch_c2r<double>(int n, dim3 g, dim3 b, size_t sh, hipStream_t s, const C2RArgs<double>& a, int pv) {
  if (pv >= 0) {
    if (n == 256) return c2r_alt<256>(pv, g, b, sh, s, a);
    return n == 512 ? c2r_alt<512>(pv, g, b, sh, s, a) : hipErrorInvalidValue;
  }
  switch (n) {
#define X(n_)                                                      \
  case n_:                                                         \
    hipLaunchKernelGGL((k_c2r_x<double, n_>), g, b, sh, s, a);        \
    return hipGetLastError();
    KW_SIZES(X)
    KW_DIRECT_SIZES(X)
#undef X
  }
  return hipErrorInvalidValue;
}

// The FP64 plane does not fit a workgroup's registers: no fused form.
template <>
bool plane_c2r_supported<double>(int, int, size_t) {
  return false;
}

template <>
hipError_t launch_plane_c2r<double>(int, int, unsigned, hipStream_t, const PlaneArgs<double>&) {
  return hipErrorInvalidValue;
}

}  // namespace kw
