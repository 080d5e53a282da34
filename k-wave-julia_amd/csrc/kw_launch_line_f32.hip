// Launchers of the single-workgroup 1-D time loop for float.
#include "kw_launch.hpp"
#include "kw_line1d.hpp"

namespace kw {

template <int N, bool BS>
static hipError_t line_one(hipStream_t s, const Line1dArgs<float>& a) {
  hipLaunchKernelGGL((k_line1d<float, N, BS>), dim3(1), dim3(Plan<N, kLineFamily<float>>::TPL),
                     (line1d_lds<float, N>()), s, a);
  return hipGetLastError();
}

template <>
hipError_t launch_line1d<float>(int n, bool bs, hipStream_t s, const Line1dArgs<float>& a) {
  if (bs) switch (n) {
#define X(n_) \
  case n_:    \
    return line_one<n_, true>(s, a);
      KW_BS_SIZES(X)
#undef X
      default:
        return hipErrorInvalidValue;
    }
  switch (n) {
#define X(n_) \
  case n_:    \
    return line_one<n_, false>(s, a);
    KW_SIZES(X)
    KW_DIRECT_SIZES(X)
#undef X
  }
  return hipErrorInvalidValue;
}

template <>
size_t line1d_lds_bytes<float>(int n) {
  switch (n) {
#define X(n_) \
  case n_:    \
    return line1d_lds<float, n_>();
    KW_SIZES(X)
    KW_DIRECT_SIZES(X)
#undef X
  }
  return 0;
}

}  // namespace kw
