// Directional-pass launchers for float.
#include "kw_launch.hpp"

namespace kw {

// the 256- and 512-point passes on another plan than the default
template <int N, int PV>
static hipError_t dir_alt(bool contig, dim3 g, dim3 b, size_t sh, hipStream_t s, const PassArgs<float>& a,
                          const RecArgs<float>& r, unsigned tiles) {
  if (contig) {
    if constexpr (alternative_kernel<N, PV, default_family<float>(kContig)>()) {
      if (a.S2)
        hipLaunchKernelGGL((k_dir_pass<float, N, true, true, false, PV>), g, b, sh, s, a, r, tiles);
      else
        hipLaunchKernelGGL((k_dir_pass<float, N, true, false, false, PV>), g, b, sh, s, a, r, tiles);
      return hipGetLastError();
    }
  } else if constexpr (alternative_kernel<N, PV, default_family<float>(kStrided)>()) {
    hipLaunchKernelGGL((k_dir_pass<float, N, false, false, false, PV>), g, b, sh, s, a, r, tiles);
    return hipGetLastError();
  }
  return hipErrorInvalidValue;
}
template <int N>
static hipError_t dir_alt(int pv, bool contig, dim3 g, dim3 b, size_t sh, hipStream_t s, const PassArgs<float>& a,
                          const RecArgs<float>& r, unsigned tiles) {
  switch (pv) {
    case 0: return dir_alt<N, 0>(contig, g, b, sh, s, a, r, tiles);
    case 1: return dir_alt<N, 1>(contig, g, b, sh, s, a, r, tiles);
    case kWideFamily: return dir_alt<N, kWideFamily>(contig, g, b, sh, s, a, r, tiles);
  }
  return hipErrorInvalidValue;
}

template <>
hipError_t launch_dir<float>(int n, bool contig, dim3 g, dim3 b, size_t sh, hipStream_t s, const PassArgs<float>& a,
                           int pv, const RecArgs<float>* rec) {
  const unsigned tiles = g.x;
  const RecArgs<float> r = rec ? *rec : RecArgs<float>{};
  if (rec && !contig) g.x += ((unsigned)r.n + b.x - 1) / b.x;
  if (pv >= 0) {
    if (n == 256) return dir_alt<256>(pv, contig, g, b, sh, s, a, r, tiles);
    return n == 512 ? dir_alt<512>(pv, contig, g, b, sh, s, a, r, tiles) : hipErrorInvalidValue;
  }
  switch (n) {
#define X(n_)                                                                  \
  case n_:                                                                     \
    if (contig && a.S2)                                                        \
      hipLaunchKernelGGL((k_dir_pass<float, n_, true, true>), g, b, sh, s, a, r, tiles);  \
    else if (contig)                                                           \
      hipLaunchKernelGGL((k_dir_pass<float, n_, true, false>), g, b, sh, s, a, r, tiles); \
    else                                                                       \
      hipLaunchKernelGGL((k_dir_pass<float, n_, false>), g, b, sh, s, a, r, tiles);       \
    return hipGetLastError();
    KW_SIZES(X)
    KW_DIRECT_SIZES(X)
#undef X
  }
  return hipErrorInvalidValue;
}

}  // namespace kw
