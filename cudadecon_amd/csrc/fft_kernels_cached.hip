// The FFT pass kernels with cached spectrum accesses (fft_kernels_cached.hpp).
#define CDN_SPEC_CACHED 1
#include "common.hpp"
#include "fft_kernels_dev.hpp"
#include "fft_kernels_cached.hpp"

namespace cdn {

#define CDN_PICK(LENGTHS, EXPR) \
  switch (n) {                  \
    LENGTHS(EXPR)               \
    default:                    \
      return nullptr;           \
  }

XR2cKernel* cached_x_r2c(int n, bool ragged) {
#define CDN_CASE(N) \
  case N:           \
    return ragged ? k_x_r2c<N, true> : k_x_r2c<N, false>;
  CDN_PICK(CDN_FFT_LENGTHS, CDN_CASE)
#undef CDN_CASE
}

XLrcoreKernel* cached_x_lrcore(int n) {
#define CDN_CASE(N) \
  case N:           \
    return k_x_lrcore<N>;
  CDN_PICK(CDN_FFT_LENGTHS, CDN_CASE)
#undef CDN_CASE
}

XUpdateKernel* cached_x_update(int n) {
#define CDN_CASE(N) \
  case N:           \
    return k_x_update<N>;
  CDN_PICK(CDN_FFT_LENGTHS, CDN_CASE)
#undef CDN_CASE
}

ColKernel* cached_col(int n, bool inverse, bool narrow) {
  if (narrow) {
#define CDN_CASE(N) \
  case N:           \
    return inverse ? k_col<N, true, true, kNarrowCols> : k_col<N, false, true, kNarrowCols>;
    CDN_PICK(CDN_NARROW_Y_LENGTHS, CDN_CASE)
#undef CDN_CASE
  }
#define CDN_CASE(N) \
  case N:           \
    return inverse ? k_col<N, true, true> : k_col<N, false, true>;
  CDN_PICK(CDN_FFT_LENGTHS, CDN_CASE)
#undef CDN_CASE
}

ZFilterKernel* cached_z_filter(int n, bool ra, bool narrow) {
  if (narrow) {
#define CDN_CASE(N) \
  case N:           \
    return ra ? k_z_filter<N, ZF_RA, true, kNarrowCols> : k_z_filter<N, ZF_ANY, zf_buf(N, ZF_ANY), kNarrowCols>;
    CDN_PICK(CDN_NARROW_LENGTHS, CDN_CASE)
#undef CDN_CASE
  }
#define CDN_CASE(N) \
  case N:           \
    return ra ? k_z_filter<N, ZF_RA> : k_z_filter<N, ZF_ANY>;
  CDN_PICK(CDN_FFT_LENGTHS, CDN_CASE)
#undef CDN_CASE
}

ColRaggedKernel* cached_col_ragged(int n, bool inverse, bool narrow) {
  if (narrow) {
#define CDN_CASE(N) \
  case N:           \
    return inverse ? k_col_ragged<N, true, false, kNarrowCols> : k_col_ragged<N, false, false, kNarrowCols>;
    CDN_PICK(CDN_NARROW_LENGTHS, CDN_CASE)
#undef CDN_CASE
  }
#define CDN_CASE(N) \
  case N:           \
    return inverse ? k_col_ragged<N, true, false> : k_col_ragged<N, false, false>;
  CDN_PICK(CDN_FFT_LENGTHS, CDN_CASE)
#undef CDN_CASE
}

ZRaggedKernel* cached_z_ragged(int n, bool ra, bool narrow) {
  if (narrow) {
#define CDN_CASE(N) \
  case N:           \
    return ra ? k_z_ragged<N, false, ZF_RA, true, kNarrowCols>    \
              : k_z_ragged<N, false, ZF_ANY, zf_buf(N, ZF_ANY), kNarrowCols>;
    CDN_PICK(CDN_NARROW_LENGTHS, CDN_CASE)
#undef CDN_CASE
  }
#define CDN_CASE(N) \
  case N:           \
    return ra ? k_z_ragged<N, false, ZF_RA> : k_z_ragged<N, false, ZF_ANY>;
  CDN_PICK(CDN_FFT_LENGTHS, CDN_CASE)
#undef CDN_CASE
}

}  // namespace cdn
