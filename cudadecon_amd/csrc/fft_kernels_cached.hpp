// The kernels of fft_kernels_dev.hpp built to keep the spectrum in cache
// (CDN_SPEC_CACHED, fft_kernels_cached.hip); null for lengths not built in.
#pragma once

#include "fft_types.hpp"

namespace cdn {

using XR2cKernel = void(const float*, const float*, float*, const double*, int, float2*, long, long, long, const long*,
                        int, const float2*);
using XLrcoreKernel = void(float2*, const float*, long, long, const float2*, float);
using XUpdateKernel = void(const float2*, const float*, float*, float*, double*, int, long, long, const float2*);
using ColKernel = void(float2*, long, long, long, long, OtfSupport, const float2*);
using ZFilterKernel = void(float2*, long, long, long, long, long, long, int, OtfParams, const float2*);

using ColRaggedKernel = void(const ColSeg*, int, long, const float2*);
using ZRaggedKernel = void(const ZSeg*, int, long, int, const float2*);

XR2cKernel* cached_x_r2c(int n, bool ragged);
XLrcoreKernel* cached_x_lrcore(int n);
XUpdateKernel* cached_x_update(int n);
// narrow: tiles of kNarrowCols columns
ColKernel* cached_col(int n, bool inverse, bool narrow);
ZFilterKernel* cached_z_filter(int n, bool ra, bool narrow);
// one workgroup per item
ColRaggedKernel* cached_col_ragged(int n, bool inverse, bool narrow);
ZRaggedKernel* cached_z_ragged(int n, bool ra, bool narrow);

}  // namespace cdn
