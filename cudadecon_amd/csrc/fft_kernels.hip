// Host launchers of the FFT pass kernels: precompiled lengths dispatch to
// template instantiations; any other 2,3,5,7-smooth length runs the same
// kernels compiled at run time (jit.cpp).
#include "common.hpp"
#include "fft_kernels_dev.hpp"
#include "fft_kernels.hpp"
#include "fft_kernels_cached.hpp"
#include "jit.hpp"

#include <algorithm>
#include <cmath>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace cdn {

// ---------------------------------------------------------------------------
// host side: length dispatch
// ---------------------------------------------------------------------------
bool fft_length_precompiled(int n) {
  switch (n) {
#define CDN_CASE(N) \
  case N:           \
    return true;
    CDN_FFT_LENGTHS(CDN_CASE)
#undef CDN_CASE
    default:
      return false;
  }
}

bool fft_length_supported(int n) { return fft_length_precompiled(n) || jit_length_ok(n); }

void fft_prepare_length(int n) {
  if (!fft_length_precompiled(n)) jit_prepare(n);
}

static Plan host_plan(int n) {
  const Plan P = make_plan(n);
  if (!P.ok || n < 1) fail("FFT length " + std::to_string(n) + " is not 2,3,5,7-smooth");
  return P;
}

int fft_twiddle_count(int n) {
  const Plan P = host_plan(n);
  return P.twsize > 0 ? P.twsize : 1;
}

void fft_twiddles(int n, float2* out) {
  const Plan P = host_plan(n);
  out[0] = make_float2(1.f, 0.f);
  for (int s = 0; s < P.ns; ++s) {
    const int R = P.r[s], lp = P.lp[s];
    if (lp == 1) continue;
    for (int k = 0; k < lp; ++k)
      for (int t = 1; t < R; ++t) {
        // exp(-2 pi i t k / (lp R)) in long double, reduced by integer modulus
        const long M = (long)lp * R;
        const long m = ((long)t * k) % M;
        const long double a = -2.0L * 3.14159265358979323846264338327950288L * (long double)m / (long double)M;
        out[P.twoff[s] + k * (R - 1) + (t - 1)] = make_float2((float)cosl(a), (float)sinl(a));
      }
  }
}

static inline unsigned grid1(long n) {
  if (n <= 0) return 0;
  if (n > 0x7fffffffL) fail("grid too large");
  return (unsigned)n;
}

// ---------------------------------------------------------------------------
// Tuned launch shapes per length (set by the autotuner).  A length with a
// variant always runs that variant's run-time compiled kernels.
// ---------------------------------------------------------------------------
namespace {
std::mutex g_vmu;
std::map<int, FftVariant> g_variants;
thread_local int t_builtin_only = 0;  // > 0: no run-time compiled variant
thread_local int t_wide = 0;          // > 0: 64-bit addresses
}  // namespace

BuiltinShapesOnly::BuiltinShapesOnly() { ++t_builtin_only; }
BuiltinShapesOnly::~BuiltinShapesOnly() { --t_builtin_only; }
WideAddresses::WideAddresses() { ++t_wide; }
WideAddresses::~WideAddresses() { --t_wide; }

void fft_set_variant(int n, const FftVariant& v) {
  std::lock_guard<std::mutex> lk(g_vmu);
  if (v.is_default())
    g_variants.erase(n);
  else
    g_variants[n] = v;
}
bool fft_get_variant(int n, FftVariant* v) {
  if (t_builtin_only > 0) return false;
  std::lock_guard<std::mutex> lk(g_vmu);
  auto it = g_variants.find(n);
  if (it == g_variants.end()) return false;
  if (v) *v = it->second;
  return true;
}
void fft_clear_variants() {
  std::lock_guard<std::mutex> lk(g_vmu);
  g_variants.clear();
}

// The tuned variant that shapes an x pass of length nx.  A variant that shapes
// only the column passes of its length leaves the x passes their built-in
// kernels (and their cached build).
static bool x_variant(int nx, FftVariant* v, bool cached = false) {
  if (!fft_get_variant(nx, v) || v->xthreads <= 0) return false;
  v->cached = cached;
  return true;
}

#define CDN_LAUNCH(kernel, N, grid, block, ...) \
  hipLaunchKernelGGL(kernel<N>, dim3(grid), dim3(block), 0, st, __VA_ARGS__)

void launch_x_r2c(int nx, hipStream_t st, const float* X, const float* Xp, float* Y, const double* lam, int mode,
                  float2* S, long rows, long pitch, const float2* tw, long stack_rows, const long* row_starts,
                  int nstk, bool cached) {
  FftVariant tv;
  const bool tuned = x_variant(nx, &tv, cached);
  const XShape xs = x_shape(nx, tuned ? tv.xthreads : -1, XK_R2C);
  const unsigned grid = grid1(((rows + 1) / 2 + xs.NL - 1) / xs.NL);
  if (stack_rows <= 0) stack_rows = rows;
  if (stack_rows != rows && stack_rows % 2) fail("launch_x_r2c: rows per stack must be even");
  const bool ragged = row_starts != nullptr;
  if (ragged && nstk < 1) fail("launch_x_r2c: no stacks");
  const JitKernel jk = ragged ? JK_X_R2C_RAGGED : JK_X_R2C;
  void* args[] = {&X, &Xp, &Y, &lam, &mode, &S, &rows, &pitch, &stack_rows, &row_starts, &nstk, &tw};
  if (tuned) {
    jit_launch(nx, jk, grid, xs.THREADS, st, args, tv);
  } else if (auto* k = cached ? cached_x_r2c(nx, ragged) : nullptr) {
    hipLaunchKernelGGL(k, dim3(grid), dim3(xs.THREADS), 0, st, X, Xp, Y, lam, mode, S, rows, pitch, stack_rows,
                       row_starts, nstk, tw);
  } else {
    switch (nx) {
#define CDN_CASE(N)                                                                                            \
  case N:                                                                                                      \
    if (ragged)                                                                                                \
      hipLaunchKernelGGL((k_x_r2c<N, true>), dim3(grid), dim3(xs.THREADS), 0, st, X, Xp, Y, lam, mode, S, rows, \
                         pitch, stack_rows, row_starts, nstk, tw);                                             \
    else                                                                                                       \
      hipLaunchKernelGGL((k_x_r2c<N, false>), dim3(grid), dim3(xs.THREADS), 0, st, X, Xp, Y, lam, mode, S,      \
                         rows, pitch, stack_rows, row_starts, nstk, tw);                                       \
    break;
      CDN_FFT_LENGTHS(CDN_CASE)
#undef CDN_CASE
      default:
        jit_launch(nx, jk, grid, xs.THREADS, st, args);
    }
  }
  CDN_HIP(hipGetLastError());
}

void launch_x_c2r(int nx, hipStream_t st, const float2* S, float* out, long rows, long pitch, const float2* tw) {
  FftVariant tv;
  const bool tuned = x_variant(nx, &tv);
  const XShape xs = x_shape(nx, tuned ? tv.xthreads : -1);
  const unsigned grid = grid1(((rows + 1) / 2 + xs.NL - 1) / xs.NL);
  void* args[] = {&S, &out, &rows, &pitch, &tw};
  if (tuned) {
    jit_launch(nx, JK_X_C2R, grid, xs.THREADS, st, args, tv);
  } else {
    switch (nx) {
#define CDN_CASE(N)                                                      \
  case N:                                                                \
    CDN_LAUNCH(k_x_c2r, N, grid, xs.THREADS, S, out, rows, pitch, tw); \
    break;
      CDN_FFT_LENGTHS(CDN_CASE)
#undef CDN_CASE
      default:
        jit_launch(nx, JK_X_C2R, grid, xs.THREADS, st, args);
    }
  }
  CDN_HIP(hipGetLastError());
}

void launch_x_lrcore(int nx, hipStream_t st, float2* S, const float* raw, long rows, long pitch, const float2* tw,
                     float eps, bool cached) {
  FftVariant tv;
  const bool tuned = x_variant(nx, &tv, cached);
  const XShape xs = x_shape(nx, tuned ? tv.xthreads : -1, XK_LR);
  const unsigned grid = grid1(((rows + 1) / 2 + xs.NL - 1) / xs.NL);
  void* args[] = {&S, &raw, &rows, &pitch, &tw, &eps};
  if (tuned) {
    jit_launch(nx, JK_X_LRCORE, grid, xs.THREADS, st, args, tv);
  } else if (auto* k = cached ? cached_x_lrcore(nx) : nullptr) {
    hipLaunchKernelGGL(k, dim3(grid), dim3(xs.THREADS), 0, st, S, raw, rows, pitch, tw, eps);
  } else {
    switch (nx) {
#define CDN_CASE(N)                                                              \
  case N:                                                                        \
    CDN_LAUNCH(k_x_lrcore, N, grid, xs.THREADS, S, raw, rows, pitch, tw, eps); \
    break;
      CDN_FFT_LENGTHS(CDN_CASE)
#undef CDN_CASE
      default:
        jit_launch(nx, JK_X_LRCORE, grid, xs.THREADS, st, args);
    }
  }
  CDN_HIP(hipGetLastError());
}

int x_update_blocks(int nx, long rows) {
  FftVariant tv;
  const bool tuned = x_variant(nx, &tv);
  const XShape xs = x_shape(nx, tuned ? tv.xthreads : -1);
  return (int)(((rows + 1) / 2 + xs.NL - 1) / xs.NL);
}

int x_update_blocks_max(long rows) { return (int)((rows + 1) / 2); }

long x_update_rows_per_block(int nx) {
  FftVariant tv;
  const bool tuned = x_variant(nx, &tv);
  return 2L * x_shape(nx, tuned ? tv.xthreads : -1).NL;
}

int launch_x_update(int nx, hipStream_t st, const float2* S, const float* Y, float* Xout, float* G, double* part,
                    int dots, long rows, long pitch, const float2* tw, bool cached) {
  FftVariant tv;
  const bool tuned = x_variant(nx, &tv, cached);
  const XShape xs = x_shape(nx, tuned ? tv.xthreads : -1);
  const int nb = (int)(((rows + 1) / 2 + xs.NL - 1) / xs.NL);
  void* args[] = {&S, &Y, &Xout, &G, &part, &dots, &rows, &pitch, &tw};
  if (tuned) {
    jit_launch(nx, JK_X_UPDATE, grid1(nb), xs.THREADS, st, args, tv);
  } else if (auto* k = cached ? cached_x_update(nx) : nullptr) {
    hipLaunchKernelGGL(k, dim3(grid1(nb)), dim3(xs.THREADS), 0, st, S, Y, Xout, G, part, dots, rows, pitch, tw);
  } else {
    switch (nx) {
#define CDN_CASE(N)                                                                                        \
  case N:                                                                                                  \
    CDN_LAUNCH(k_x_update, N, grid1(nb), xs.THREADS, S, Y, Xout, G, part, dots, rows, pitch, tw);        \
    break;
      CDN_FFT_LENGTHS(CDN_CASE)
#undef CDN_CASE
      default:
        jit_launch(nx, JK_X_UPDATE, grid1(nb), xs.THREADS, st, args);
    }
  }
  CDN_HIP(hipGetLastError());
  return nb;
}

// Column tiles: when a slab's columns need two built-in tiles, the second
// one a quarter or less full (65 columns of a 128 x 128 plane in tiles of
// 64), one tile holding all of them instead, if it fits (threads <= 1024,
// LDS within the built-in budget class): a run-time compiled variant,
// bitwise the same results.  (Measured: 8% on stacks of 64 x 128 x 128; a
// wider single tile, 129 columns for 3 built-in tiles, was slower.)
bool fft_balanced_cols(int len, long ncols, FftVariant* v) {
  if (t_builtin_only > 0) return false;
  const CShape d = c_shape(len);
  if (ncols <= d.L || ncols >= 2 * d.L || 4 * (ncols - d.L) > d.L) return false;
  const long budget = len >= 768 ? 160L * 1024 : 80L * 1024;
  if (ncols * c_shape(len, 1).TPT > 1024 || (long)len * ncols * 8 > budget) return false;
  if (v) {
    *v = FftVariant();
    v->cols = (int)ncols;
  }
  return true;
}

// Tiles of 16 columns (128-byte rows) instead of 32 or 64, built for lengths
// 64, 128 and 256.  Up to 160 columns they leave less of the last tile empty
// (65 columns: 80 instead of 96 or 128), cut the support's edge finer and give
// more, smaller workgroups; with more columns the y passes of 64 and 256 still
// gain, while the z filters lose the longer rows of their far-apart planes.
// ms per launch, wide -> 16: z filter of 64, 65 columns (48 stacks of
// 64 x 128 x 128) 0.107 -> 0.095, 129 columns 0.0157 -> 0.0151, 513 columns
// 0.102 -> 0.106; of 128, 129 columns 0.0212 -> 0.0196, 257 columns 0.0502 ->
// 0.0518; of 256, 129 columns 0.0355 -> 0.0334, 513 columns 0.354 -> 0.384;
// y of 256, 1025 columns 0.072 -> 0.066, 129 columns 0.0136 -> 0.0119; y of
// 128, 65 columns 0.077 -> 0.074, 513 columns 0.0442 -> 0.0450; y of 64 0.0259
// -> 0.0253 at 513 columns.  Lengths 96 and 192 (24 elements per thread, 64
// threads in such a tile): z 0.0166 -> 0.0173.
//
// 2048-point y columns run 8 to a tile (64-byte rows); 16 of them with 64
// threads and 32 elements each (one workgroup per CU) read whole 128-byte
// lines: 0.693 -> 0.632 ms at 96 x 2048 x 2048, 0.180 -> 0.177 at
// 64 x 2048 x 768 (1600 workgroups), but 0.0425 -> 0.0477 at 32 x 2048 x 256 (288
// workgroups, a second round of 32), so from 4 rounds of 256 workgroups on.
constexpr long kNarrowMax = 160;
// slabs: of the launch (planes)
static bool y_narrow(int len, long ncols, long slabs) {
  if (len == 2048) return (ncols + kNarrowCols - 1) / kNarrowCols * slabs >= 1024;
  return len == 64 || len == 256 || (len == 128 && ncols <= kNarrowMax);
}
static bool z_narrow(int len, long ncols) {
  return (len == 64 || len == 128 || len == 256) && ncols <= kNarrowMax;
}

// How a column pass runs: the tuned variant of the length, else narrow tiles,
// else one tile of all columns, else the length's own shape.  A variant that
// leaves the tile's shape alone (loads, renumbering, OTF rows) runs narrow
// tiles where the built-in kernels do, and every tuned variant the build that
// keeps the spectrum in cache where they do.
struct ColRun {
  CShape cs;
  bool jit, narrow;
  FftVariant v;
};
static FftVariant col_flavour(FftVariant v, int len, bool narrow, bool cached) {
  if (narrow && v.cols == 0 && v.col_tpt == 0) {
    v.cols = kNarrowCols;
    if (c_shape(len, kNarrowCols).TPT != c_shape(len).TPT) v.col_tpt = c_shape(len, kNarrowCols).TPT;
  }
  v.cached = cached;
  return v;
}
static ColRun col_run(int len, long ncols, bool narrow, bool cached) {
  ColRun r{};
  r.jit = fft_get_variant(len, &r.v) && r.v.shapes_cols();
  r.narrow = !r.jit && narrow;
  if (r.jit)
    r.v = col_flavour(r.v, len, narrow, cached);
  else
    r.v = FftVariant();
  if (!r.jit && !r.narrow) r.jit = fft_balanced_cols(len, ncols, &r.v);
  r.cs = r.narrow ? c_shape(len, kNarrowCols) : c_shape(len, r.jit ? r.v.cols : -1, r.jit ? r.v.col_tpt : -1);
  return r;
}

// the z filter's buffers (TPT planes each) take 32-bit offsets
static bool z_buf(const CShape& cs, long line_stride) {
  return t_wide == 0 && (double)cs.TPT * (double)line_stride * 8.0 < 2147483648.0;
}
bool z_ragged_buf(int nz, long line_stride) { return z_buf(c_shape(nz), line_stride); }

static bool z_runs_narrow(int nz, long ncols, long line_stride) {
  return z_narrow(nz, ncols) && z_buf(c_shape(nz), line_stride);
}
static ColRun z_run(int nz, long ncols, long line_stride, bool cached) {
  return col_run(nz, ncols, z_runs_narrow(nz, ncols, line_stride), cached);
}
// a slab's rows by 32-bit offsets (always the case for y transforms: at most
// 16384 rows of 8208 columns)
static bool col_buf32(int len, long line_stride) { return (double)len * (double)line_stride * 8.0 < 2147483648.0; }
static bool col_runs_narrow(int len, long ncols, long line_stride, long n_outer) {
  return col_buf32(len, line_stride) && y_narrow(len, ncols, n_outer);
}

void fft_prepare_cols(int len, long ncols, long line_stride, bool z) {
  FftVariant v;
  // compile and load (grid 0: no launch) before any stream capture
  if (!(fft_get_variant(len, &v) && v.shapes_cols()) && !(z ? z_narrow(len, ncols) : y_narrow(len, ncols, 1)) &&
      fft_balanced_cols(len, ncols, &v))
    for (JitKernel k : {JK_COL_F, JK_COL_I, JK_Z_FILTER, JK_Z_FILTER_RA})
      jit_launch(len, k, 0, 1, nullptr, nullptr, v);
  if (!z) return;
  const ColRun run = z_run(len, ncols, line_stride, false);
  if (!z_buf(run.cs, line_stride) && (run.jit || !fft_length_precompiled(len)))
    for (JitKernel k : {JK_Z_FILTER_W, JK_Z_FILTER_RA_W}) jit_launch(len, k, 0, 1, nullptr, nullptr, run.v);
}

GridFlavours grid_flavours(int nx, int ny, int nz, long nxh, long pitch, int nstacks) {
  GridFlavours f;
  f.cached = spec_cached(sizeof(float2) * (size_t)pitch * ny * nz * nstacks);
  f.y_narrow = col_runs_narrow(ny, nxh, pitch, (long)nz * nstacks);
  f.z_narrow = z_runs_narrow(nz, nxh, (long)ny * pitch);
  return f;
}
FftVariant fft_column_flavour(int len, const FftVariant& v, bool narrow, bool cached) {
  return col_flavour(v, len, narrow, cached);
}

void fft_prepare_variants(int nx, int ny, int nz, long nxh, long pitch, int nstacks) {
  FftVariant v;
  const bool any_x = x_variant(nx, &v);
  const bool any_y = fft_get_variant(ny, &v) && v.shapes_cols(), any_z = fft_get_variant(nz, &v) && v.shapes_cols();
  if (!any_x && !any_y && !any_z) return;
  const GridFlavours f = grid_flavours(nx, ny, nz, nxh, pitch, nstacks);
  if (any_x && x_variant(nx, &v, f.cached)) jit_launch(nx, JK_X_R2C, 0, 1, nullptr, nullptr, v);
  if (any_y) jit_launch(ny, JK_COL_F, 0, 1, nullptr, nullptr, col_run(ny, nxh, f.y_narrow, f.cached).v);
  if (any_z) jit_launch(nz, JK_Z_FILTER, 0, 1, nullptr, nullptr, col_run(nz, nxh, f.z_narrow, f.cached).v);
}
void fft_prepare_x_variant(int nx, bool cached) {
  FftVariant v;
  if (x_variant(nx, &v, cached)) jit_launch(nx, JK_X_R2C, 0, 1, nullptr, nullptr, v);
}

void launch_col_fft(int len, int inverse, hipStream_t st, float2* S, long ncols, long line_stride,
                    long outer_stride, long n_outer, const float2* tw, const OtfSupport& sup, bool cached) {
  const bool buf = col_buf32(len, line_stride) && !(t_wide > 0 && sup.r2 < 0.f);
  const ColRun run = col_run(len, ncols, buf && col_runs_narrow(len, ncols, line_stride, n_outer), cached);
  const CShape cs = run.cs;
  long ntiles = (ncols + cs.L - 1) / cs.L;
  const unsigned grid = grid1(ntiles * n_outer);
  OtfSupport sp = sup;
  if (!buf && sp.r2 >= 0.f) fail("launch_col_fft: support bound on a slab of 2 GiB or more");
  void* args[] = {&S, &ncols, &line_stride, &outer_stride, &ntiles, &sp, &tw};
  const JitKernel jk = inverse ? (buf ? JK_COL_I : JK_COL_IW) : (buf ? JK_COL_F : JK_COL_FW);
  if (run.jit) {
    jit_launch(len, jk, grid, cs.THREADS, st, args, run.v);
  } else if (auto* k = cached && buf ? cached_col(len, inverse != 0, run.narrow) : nullptr) {
    hipLaunchKernelGGL(k, dim3(grid), dim3(cs.THREADS), 0, st, S, ncols, line_stride, outer_stride, ntiles, sp, tw);
  } else if (run.narrow) {
    switch (len) {
#define CDN_CASE(N)                                                                                                  \
  case N: {                                                                                                          \
    auto* k = inverse ? k_col<N, true, true, kNarrowCols> : k_col<N, false, true, kNarrowCols>;                      \
    hipLaunchKernelGGL(k, dim3(grid), dim3(cs.THREADS), 0, st, S, ncols, line_stride, outer_stride, ntiles, sp, tw); \
    break;                                                                                                           \
  }
      CDN_NARROW_Y_LENGTHS(CDN_CASE)
#undef CDN_CASE
    }
  } else {
    switch (len) {
#define CDN_CASE(N)                                                                                                  \
  case N: {                                                                                                          \
    auto* k = inverse ? (buf ? k_col<N, true, true> : k_col<N, true, false>)                                         \
                      : (buf ? k_col<N, false, true> : k_col<N, false, false>);                                      \
    hipLaunchKernelGGL(k, dim3(grid), dim3(cs.THREADS), 0, st, S, ncols, line_stride, outer_stride, ntiles, sp, tw); \
    break;                                                                                                           \
  }
      CDN_FFT_LENGTHS(CDN_CASE)
#undef CDN_CASE
      default:
        jit_launch(len, jk, grid, cs.THREADS, st, args);
    }
  }
  CDN_HIP(hipGetLastError());
}

void launch_z_filter(int nz, hipStream_t st, float2* S, long ncols, long line_stride, long outer_stride, long ny,
                     int conj, const OtfParams& otf, const float2* tw, int nstacks, long stack_stride, bool cached) {
  const ColRun run = z_run(nz, ncols, line_stride, cached);
  const CShape cs = run.cs;
  long ntiles = (ncols + cs.L - 1) / cs.L;
  if (nstacks < 1) fail("launch_z_filter: no stacks");
  const unsigned grid = grid1(ntiles * ny * nstacks);
  OtfParams op = otf;
  void* args[] = {&S, &ncols, &line_stride, &outer_stride, &ntiles, &ny, &stack_stride, &conj, &op, &tw};
  // the averaged-table kind for a rotationally averaged OTF
  const bool ra = op.ra != 0, buf = z_buf(cs, line_stride);
  const JitKernel jk = ra ? (buf ? JK_Z_FILTER_RA : JK_Z_FILTER_RA_W) : (buf ? JK_Z_FILTER : JK_Z_FILTER_W);
  if (run.jit) {
    jit_launch(nz, jk, grid, cs.THREADS, st, args, run.v);
  } else if (auto* k = cached && buf ? cached_z_filter(nz, ra, run.narrow) : nullptr) {
    hipLaunchKernelGGL(k, dim3(grid), dim3(cs.THREADS), 0, st, S, ncols, line_stride, outer_stride, ntiles, ny,
                       stack_stride, conj, op, tw);
  } else if (run.narrow) {
    switch (nz) {
#define CDN_CASE(N)                                                                                             \
  case N: {                                                                                                     \
    auto* k = ra ? k_z_filter<N, ZF_RA, true, kNarrowCols>                                                      \
                 : k_z_filter<N, ZF_ANY, zf_buf(N, ZF_ANY), kNarrowCols>;                                       \
    hipLaunchKernelGGL(k, dim3(grid), dim3(cs.THREADS), 0, st, S, ncols, line_stride, outer_stride, ntiles, ny, \
                       stack_stride, conj, op, tw);                                                             \
    break;                                                                                                      \
  }
      CDN_NARROW_LENGTHS(CDN_CASE)
#undef CDN_CASE
    }
  } else {
    switch (nz) {
#define CDN_CASE(N)                                                                                             \
  case N: {                                                                                                     \
    auto* k = ra ? (buf ? k_z_filter<N, ZF_RA> : k_z_filter<N, ZF_RA, false>)                                   \
                 : (buf ? k_z_filter<N, ZF_ANY> : k_z_filter<N, ZF_ANY, false>);                                \
    hipLaunchKernelGGL(k, dim3(grid), dim3(cs.THREADS), 0, st, S, ncols, line_stride, outer_stride, ntiles, ny, \
                       stack_stride, conj, op, tw);                                                             \
    break;                                                                                                      \
  }
      CDN_FFT_LENGTHS(CDN_CASE)
#undef CDN_CASE
      default:
        jit_launch(nz, jk, grid, cs.THREADS, st, args);
    }
  }
  CDN_HIP(hipGetLastError());
}

// (of many stacks: 2048-point columns in their own width)
long y_tile_cols(int len, long ncols) { return y_narrow(len, ncols, 0) ? kNarrowCols : c_shape(len).L; }
long z_tile_cols(int len, long ncols) { return z_narrow(len, ncols) ? kNarrowCols : c_shape(len).L; }

void fft_prepare_ragged(int len, bool buf) {
  if (fft_length_precompiled(len)) return;
  if (!buf)
    for (JitKernel k : {JK_Z_RAGGED_W, JK_Z_RAGGED_RA_W}) jit_launch(len, k, 0, 1, nullptr, nullptr);
  for (JitKernel k : {JK_X_R2C_RAGGED, JK_COL_RAGGED_F, JK_COL_RAGGED_I, JK_Z_RAGGED, JK_COL_RAGGED_FP,
                      JK_COL_RAGGED_IP, JK_Z_RAGGED_P, JK_Z_RAGGED_RA, JK_Z_RAGGED_P_RA, JK_X_C2R, JK_X_LRCORE,
                      JK_X_UPDATE})
    jit_launch(len, k, 0, 1, nullptr, nullptr);
}

// grid of a launch over `total` items: one workgroup per item, or at most
// `cap` workgroups (a multiple of 8) that walk the items
static unsigned ragged_grid(long total, long cap) {
  if (cap > 0 && cap < total) return grid1(std::max(8L, cap / 8 * 8));
  return grid1(total);
}

// the kernel instance for (inverse, persistent)
template <int N, int COLS>
static auto col_ragged_n(bool inv, bool pers) {
  return inv ? (pers ? k_col_ragged<N, true, true, COLS> : k_col_ragged<N, true, false, COLS>)
             : (pers ? k_col_ragged<N, false, true, COLS> : k_col_ragged<N, false, false, COLS>);
}

void launch_col_ragged(int len, int inverse, hipStream_t st, const ColSeg* segs, int nseg, long total, long cols,
                       const float2* tw, long grid_cap, bool cached) {
  if (total <= 0) return;
  const bool narrow = cols != c_shape(len).L;
  const CShape cs = c_shape(len, narrow ? (int)cols : -1);
  const unsigned grid = ragged_grid(total, grid_cap);
  const bool inv = inverse != 0, pers = grid < total;
  void* args[] = {&segs, &nseg, &total, &tw};
  ColRaggedKernel* k = cached && !pers ? cached_col_ragged(len, inv, narrow) : nullptr;
  if (k) {
  } else if (narrow) {
    switch (len) {
#define CDN_CASE(N) \
  case N: k = col_ragged_n<N, kNarrowCols>(inv, pers); break;
      CDN_NARROW_LENGTHS(CDN_CASE)
#undef CDN_CASE
    }
    if (!k || cols != kNarrowCols) fail("launch_col_ragged: no tile of " + std::to_string(cols) + " columns");
  } else {
    switch (len) {
#define CDN_CASE(N) \
  case N: k = col_ragged_n<N, 0>(inv, pers); break;
      CDN_FFT_LENGTHS(CDN_CASE)
#undef CDN_CASE
    }
  }
  if (k)
    hipLaunchKernelGGL(k, dim3(grid), dim3(cs.THREADS), 0, st, segs, nseg, total, tw);
  else
    jit_launch(len, pers ? (inv ? JK_COL_RAGGED_IP : JK_COL_RAGGED_FP) : (inv ? JK_COL_RAGGED_I : JK_COL_RAGGED_F),
               grid, cs.THREADS, st, args);
  CDN_HIP(hipGetLastError());
}

// the kernel instance for (persistent, kind, buffer addressing); stacks that
// need 64-bit addresses fill the GPU one item per workgroup
template <int N, int COLS>
static auto z_ragged_n(bool pers, bool ra, bool buf) {
  if (COLS == 0 && !buf) return ra ? k_z_ragged<N, false, ZF_RA, false> : k_z_ragged<N, false, ZF_ANY, false>;
  constexpr bool B = zf_buf(N, ZF_ANY);
  return pers ? (ra ? k_z_ragged<N, true, ZF_RA, true, COLS> : k_z_ragged<N, true, ZF_ANY, B, COLS>)
              : (ra ? k_z_ragged<N, false, ZF_RA, true, COLS> : k_z_ragged<N, false, ZF_ANY, B, COLS>);
}

void launch_z_ragged(int nz, hipStream_t st, const ZSeg* segs, int nseg, long total, long cols, int conj,
                     const float2* tw, long grid_cap, bool ra, bool buf, bool cached) {
  if (total <= 0) return;
  const bool narrow = cols != c_shape(nz).L;
  const CShape cs = c_shape(nz, narrow ? (int)cols : -1);
  const unsigned grid = ragged_grid(total, buf ? grid_cap : 0);
  const bool pers = grid < total;
  void* args[] = {&segs, &nseg, &total, &conj, &tw};
  ZRaggedKernel* k = cached && buf && !pers ? cached_z_ragged(nz, ra, narrow) : nullptr;
  if (k) {
  } else if (narrow) {
    switch (nz) {
#define CDN_CASE(N) \
  case N: k = z_ragged_n<N, kNarrowCols>(pers, ra, true); break;
      CDN_NARROW_LENGTHS(CDN_CASE)
#undef CDN_CASE
    }
    if (!k || !buf || cols != kNarrowCols)
      fail("launch_z_ragged: no tile of " + std::to_string(cols) + " columns");
  } else {
    switch (nz) {
#define CDN_CASE(N) \
  case N: k = z_ragged_n<N, 0>(pers, ra, buf); break;
      CDN_FFT_LENGTHS(CDN_CASE)
#undef CDN_CASE
    }
  }
  if (k) {
    hipLaunchKernelGGL(k, dim3(grid), dim3(cs.THREADS), 0, st, segs, nseg, total, conj, tw);
  } else {
    const JitKernel b[4] = {JK_Z_RAGGED, JK_Z_RAGGED_P, JK_Z_RAGGED_RA, JK_Z_RAGGED_P_RA};
    const JitKernel w[2] = {JK_Z_RAGGED_W, JK_Z_RAGGED_RA_W};
    jit_launch(nz, buf ? b[2 * ra + pers] : w[ra], grid, cs.THREADS, st, args);
  }
  CDN_HIP(hipGetLastError());
}

}  // namespace cdn
