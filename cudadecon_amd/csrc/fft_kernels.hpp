// Host-side launch interface of the 3-D FFT pass kernels (fft_kernels.hip).
//
// Volume layout: real (nz, ny, nx), x fastest, no padding.  Half spectrum:
// (nz, ny, nx/2+1) complex64 with row pitch `pitch` >= nx/2+1 (padded to a
// multiple of 16 so column tiles start on 128-byte boundaries).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "fft_types.hpp"
#include "jit.hpp"

namespace cdn {

// Length is compiled in, or can be compiled at run time (2,3,5,7-smooth).
bool fft_length_supported(int n);
// Length is among the lengths built into the library.
bool fft_length_precompiled(int n);
// Compile the kernels of a length that is not precompiled (no-op otherwise);
// throws with the compiler log on failure.  Needs no GPU.
void fft_prepare_length(int n);
// Twiddle table for a supported length (host, FP64-derived float2 values).
int fft_twiddle_count(int n);
void fft_twiddles(int n, float2* out);

// Whether an iteration's passes should keep a spectrum of `bytes` in the
// memory-side cache (256 MB): `cached` of the launchers below, which then run
// the kernels that access it with cached instructions (real volumes stream as
// before; lengths without built-in kernels ignore it unless tuned).  Each
// pass then finds the spectrum where the one before left it.  ms per iteration,
// streaming -> cached: 64 x 512 x 512 (69 MB) 0.329 -> 0.306, 128 x 512 x 512
// (138 MB) 0.567 -> 0.517, 64 x 768 x 768 (151 MB) 0.687 -> 0.595, 192 x 512 x 512
// (208 MB) 0.853 -> 0.786, 48 stacks of 64 x 128 x 128 (252 MB) 0.884 -> 0.777; 24
// uneven stacks in one graph (156 MB) 0.96 -> 0.87.  At the lower edge: 36 MB
// 0.188 -> 0.175 (64 x 256 x 512) and 38 MB 0.187 -> 0.168 (128 x 256 x 256); 27 MB
// would still gain (0.162 -> 0.148 at 64 x 256 x 384), 19 MB loses (0.119 -> 0.128 at
// 64 x 256 x 256).  At the upper edge 285 MB would gain 2 to 4% (1.091 -> 1.064 at
// 256 x 512 x 512), 314 MB and more lose 1 to 2% (96 x 1024 x 768, 192 x 512 x 810).
// Engines side by side, whose spectra together exceed the cache, lose nothing by
// it (iterations of 8 of 71 MB on 4 streams 2.14 -> 2.12, 16 of 36 MB on 16 2.25 ->
// 2.13, 4 of 138 MB on 2 2.09 -> 2.04).
constexpr bool spec_cached(size_t bytes) { return bytes >= (32UL << 20) && bytes <= (256UL << 20); }

// R2C along x of row pairs with the prediction fused in; writes S.  Rows
// come in stacks of stack_rows (even; 0: one stack), stack s using the
// factor lam[4 s]; or, with row_starts (device, nstk ascending even rows,
// the first 0), in stacks of different heights.
void launch_x_r2c(int nx, hipStream_t st, const float* X, const float* Xp, float* Y, const double* lam,
                  int mode, float2* S, long rows, long pitch, const float2* tw, long stack_rows = 0,
                  const long* row_starts = nullptr, int nstk = 0, bool cached = false);
// plain C2R along x (ignores imag of kx = 0 and kx = nx/2).
void launch_x_c2r(int nx, hipStream_t st, const float2* S, float* out, long rows, long pitch,
                  const float2* tw);
// C2R along x -> LRcore with raw -> R2C along x, in place on S.
void launch_x_lrcore(int nx, hipStream_t st, float2* S, const float* raw, long rows, long pitch,
                     const float2* tw, float eps, bool cached = false);
// C2R along x -> X = max(C Y, 0), G_new = X - Y written over G; if dots:
// per-block partial sums of G_new.G_old and G_old.G_old (FP32 products,
// FP64 sums) into part[2*block..].  Returns the number of blocks launched.
int launch_x_update(int nx, hipStream_t st, const float2* S, const float* Y, float* Xout, float* G,
                    double* part, int dots, long rows, long pitch, const float2* tw, bool cached = false);
int x_update_blocks(int nx, long rows);
// rows per x-update workgroup of the launch shape in use for nx
long x_update_rows_per_block(int nx);
// upper bound of x_update_blocks over every launch shape (one row pair per block)
int x_update_blocks_max(long rows);

// Tuned launch shapes: a length with a variant runs that variant's run-time
// compiled kernels (results are bitwise those of the default shapes).
void fft_set_variant(int n, const FftVariant& v);
// One column tile of all `ncols` columns of length `len` when they would
// need two built-in tiles, the second a quarter full or less, and the tile
// fits (v: the variant); the column launchers use it unless the length has
// a tuned variant.
bool fft_balanced_cols(int len, long ncols, FftVariant* v);
// compile and load the kernels those launches will need (no GPU work); z: as
// a z filter of planes line_stride apart, else as a y transform
void fft_prepare_cols(int len, long ncols, long line_stride, bool z);
bool fft_get_variant(int n, FftVariant* v);
// What the passes of a grid run: the spectrum kept in cache, tiles of 16
// columns in the y passes and in the z filter.
struct GridFlavours {
  bool cached = false, y_narrow = false, z_narrow = false;
};
GridFlavours grid_flavours(int nx, int ny, int nz, long nxh, long pitch, int nstacks = 1);
// a column variant as a launch of such a grid compiles it
FftVariant fft_column_flavour(int len, const FftVariant& v, bool narrow, bool cached);
// compile and load what the tuned variants of a grid's lengths will launch (no
// GPU work; before any stream capture); x: of one x length
void fft_prepare_variants(int nx, int ny, int nz, long nxh, long pitch, int nstacks);
void fft_prepare_x_variant(int nx, bool cached);
// While one exists on this thread, every launch uses the built-in kernels of
// its length: no tuned or single-tile variant, whose run-time compiled code
// would have to be loaded (column results are bitwise the same).
struct BuiltinShapesOnly {
  BuiltinShapesOnly();
  ~BuiltinShapesOnly();
};
void fft_clear_variants();
// While one exists on this thread, launches take the kernels with 64-bit
// addresses whatever the stack's size (a pass with a support bound keeps its
// buffers): the tests compare both on small stacks.
struct WideAddresses {
  WideAddresses();
  ~WideAddresses();
  WideAddresses(const WideAddresses&) = delete;
};

// a bound that no column exceeds
constexpr OtfSupport kNoSupport{-1.f, 0.f, 0.f};

// Column FFT (forward or inverse) over `len` points at element stride
// line_stride, for columns [0, ncols) of each of n_outer slabs.  sup: for the
// y transforms around a z filter, the support of its OTF (the rows outside it
// are not stored by the forward and taken as zero by the inverse transform).
void launch_col_fft(int len, int inverse, hipStream_t st, float2* S, long ncols, long line_stride,
                    long outer_stride, long n_outer, const float2* tw, const OtfSupport& sup = kNoSupport,
                    bool cached = false);
// z forward -> x H (or conj H) / N -> z inverse; slab index = ky, for
// nstacks spectra stack_stride complex elements apart.
void launch_z_filter(int nz, hipStream_t st, float2* S, long ncols, long line_stride, long outer_stride,
                     long ny, int conj, const OtfParams& otf, const float2* tw, int nstacks = 1,
                     long stack_stride = 0, bool cached = false);

// Column passes spanning stacks of different shapes: one launch for every
// stack whose transform length is `len`, segs (device) one per stack with
// items numbered by tiles of `cols` columns (y_tile_cols / z_tile_cols of the
// launch's largest column count), `total` items in all.  grid_cap > 0 bounds the workgroups, which then walk the items.
long y_tile_cols(int len, long ncols);
long z_tile_cols(int len, long ncols);
// compile and load the run-time kernels the ragged launches of a length not
// built in will use (no GPU work; call before any stream capture); buf as
// launch_z_ragged's
void fft_prepare_ragged(int len, bool buf = true);
void launch_col_ragged(int len, int inverse, hipStream_t st, const ColSeg* segs, int nseg, long total,
                       long cols, const float2* tw, long grid_cap = 0, bool cached = false);
// ra: every segment's OTF is rotationally averaged (the kernel kind the
// one-stack z filter uses for such a table)
void launch_z_ragged(int nz, hipStream_t st, const ZSeg* segs, int nseg, long total, long cols, int conj,
                     const float2* tw, long grid_cap = 0, bool ra = false, bool buf = true,
                     bool cached = false);
// whether a stack's z filter can address its planes (line_stride apart) by
// 32-bit offsets: buf above, for every segment of the launch
bool z_ragged_buf(int nz, long line_stride);

}  // namespace cdn
