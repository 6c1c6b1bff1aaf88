// Host-side declarations shared by the library's translation units.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <string>

#include "pf_fft.hpp"

namespace pf {

// Error state behind pf_last_error().
void set_error(const std::string& msg);
int fail(int code, const std::string& msg);

#define PF_HIP(call)                                                                   \
  do {                                                                                 \
    hipError_t e_ = (call);                                                            \
    if (e_ != hipSuccess)                                                              \
      return ::pf::fail(-3, std::string(#call " failed: ") + hipGetErrorString(e_) +  \
                                 " (" __FILE__ ":" + std::to_string(__LINE__) + ")"); \
  } while (0)

// Grid sizes with compiled transform kernels (every axis must be one of them).
#define PF_GRID_SIZES(X) \
  X(8) X(12) X(16) X(24) X(32) X(48) X(64) X(96) X(128) X(160) X(192) X(256) X(512)
bool grid_size_supported(int n);
const char* supported_sizes_text();

// Device table of exp(-2 pi i q/n), q in [0, n), in precision R (cached per device).
template <typename R> const c2<R>* twiddle_table(int n);

// Whole 3-D forward transforms of a batch of real fields at src: the passes run in
// the split-Nyquist layout at main, nyq
//   main: batch * (nx/2)*ny*nz complex == batch * nx*ny*nz reals (may be src)
//   nyq : batch * ny*nz complex
// and leave the spectrum there (fwd3d_split), or in the column-tile layout of the
// carried spectrum at tiled (fwd3d_tiled).
template <typename R>
int fwd3d_split(const c2<R>* src, c2<R>* main, c2<R>* nyq, int nx, int ny, int nz, int batch, R scale, hipStream_t s);
template <typename R>
int fwd3d_tiled(const c2<R>* src, c2<R>* main, c2<R>* nyq, c2<R>* tiled, int nx, int ny, int nz, int batch, R scale,
                hipStream_t s);

// Individual passes (used by the step pipelines).  x: real lines at src to half
// lines at dst and back (src == dst in place); y: nlines = panels of M columns,
// and as many Nyquist-plane lines, in one launch.
template <typename R>
int x_r2c(int nx, const c2<R>* src, c2<R>* dst, c2<R>* nyq, long nlines, R scale, hipStream_t s);
template <typename R>
int x_c2r(int nx, const c2<R>* src, c2<R>* dst, const c2<R>* nyq, long nlines, hipStream_t s);
// With the x line's plan: the bits of k_xline's own inverse x transform.
int x_c2r_as_xline(int nx, const double2* src, double2* dst, const double2* nyq, long nlines, hipStream_t s);
template <typename R>
int y_pass(int ny, bool inv, c2<R>* main, c2<R>* nyq, long M, long nlines, hipStream_t s);
// Copies between device memory and the caller's (pageable) host arrays on
// stream s; both return once the copy has finished.  Copies of 128 MiB and more
// go through two pinned bounce buffers of 64 MiB (process-wide, made on first
// use): the GPU moves one chunk while host threads move the neighbouring chunk
// between the other buffer and the caller's array.
int to_host(void* dst, const void* src, size_t bytes, hipStream_t s);
int to_device(void* dst, const void* src, size_t bytes, hipStream_t s);

}  // namespace pf
