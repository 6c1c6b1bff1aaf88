// 3-D real<->half-complex transforms on gfx950: twiddle tables, size dispatch,
// whole-transform drivers, layout packing and the transform entry points of the
// C-ABI (pf_fft_r2c / pf_fft_c2r on device buffers, pf_f_trans / pf_inv_trans
// on host buffers with the reference's f_trans / inv_trans semantics).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <memory>
#include <string>
#include <mutex>
#include <thread>
#include <vector>

#include "../../include/pf.h"
#include "pf_internal.hpp"
#include "pf_passes.hpp"

namespace pf {

bool grid_size_supported(int n) {
  switch (n) {
#define PF_CASE(N) case N:
    PF_GRID_SIZES(PF_CASE)
#undef PF_CASE
    return true;
    default: return false;
  }
}
const char* supported_sizes_text() { return "8 12 16 24 32 48 64 96 128 160 192 256 512"; }

// ---------------------------------------------------------------------------
// Host transfers through pinned bounce buffers.
// ---------------------------------------------------------------------------

namespace {
constexpr size_t kBounceBytes = size_t(64) << 20;
constexpr size_t kBounceMin = size_t(128) << 20;
std::mutex g_bounce_mu;
void* g_bounce[2] = {nullptr, nullptr};

// memcpy split over up to 8 host threads
void par_copy(void* dst, const void* src, size_t n) {
  const int nth = (int)std::max(1u, std::min<unsigned>(8, std::thread::hardware_concurrency()));
  if (nth == 1 || n < (size_t(4) << 20)) {
    std::memcpy(dst, src, n);
    return;
  }
  const size_t per = (n + nth - 1) / nth;
  std::vector<std::thread> th;
  for (int w = 0; w < nth; ++w) {
    const size_t a = std::min(n, per * w), b = std::min(n, a + per);
    if (a < b) th.emplace_back([=] { std::memcpy((char*)dst + a, (const char*)src + a, b - a); });
  }
  for (auto& t : th) t.join();
}

// Under g_bounce_mu.  Pinned memory is allocated once and kept until exit.
bool bounce_ready() {
  for (int i = 0; i < 2; ++i)
    if (!g_bounce[i] && hipHostMalloc(&g_bounce[i], kBounceBytes, hipHostMallocDefault) != hipSuccess) {
      g_bounce[i] = nullptr;
      (void)hipGetLastError();
      return false;
    }
  return true;
}

struct EventPair {
  hipEvent_t e[2] = {nullptr, nullptr};
  bool ok = true;
  EventPair() {
    for (auto& x : e)
      if (hipEventCreateWithFlags(&x, hipEventDisableTiming) != hipSuccess) ok = false;
  }
  ~EventPair() {
    for (auto& x : e)
      if (x) (void)hipEventDestroy(x);
  }
};
}  // namespace

namespace {
// Under g_bounce_mu.
int to_host_locked(void* dst, const void* src, size_t bytes, hipStream_t s) {
  EventPair ev;
  if (bytes < kBounceMin || !ev.ok || !bounce_ready()) {
    PF_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s));
    PF_HIP(hipStreamSynchronize(s));
    return 0;
  }
  const size_t nch = (bytes + kBounceBytes - 1) / kBounceBytes;
  // chunk k goes into buffer k & 1; chunk k - 2 was moved out of it on the host
  // in the previous iteration
  for (size_t k = 0; k <= nch; ++k) {
    if (k < nch) {
      const size_t off = k * kBounceBytes, len = std::min(kBounceBytes, bytes - off);
      PF_HIP(hipMemcpyAsync(g_bounce[k & 1], (const char*)src + off, len, hipMemcpyDeviceToHost, s));
      PF_HIP(hipEventRecord(ev.e[k & 1], s));
    }
    if (k > 0) {
      const size_t j = k - 1, off = j * kBounceBytes, len = std::min(kBounceBytes, bytes - off);
      PF_HIP(hipEventSynchronize(ev.e[j & 1]));
      par_copy((char*)dst + off, g_bounce[j & 1], len);
    }
  }
  return 0;
}

int to_device_locked(void* dst, const void* src, size_t bytes, hipStream_t s) {
  EventPair ev;
  if (bytes < kBounceMin || !ev.ok || !bounce_ready()) {
    PF_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s));
    PF_HIP(hipStreamSynchronize(s));
    return 0;
  }
  const size_t nch = (bytes + kBounceBytes - 1) / kBounceBytes;
  for (size_t k = 0; k < nch; ++k) {
    const size_t off = k * kBounceBytes, len = std::min(kBounceBytes, bytes - off);
    // buffer k & 1 is free once the copy of chunk k - 2 out of it has finished
    if (k >= 2) PF_HIP(hipEventSynchronize(ev.e[k & 1]));
    par_copy(g_bounce[k & 1], (const char*)src + off, len);
    PF_HIP(hipMemcpyAsync((char*)dst + off, g_bounce[k & 1], len, hipMemcpyHostToDevice, s));
    PF_HIP(hipEventRecord(ev.e[k & 1], s));
  }
  // the bounce buffers are shared: they must be drained before the lock goes
  PF_HIP(hipStreamSynchronize(s));
  return 0;
}
}  // namespace

// The bounce buffers are released with the lock: on an error part-way through,
// the stream is drained first so that no copy into or out of them is still in
// flight when the next transfer takes them.
int to_host(void* dst, const void* src, size_t bytes, hipStream_t s) {
  std::lock_guard<std::mutex> lk(g_bounce_mu);
  const int rc = to_host_locked(dst, src, bytes, s);
  if (rc) (void)hipStreamSynchronize(s);
  return rc;
}

int to_device(void* dst, const void* src, size_t bytes, hipStream_t s) {
  std::lock_guard<std::mutex> lk(g_bounce_mu);
  const int rc = to_device_locked(dst, src, bytes, s);
  if (rc) (void)hipStreamSynchronize(s);
  return rc;
}

// ---------------------------------------------------------------------------
// Twiddle tables.
// ---------------------------------------------------------------------------

// Every length's table W_n^t = exp(-2 pi i t/n), t < n, back to back in the
// order of PF_GRID_SIZES, one array per precision in static device memory.
// Each device's copy is filled once (a host-to-device copy, no allocation), on
// the first use of any table on that device.
namespace {
#define PF_SUM(N) +N
constexpr int kTwTotal = 0 PF_GRID_SIZES(PF_SUM);
#undef PF_SUM
__device__ __align__(256) double2 g_tw64[kTwTotal];
__device__ __align__(256) float2 g_tw32[kTwTotal];

int tw_offset(int n) {
  int off = 0;
#define PF_OFF(N) \
  if (n == N) return off; \
  off += N;
  PF_GRID_SIZES(PF_OFF)
#undef PF_OFF
  return -1;
}

std::mutex g_tw_mu;
std::map<int, std::pair<double2*, float2*>> g_tw;  // device -> its copies of g_tw64, g_tw32

// Under g_tw_mu: the device's table addresses, filling them on first use.
bool tw_ready(int dev, std::pair<double2*, float2*>* out) {
  auto it = g_tw.find(dev);
  if (it != g_tw.end()) { *out = it->second; return true; }
  void *p64 = nullptr, *p32 = nullptr;
  if (hipGetSymbolAddress(&p64, HIP_SYMBOL(g_tw64)) != hipSuccess ||
      hipGetSymbolAddress(&p32, HIP_SYMBOL(g_tw32)) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  std::vector<double2> h64(kTwTotal);
  std::vector<float2> h32(kTwTotal);
  int off = 0;
  auto fill = [&](int n) {
    std::vector<double> re(n), im(n);
    host_twiddles(n, re.data(), im.data());
    for (int t = 0; t < n; ++t) {
      h64[off + t].x = re[t]; h64[off + t].y = im[t];
      h32[off + t].x = (float)re[t]; h32[off + t].y = (float)im[t];
    }
    off += n;
  };
#define PF_FILL(N) fill(N);
  PF_GRID_SIZES(PF_FILL)
#undef PF_FILL
  if (hipMemcpy(p64, h64.data(), sizeof(double2) * kTwTotal, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(p32, h32.data(), sizeof(float2) * kTwTotal, hipMemcpyHostToDevice) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  *out = g_tw[dev] = std::make_pair((double2*)p64, (float2*)p32);
  return true;
}
}  // namespace

template <typename R> const c2<R>* twiddle_table(int n) {
  int dev = 0;
  const int off = tw_offset(n);
  if (off < 0 || hipGetDevice(&dev) != hipSuccess) return nullptr;
  std::pair<double2*, float2*> t;
  {
    std::lock_guard<std::mutex> lk(g_tw_mu);
    if (!tw_ready(dev, &t)) return nullptr;
  }
  if constexpr (sizeof(R) == 8) return t.first + off;
  else return t.second + off;
}
template const c2<float>* twiddle_table<float>(int);
template const c2<double>* twiddle_table<double>(int);

// ---------------------------------------------------------------------------
// Pass launchers with compile-time sizes.
// ---------------------------------------------------------------------------
static inline unsigned ceil_div(long a, long b) { return (unsigned)((a + b - 1) / b); }

template <typename R>
int x_r2c(int nx, const c2<R>* src, c2<R>* dst, c2<R>* nyq, long nlines, R scale, hipStream_t s) {
  const c2<R>* tw = twiddle_table<R>(nx);
  if (!tw) return fail(PF_EHIP, "twiddle table set-up failed");
  switch (nx) {
#define PF_CASE(N)                                                                      \
  case N: {                                                                             \
    constexpr int LPB = x_lines<R>(N / 2);                                              \
    hipLaunchKernelGGL((k_x_r2c<R, N>), dim3(ceil_div(nlines, LPB)),                    \
                       dim3(LPB * plan_T(N / 2)), 0, s, src, dst, nyq, nlines, tw, scale); \
    break;                                                                              \
  }
    PF_GRID_SIZES(PF_CASE)
#undef PF_CASE
    default: return fail(PF_EINVAL, "unsupported nx " + std::to_string(nx));
  }
  return 0;
}

namespace {
// V: plan variant, for the lengths that have it.
template <typename R, int V>
int x_c2r_plan(int nx, const c2<R>* src, c2<R>* dst, const c2<R>* nyq, long nlines, hipStream_t s) {
  const c2<R>* tw = twiddle_table<R>(nx);
  if (!tw) return fail(PF_EHIP, "twiddle table set-up failed");
  switch (nx) {
#define PF_CASE(N)                                                                   \
  case N: {                                                                          \
    constexpr int W = plan_alt(N / 2, V, 0) ? V : 0, LPB = x_c2r_lines<R>(N / 2, W); \
    constexpr bool SHORT = x_c2r_short(N / 2, W);                                    \
    auto kernel = SHORT && nlines * N * sizeof(R) >= kStageBytes ? &k_x_c2r<R, N, W, SHORT> \
                                                                 : &k_x_c2r<R, N, W, false>; \
    hipLaunchKernelGGL(kernel, dim3(ceil_div(nlines, LPB)), dim3(LPB * plan_T(N / 2, W)), 0, s, src, dst, nyq, \
                       nlines, tw);                                                  \
    break;                                                                           \
  }
    PF_GRID_SIZES(PF_CASE)
#undef PF_CASE
    default: return fail(PF_EINVAL, "unsupported nx " + std::to_string(nx));
  }
  return 0;
}
}  // namespace

template <typename R>
int x_c2r(int nx, const c2<R>* src, c2<R>* dst, const c2<R>* nyq, long nlines, hipStream_t s) {
  return x_c2r_plan<R, 0>(nx, src, dst, nyq, nlines, s);
}
int x_c2r_as_xline(int nx, const double2* src, double2* dst, const double2* nyq, long nlines, hipStream_t s) {
  return x_c2r_plan<double, xline_plan(sizeof(double2))>(nx, src, dst, nyq, nlines, s);
}

template <typename R>
int y_pass(int ny, bool inv, c2<R>* main, c2<R>* nyq, long M, long nlines, hipStream_t s) {
  const c2<R>* tw = twiddle_table<R>(ny);
  if (!tw) return fail(PF_EHIP, "twiddle table set-up failed");
  switch (ny) {
#define PF_CASE(N)                                                                                     \
  case N: {                                                                                            \
    constexpr int TX = col_tile(N, sizeof(c2<R>));                                                     \
    dim3 grid(ypass_grid(ceil_div(M * nlines, TX), ceil_div(nlines, TX))), block(TX * plan_T(N));      \
    const bool keep = bank_stays(2ul * sizeof(R) * M * N * nlines);                                    \
    auto kernel = inv ? (keep ? &k_ypass<R, N, true, false, true> : &k_ypass<R, N, true>)              \
                      : (keep ? &k_ypass<R, N, false, false, true> : &k_ypass<R, N, false>);           \
    hipLaunchKernelGGL(kernel, grid, block, 0, s, main, nyq, M, nlines, nlines, tw,                    \
                       (const Member<R>*)nullptr, 0L);                                                 \
    break;                                                                                             \
  }
    PF_GRID_SIZES(PF_CASE)
#undef PF_CASE
    default: return fail(PF_EINVAL, "unsupported ny " + std::to_string(ny));
  }
  return 0;
}

template <typename R, bool INV, int FAR>
int z_pass(int nz, c2<R>* near, c2<R>* nearn, c2<R>* far, c2<R>* farn, int M, int ny, int nf, hipStream_t s) {
  const c2<R>* tw = twiddle_table<R>(nz);
  if (!tw) return fail(PF_EHIP, "twiddle table set-up failed");
  switch (nz) {
#define PF_CASE(N)                                                                                         \
  case N: {                                                                                                \
    constexpr int TX = col_tile(N, sizeof(c2<R>));                                                         \
    const unsigned tm = ceil_div((long)M * ny, TX), tn = ceil_div(ny, TX), run = ceil_div(M, TX);          \
    const unsigned tiles = (tm + tn) * (unsigned)nf;                                                       \
    hipLaunchKernelGGL((k_zpass<R, N, INV, FAR>), dim3(ceil_div(tiles, 8 * run) * 8 * run),                \
                       dim3(TX * plan_T(N)), 0, s, near, nearn, far, farn, (unsigned)M, (unsigned)ny,      \
                       (unsigned)nf, tm, tn, run, tw);                                                     \
    break;                                                                                                 \
  }
    PF_GRID_SIZES(PF_CASE)
#undef PF_CASE
    default: return fail(PF_EINVAL, "unsupported nz " + std::to_string(nz));
  }
  return 0;
}

#define PF_INST(R)                                                                \
  template int x_r2c<R>(int, const c2<R>*, c2<R>*, c2<R>*, long, R, hipStream_t); \
  template int x_c2r<R>(int, const c2<R>*, c2<R>*, const c2<R>*, long, hipStream_t); \
  template int y_pass<R>(int, bool, c2<R>*, c2<R>*, long, long, hipStream_t);
PF_INST(float)
PF_INST(double)
#undef PF_INST

// ---------------------------------------------------------------------------
// Whole 3-D transforms (P3DFFT order: forward x, y, z; inverse z, y, x), three
// launches each: the x pass takes the caller's real fields into the split
// layout, the z pass leaves it for the requested one (FAR_*), so neither end
// needs a copy.
// ---------------------------------------------------------------------------
template <typename R, int FAR>
int fwd3d(const c2<R>* src, c2<R>* main, c2<R>* nyq, c2<R>* far, c2<R>* farn, int nx, int ny, int nz, int batch,
          R scale, hipStream_t s) {
  const int M = nx / 2;
  int rc = x_r2c<R>(nx, src, main, nyq, (long)ny * nz * batch, scale, s);
  if (!rc) rc = y_pass<R>(ny, false, main, nyq, M, (long)nz * batch, s);
  if (!rc) rc = z_pass<R, false, FAR>(nz, main, nyq, far, farn, M, ny, batch, s);
  return rc;
}
template <typename R>
int fwd3d_split(const c2<R>* src, c2<R>* main, c2<R>* nyq, int nx, int ny, int nz, int batch, R scale, hipStream_t s) {
  return fwd3d<R, FAR_SPLIT>(src, main, nyq, main, nyq, nx, ny, nz, batch, scale, s);
}
template <typename R>
int fwd3d_tiled(const c2<R>* src, c2<R>* main, c2<R>* nyq, c2<R>* tiled, int nx, int ny, int nz, int batch, R scale,
                hipStream_t s) {
  return fwd3d<R, FAR_TILED>(src, main, nyq, tiled, nullptr, nx, ny, nz, batch, scale, s);
}
template int fwd3d_split<double>(const c2<double>*, c2<double>*, c2<double>*, int, int, int, int, double, hipStream_t);
template int fwd3d_tiled<float>(const c2<float>*, c2<float>*, c2<float>*, c2<float>*, int, int, int, int, float,
                                hipStream_t);
template int fwd3d_tiled<double>(const c2<double>*, c2<double>*, c2<double>*, c2<double>*, int, int, int, int, double,
                                 hipStream_t);

}  // namespace pf

// ===========================================================================
// C-ABI transform entry points.
// ===========================================================================
namespace {
using namespace pf;

int check_dims(int nx, int ny, int nz, int batch) {
  if (!grid_size_supported(nx) || !grid_size_supported(ny) || !grid_size_supported(nz))
    return fail(PF_EINVAL, std::string("grid ") + std::to_string(nx) + "x" + std::to_string(ny) +
                               "x" + std::to_string(nz) + " not supported; each axis must be one of " +
                               supported_sizes_text());
  if (batch < 1) return fail(PF_EINVAL, "batch must be >= 1");
  return 0;
}

// Scratch of pf_fft_r2c / pf_fft_c2r: one buffer per device, shared by every
// caller and stream.  A call holds the device's lock from taking the buffer
// until its work is enqueued; that work first waits (on the caller's stream)
// for the event the previous user recorded after its last use, and records the
// event again afterwards, so uses on different streams or threads run one after
// another on the GPU.  A buffer that must grow is freed only after that event
// has completed.
struct Workspace {
  std::mutex mu;
  void* p = nullptr;
  size_t bytes = 0;
  hipEvent_t done = nullptr;
};
std::mutex g_ws_mu;
std::map<int, std::unique_ptr<Workspace>> g_ws;

Workspace* device_workspace() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return nullptr;
  std::lock_guard<std::mutex> lk(g_ws_mu);
  auto& w = g_ws[dev];
  if (!w) w.reset(new Workspace);
  return w.get();
}

// Holds the device workspace (locked) for one call on stream s.
struct WorkspaceLease {
  Workspace* w = nullptr;
  std::unique_lock<std::mutex> lk;
  hipStream_t s;
  void* p = nullptr;
  std::string err;
  WorkspaceLease(size_t bytes, hipStream_t s_) : s(s_) {
    w = device_workspace();
    if (!w) { err = "no current device"; return; }
    lk = std::unique_lock<std::mutex>(w->mu);
    if (!w->done && hipEventCreateWithFlags(&w->done, hipEventDisableTiming) != hipSuccess) {
      w->done = nullptr;
      err = "event creation failed";
      return;
    }
    if (w->bytes < bytes) {
      if (w->p) {
        if (hipEventSynchronize(w->done) != hipSuccess) { err = "waiting for the previous use failed"; return; }
        (void)hipFree(w->p);
      }
      w->p = nullptr;
      w->bytes = 0;
      if (hipMalloc(&w->p, bytes) != hipSuccess) {
        w->p = nullptr;
        (void)hipGetLastError();
        err = "workspace allocation of " + std::to_string(bytes) + " bytes failed";
        return;
      }
      w->bytes = bytes;
    } else if (hipStreamWaitEvent(s, w->done, 0) != hipSuccess) {
      err = "hipStreamWaitEvent failed";
      return;
    }
    p = w->p;
  }
  // Marks the end of this call's use (after its last enqueued access).
  ~WorkspaceLease() {
    if (p) (void)hipEventRecord(w->done, s);
  }
};

// Bytes of scratch a batch of transforms needs: the split-layout copy (main
// block + Nyquist planes).
template <typename R> size_t r2c_scratch_bytes(int nx, int ny, int nz, int batch) {
  return sizeof(R) * (size_t)nx * ny * nz * batch + sizeof(c2<R>) * (size_t)ny * nz * batch;
}

// Whether complex accesses at p are aligned (a caller's real array need only be
// aligned for its reals).
template <typename R> bool complex_aligned(const void* p) { return reinterpret_cast<uintptr_t>(p) % sizeof(c2<R>) == 0; }

// The forward transform with its scratch at ws.  A real array that is not aligned
// for complex accesses is copied into the scratch first.
template <typename R>
int r2c_core(int nx, int ny, int nz, int batch, const void* in, void* out, int layout, double scale,
             void* wsp, hipStream_t s) {
  const size_t P = (size_t)nx * ny * nz;
  char* ws = (char*)wsp;
  c2<R>* main = (c2<R>*)ws;
  c2<R>* nyq = (c2<R>*)(ws + sizeof(R) * P * batch);
  const c2<R>* src = (const c2<R>*)in;
  if (!complex_aligned<R>(in)) {
    PF_HIP(hipMemcpyAsync(main, in, sizeof(R) * P * batch, hipMemcpyDeviceToDevice, s));
    src = main;
  }
  const int rc = layout == PF_LAYOUT_XFAST
                     ? fwd3d<R, FAR_XFAST>(src, main, nyq, (c2<R>*)out, nullptr, nx, ny, nz, batch, (R)scale, s)
                     : fwd3d<R, FAR_ZFAST>(src, main, nyq, (c2<R>*)out, nullptr, nx, ny, nz, batch, (R)scale, s);
  if (rc) return rc;
  PF_HIP(hipGetLastError());
  return 0;
}

template <typename R>
int r2c_dev(int nx, int ny, int nz, int batch, const void* in, void* out, int layout, double scale,
            hipStream_t s) {
  WorkspaceLease lease(r2c_scratch_bytes<R>(nx, ny, nz, batch), s);
  if (!lease.p) return fail(PF_ENOMEM, lease.err);
  return r2c_core<R>(nx, ny, nz, batch, in, out, layout, scale, lease.p, s);
}

template <typename R>
int c2r_dev(int nx, int ny, int nz, int batch, const void* in, void* out, int layout, hipStream_t s) {
  const size_t P = (size_t)nx * ny * nz, plane = (size_t)ny * nz;
  WorkspaceLease lease(sizeof(R) * P * batch + sizeof(c2<R>) * plane * batch, s);
  if (!lease.p) return fail(PF_ENOMEM, lease.err);
  char* ws = (char*)lease.p;
  c2<R>* main = (c2<R>*)ws;
  c2<R>* nyq = (c2<R>*)(ws + sizeof(R) * P * batch);
  c2<R>* spec = (c2<R>*)const_cast<void*>(in);  // read only
  int rc = layout == PF_LAYOUT_XFAST ? z_pass<R, true, FAR_XFAST>(nz, main, nyq, spec, nullptr, nx / 2, ny, batch, s)
                                     : z_pass<R, true, FAR_ZFAST>(nz, main, nyq, spec, nullptr, nx / 2, ny, batch, s);
  if (!rc) rc = y_pass<R>(ny, true, main, nyq, nx / 2, (long)nz * batch, s);
  // a real array not aligned for complex stores is filled by a copy
  const bool direct = complex_aligned<R>(out);
  if (!rc) rc = x_c2r<R>(nx, main, direct ? (c2<R>*)out : main, nyq, (long)ny * nz * batch, s);
  if (rc) return rc;
  if (!direct) PF_HIP(hipMemcpyAsync(out, main, sizeof(R) * P * batch, hipMemcpyDeviceToDevice, s));
  PF_HIP(hipGetLastError());
  return 0;
}
}  // namespace

extern "C" int pf_fft_r2c(int nx, int ny, int nz, int batch, int prec, const void* d_in, void* d_out,
                          int layout, double scale, void* stream) {
  int rc = check_dims(nx, ny, nz, batch);
  if (rc) return rc;
  if (!d_in || !d_out) return fail(PF_EINVAL, "null buffer");
  if (layout != PF_LAYOUT_XFAST && layout != PF_LAYOUT_ZFAST) return fail(PF_EINVAL, "bad layout");
  hipStream_t s = (hipStream_t)stream;
  if (prec == PF_PREC_FP64) return r2c_dev<double>(nx, ny, nz, batch, d_in, d_out, layout, scale, s);
  if (prec == PF_PREC_FP32) return r2c_dev<float>(nx, ny, nz, batch, d_in, d_out, layout, scale, s);
  return fail(PF_EINVAL, "bad precision");
}

extern "C" int pf_fft_c2r(int nx, int ny, int nz, int batch, int prec, const void* d_in, void* d_out,
                          int layout, void* stream) {
  int rc = check_dims(nx, ny, nz, batch);
  if (rc) return rc;
  if (!d_in || !d_out) return fail(PF_EINVAL, "null buffer");
  if (layout != PF_LAYOUT_XFAST && layout != PF_LAYOUT_ZFAST) return fail(PF_EINVAL, "bad layout");
  hipStream_t s = (hipStream_t)stream;
  if (prec == PF_PREC_FP64) return c2r_dev<double>(nx, ny, nz, batch, d_in, d_out, layout, s);
  if (prec == PF_PREC_FP32) return c2r_dev<float>(nx, ny, nz, batch, d_in, d_out, layout, s);
  return fail(PF_EINVAL, "bad precision");
}

// ---------------------------------------------------------------------------
// pf_fft_r2c_noalloc: pf_fft_r2c with its scratch in static device memory.
// scratch is this file's array; in host code its name only stands for the
// symbol, so every use goes through the address hipGetSymbolAddress returns for
// the current device (each device holds its own copy).
// ---------------------------------------------------------------------------
namespace {
constexpr size_t kNoAllocScratchBytes = size_t(64) << 20;
__device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];
std::mutex g_scratch_mu;
std::map<int, void*> g_scratch;  // device -> the address of its copy of scratch

// Set-up, once per device with that device current: the device address of
// scratch (and, through twiddle_table, the static twiddle tables).
void* scratch_ptr() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return nullptr;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  auto it = g_scratch.find(dev);
  if (it != g_scratch.end()) return it->second;
  void* ptr = nullptr;
  const hipError_t e = hipGetSymbolAddress((void**)&ptr, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !ptr) {
    (void)hipGetLastError();
    return nullptr;
  }
  g_scratch[dev] = ptr;
  return ptr;
}
}  // namespace

extern "C" int pf_fft_r2c_noalloc(int nx, int ny, int nz, int batch, int prec, const void* d_in, void* d_out,
                                  int layout, double scale, void* stream) {
  int rc = check_dims(nx, ny, nz, batch);
  if (rc) return rc;
  if (!d_in || !d_out) return fail(PF_EINVAL, "null buffer");
  if (layout != PF_LAYOUT_XFAST && layout != PF_LAYOUT_ZFAST) return fail(PF_EINVAL, "bad layout");
  if (prec != PF_PREC_FP64 && prec != PF_PREC_FP32) return fail(PF_EINVAL, "bad precision");
  const size_t need = prec == PF_PREC_FP64 ? r2c_scratch_bytes<double>(nx, ny, nz, batch)
                                           : r2c_scratch_bytes<float>(nx, ny, nz, batch);
  if (need > kNoAllocScratchBytes)
    return fail(PF_EINVAL, "pf_fft_r2c_noalloc: " + std::to_string(batch) + " field(s) of " + std::to_string(nx) +
                               "x" + std::to_string(ny) + "x" + std::to_string(nz) + " need " +
                               std::to_string(need) + " bytes of scratch; the limit is " +
                               std::to_string(kNoAllocScratchBytes));
  void* ws = scratch_ptr();
  if (!ws) return fail(PF_EHIP, "pf_fft_r2c_noalloc: no device address for the static scratch");
  hipStream_t s = (hipStream_t)stream;
  if (prec == PF_PREC_FP64) return r2c_core<double>(nx, ny, nz, batch, d_in, d_out, layout, scale, ws, s);
  return r2c_core<float>(nx, ny, nz, batch, d_in, d_out, layout, scale, ws, s);
}

// Device buffers of pf_f_trans / pf_inv_trans, per device, grown as needed and
// kept until the process ends.  These calls are synchronous: the lock is held
// for the whole call, so calls from several threads take turns.
namespace {
struct HostCallBuffers {
  std::mutex mu;
  void* in = nullptr;
  void* out = nullptr;
  size_t in_bytes = 0, out_bytes = 0;
};
std::mutex g_hcb_mu;
std::map<int, std::unique_ptr<HostCallBuffers>> g_hcb;

HostCallBuffers* host_call_buffers() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return nullptr;
  std::lock_guard<std::mutex> lk(g_hcb_mu);
  auto& b = g_hcb[dev];
  if (!b) b.reset(new HostCallBuffers);
  return b.get();
}

int grow(void** p, size_t* have, size_t want) {
  if (*have >= want) return 0;
  if (*p) (void)hipFree(*p);
  *p = nullptr;
  *have = 0;
  if (hipMalloc(p, want) != hipSuccess) {
    *p = nullptr;
    (void)hipGetLastError();
    return fail(PF_ENOMEM, "device allocation of " + std::to_string(want) + " bytes failed");
  }
  *have = want;
  return 0;
}
}  // namespace

// Host-buffer drop-ins for f_trans (src/f_trans.f90:1-15) and inv_trans
// (src/inv_trans.f90:1-13): FP64, the spectrum in the reference's Z-pencil order.
extern "C" int pf_f_trans(const double* in, double* out, int nx, int ny, int nz) {
  int rc = check_dims(nx, ny, nz, 1);
  if (rc) return rc;
  if (!in || !out) return fail(PF_EINVAL, "null buffer");
  const size_t P = (size_t)nx * ny * nz, H = (size_t)(nx / 2 + 1) * ny * nz;
  HostCallBuffers* b = host_call_buffers();
  if (!b) return fail(PF_EHIP, "no current device");
  std::lock_guard<std::mutex> lk(b->mu);
  if ((rc = grow(&b->in, &b->in_bytes, sizeof(double) * P))) return rc;
  if ((rc = grow(&b->out, &b->out_bytes, sizeof(double) * 2 * H))) return rc;
  rc = to_device(b->in, in, sizeof(double) * P, nullptr);
  const double scale = 1.0 / (double)(float)((long)nx * ny * nz);
  if (!rc) rc = pf_fft_r2c(nx, ny, nz, 1, PF_PREC_FP64, b->in, b->out, PF_LAYOUT_ZFAST, scale, nullptr);
  if (!rc) rc = to_host(out, b->out, sizeof(double) * 2 * H, nullptr);
  return rc;
}

extern "C" int pf_inv_trans(const double* in, double* out, int nx, int ny, int nz) {
  int rc = check_dims(nx, ny, nz, 1);
  if (rc) return rc;
  if (!in || !out) return fail(PF_EINVAL, "null buffer");
  const size_t P = (size_t)nx * ny * nz, H = (size_t)(nx / 2 + 1) * ny * nz;
  HostCallBuffers* b = host_call_buffers();
  if (!b) return fail(PF_EHIP, "no current device");
  std::lock_guard<std::mutex> lk(b->mu);
  if ((rc = grow(&b->in, &b->in_bytes, sizeof(double) * 2 * H))) return rc;
  if ((rc = grow(&b->out, &b->out_bytes, sizeof(double) * P))) return rc;
  rc = to_device(b->in, in, sizeof(double) * 2 * H, nullptr);
  if (!rc) rc = pf_fft_c2r(nx, ny, nz, 1, PF_PREC_FP64, b->in, b->out, PF_LAYOUT_ZFAST, nullptr);
  if (!rc) rc = to_host(out, b->out, sizeof(double) * P, nullptr);
  return rc;
}
