// Internal helpers shared by the dlux_amd HIP translation units (gfx950 only).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stddef.h>
#include <cstdio>
#include <string>
#include <vector>
#include <algorithm>

#include "../../include/dlux_amd.h"

namespace dlx {

// Per-thread error message returned by dlx_last_error().
void set_error(const char* fmt, ...);
void clear_error();

#define DLX_CHECK_ARG(cond, ...)          \
  do {                                    \
    if (!(cond)) {                        \
      ::dlx::set_error(__VA_ARGS__);      \
      return DLX_ERR_INVALID;             \
    }                                     \
  } while (0)

#define DLX_HIP(call)                                                        \
  do {                                                                       \
    hipError_t _e = (call);                                                  \
    if (_e != hipSuccess) {                                                  \
      ::dlx::set_error("%s failed: %s", #call, hipGetErrorString(_e));       \
      return DLX_ERR_HIP;                                                    \
    }                                                                        \
  } while (0)

// Status of the last kernel launch on this thread.
inline int launch_status(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error("launch of %s failed: %s", what, hipGetErrorString(e));
    return DLX_ERR_HIP;
  }
  return DLX_OK;
}

// V consecutive floats of a plane, one access (V = 4: 16-byte aligned).
template <int V>
struct PixelRun {
  float v[V];
  __device__ __forceinline__ void load(const float* p) {
    if constexpr (V == 4) {
      const float4 t = *(const float4*)p;
      v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
    } else {
      v[0] = *p;
    }
  }
  __device__ __forceinline__ void store(float* p) const {
    if constexpr (V == 4) *(float4*)p = make_float4(v[0], v[1], v[2], v[3]);
    else *p = v[0];
  }
};

inline size_t align_up(size_t x, size_t a = 256) { return (x + a - 1) / a * a; }

// Device-side per-instance MFT parameters (one per wavelength / source).
struct MftInst {
  double a_scale;   // 1 / N_in
  double a_off;     // -(N_in-1)/2 / N_in - shift_a / N_in    (a_k = k*a_scale + a_off)
  double b_scale;   // p_out / fringe [/(f+df)]
  double b_off;     // (-(N_out-1)/2 - shift_b) * b_scale      (b_l = l*b_scale + b_off)
};

// Host-side builder: the per-axis coordinate vectors of transfer_matrix
// (utils/propagation.py:109-121), in FP64.
inline MftInst make_inst(const dlx_mft_geom& g, double wavelength, double dx_in,
                         double p_out, double shift) {
  MftInst p;
  const double n_in = g.n_in, n_out = g.n_out;
  const double fringe = wavelength / (dx_in * n_in);
  double so = p_out / fringe;
  if (g.has_focal) so /= (g.focal_length + g.focal_shift);
  p.a_scale = 1.0 / n_in;
  p.a_off = -(n_in - 1.0) / 2.0 / n_in - shift / n_in;
  p.b_scale = so;
  p.b_off = (-(n_out - 1.0) / 2.0 - shift) * so;
  return p;
}

// nfringes / (N_in N_out)  (utils/propagation.py:130-175, :246-254).
inline double mft_norm(const dlx_mft_geom& g, double wavelength, double dx_in,
                       double p_out) {
  const double diameter = g.n_in * dx_in;
  const double fringe = wavelength / diameter;
  double out_size = g.n_out * p_out;
  if (g.has_focal) out_size /= (g.focal_length + g.focal_shift);
  const double nfr = out_size / fringe;
  return nfr / ((double)g.n_in * (double)g.n_out);
}

// ---------------------------------------------------------------------------
// kernels implemented in the .hip files, launched from the host orchestration
// ---------------------------------------------------------------------------

// Per-launch instance parameters passed by value (kernel arguments), so no
// device-side parameter buffer is needed.
struct DftChunk {
  static constexpr int kMax = 48;
  double a_scale[kMax], a_off[kMax], b_scale[kMax], b_off[kMax];
};
struct PupilChunk {
  static constexpr int kMax = 128;
  double inv_wl[kMax];
};

struct GradChunk {
  static constexpr int kMax = 64;
  float kw[kMax];   // 2 pi / lambda per plane
};

hipError_t launch_dft_chunk(const DftChunk& c, int nb, int n_in, int n_out, int inverse,
                            float2* out, long bstride, hipStream_t s);

// Linear canonical transforms (dlx_lct.hip): per-instance phase polynomials in turns.
struct LctChirpChunk {
  static constexpr int kMax = 48;
  double q2[kMax], q1[kMax], q0[kMax], x0[kMax], dx[kMax];   // grid x_k = x0 + k dx
};
hipError_t launch_lct_chirp(const LctChirpChunk& c, int nb, int n, const float2* in,
                            float2* out, hipStream_t s);
hipError_t launch_pupil_chunk(const PupilChunk& c, int nb, int n, double dx, double x0,
                              double tx, double ty, const float* amp, const float* opd,
                              const float* phase, float scale, const float2* in,
                              float2* out, hipStream_t s);
hipError_t launch_eval_basis(int nbasis, long npix, int nsets, const float* basis,
                             const float* coeffs, const float* base, float* out,
                             hipStream_t s);
hipError_t launch_power(long npix, int batch, const float2* f, float* out, hipStream_t s);
hipError_t launch_intensity(long npix, int batch, const float2* f, int sum_batch, float* out,
                            hipStream_t s);
hipError_t launch_sum_planes(long npix, int nplanes, const float* planes, int accumulate,
                             float* psf, hipStream_t s);

// Backward reductions (dlx_grad.hip).  partial holds nbasis * nsets * project_parts(npix)
// floats.
hipError_t launch_grad_reduce(const GradChunk& c, int nb, long npix, const float* h,
                              int accumulate, float* g_opd, float* g_phase, hipStream_t s);
int project_parts(long npix);
hipError_t launch_project_basis(int nbasis, long npix, int nsets, const float* basis,
                                const float* g, float* partial, float* out, hipStream_t s);

// Bytes of an R x K complex array in the plain layouts that the workspace sizes
// are stated in: complex64, or (split) four bf16 planes of k in chunks of 8.
size_t mat_bytes(long rows, long k, bool split);

// Device-resident cache of tables (dlx_cache.hip), keyed by the caller: on a
// hit (*fresh false) the block is ready for work on s; on a miss (*fresh true)
// the caller fills it on s and then calls cache_ready.  *ptr == NULL (and
// *fresh true) when bypassed (capture, budget, memory): the caller generates
// into its own buffer.  The block is allocated on a key's second sighting, or
// on the first with `eager`.  cache_release records the entry's last use on s.
int cache_release(void* handle, hipStream_t s);
int cache_acquire_raw(const std::vector<double>& key, size_t bytes, hipStream_t s,
                      void** ptr, void** handle, bool* fresh, bool eager = false);
int cache_ready(void* handle, hipStream_t s);

// The detector chain (dlx_detector.hip) on one image that is the in-order sum
// of nsum planes sum_stride floats apart (nsum = 1: `batch` images), and its
// workspace size for nsum planes n^2 floats apart.
size_t detector_ws_bytes(int n, int batch, const dlx_detector_op* ops, int nops, int nsum = 1);
int detector_apply_sum(int n, int batch, int nsum, long sum_stride, const float* in,
                       const dlx_detector_op* ops, int nops, float* out, void* workspace,
                       size_t workspace_bytes, hipStream_t s);

// Holds a cache entry from its acquire (pass &lease.h) to its release, and
// releases it on scope exit too, so an error return never leaves an entry
// pinned.  release() records the last use on the stream after the work that
// reads the entry has been enqueued.
struct CacheLease {
  void* h = nullptr;
  hipStream_t s = nullptr;
  explicit CacheLease(hipStream_t st) : s(st) {}
  CacheLease(const CacheLease&) = delete;
  CacheLease& operator=(const CacheLease&) = delete;
  int release() {
    void* x = h;
    h = nullptr;
    return cache_release(x, s);
  }
  ~CacheLease() {
    if (h) (void)cache_release(h, s);
  }
};

}  // namespace dlx
