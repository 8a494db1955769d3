// Transfer-matrix generation and the lambda-independent / elementwise passes
// of the hot path (gfx950): pupil-field synthesis, basis evaluation, power and
// intensity reductions.  All are HBM-bound; they are written for coalesced
// 8/16-byte accesses with one pixel (or four) per lane.
#include <type_traits>

#include "dlx_internal.h"
#include "dlx_phasor.h"

namespace dlx {

// ---------------------------------------------------------------------------
// Transfer matrix  W[b][l][k] = exp(sign * 2 pi i * a_k * b_l)
// (utils/propagation.py:109-127, stored transposed: N_out x N_in).
// The product a_k*b_l is formed in FP64 and reduced to [-1/2, 1/2] turns, so
// the FP32 sincospi sees an argument with an absolute error of ~1e-17 turns.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256)
dft_matrix_kernel(DftChunk c, int n_in, int n_out, int inverse, float2* __restrict__ out,
                  long bstride) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  const int l = blockIdx.y;
  const int b = blockIdx.z;
  if (k >= n_in) return;
  const double a = (double)k * c.a_scale[b] + c.a_off[b];
  const double bb = (double)l * c.b_scale[b] + c.b_off[b];
  double t = a * bb;
  t -= rint(t);
  float s, co;
  sincospif(2.0f * (float)t, &s, &co);
  out[(long)b * bstride + (long)l * n_in + k] = make_float2(co, inverse ? s : -s);
}

hipError_t launch_dft_chunk(const DftChunk& c, int nb, int n_in, int n_out, int inverse,
                            float2* out, long bstride, hipStream_t s) {
  dim3 grid((n_in + 255) / 256, n_out, nb);
  hipLaunchKernelGGL(dft_matrix_kernel, grid, dim3(256), 0, s, c, n_in, n_out, inverse, out,
                     bstride);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Pupil field for a chunk of wavelengths:
//   out[b](y,x) = s * amp * exp(2 pi i * ((opd + tx X + ty Y)/lambda_b + phase/(2 pi)))
//                 [* in[b](y,x)]
// The argument is accumulated in FP64 turns and reduced to [-1/2, 1/2] before
// the hardware sine / cosine (which take turns).
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256)
pupil_field_kernel(PupilChunk c, int n, double dx, double x0, double tx, double ty,
                   const float* __restrict__ amp, const float* __restrict__ opd,
                   const float* __restrict__ phase, float scale,
                   const float2* __restrict__ in, float2* __restrict__ out, long npix) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int b = blockIdx.y;
  if (p >= npix) return;
  const int y = (int)(p / n), x = (int)(p - (long)y * n);
  const double path = pupil_path(tx, pupil_coord(x, dx, x0), ty * pupil_coord(y, dx, x0),
                                 opd ? (double)opd[p] : 0.0);
  const double turns0 = phase ? (double)phase[p] * 0.15915494309189535 : 0.0;  // 1 / (2 pi)
  float2 v = pupil_phasor(path, c.inv_wl[b], turns0, scale * (amp ? amp[p] : 1.0f));
  if (in) {
    const float2 e = in[(long)b * npix + p];
    v = make_float2(e.x * v.x - e.y * v.y, e.x * v.y + e.y * v.x);
  }
  out[(long)b * npix + p] = v;
}

hipError_t launch_pupil_chunk(const PupilChunk& c, int nb, int n, double dx, double x0,
                              double tx, double ty, const float* amp, const float* opd,
                              const float* phase, float scale, const float2* in,
                              float2* out, hipStream_t s) {
  const long npix = (long)n * n;
  dim3 grid((unsigned)((npix + 255) / 256), nb);
  hipLaunchKernelGGL(pupil_field_kernel, grid, dim3(256), 0, s, c, n, dx, x0, tx, ty, amp,
                     opd, phase, scale, in, out, npix);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Basis evaluation: out[s][p] = sum_j coeffs[s][j] * basis[j][p] (+ base[p]).
// V pixels a lane: four (16-byte accesses) where the planes are aligned, one
// elsewhere.  The basis is streamed once for up to kSets coefficient sets
// (utils/math.py:177-196 tensordot), kDepth planes of it in flight per lane, and
// kRest of the last ones, missing planes loading the last again: a plane loaded
// by itself costs a full latency.  21 planes of 401^2 (one-pixel lanes, which
// coalesce) 8.8 -> 5.6 us; 36 of 512^2 7.6 -> 7.0 us, 5.4 TB/s.
// ---------------------------------------------------------------------------
constexpr int kSets = 8;

template <int NS, int V>
__global__ void __launch_bounds__(256)
eval_basis_kernel(int nbasis, long npix, int nsets, const float* __restrict__ basis,
                  const float* __restrict__ coeffs, const float* __restrict__ base,
                  float* __restrict__ out) {
  constexpr int kDepth = NS == 1 ? 12 : 6, kRest = NS == 1 ? 6 : 3;
  const long p = ((long)blockIdx.x * blockDim.x + threadIdx.x) * V;
  if (p >= npix) return;
  float acc[NS][V];
#pragma unroll
  for (int s = 0; s < NS; ++s)
#pragma unroll
    for (int q = 0; q < V; ++q) acc[s][q] = 0.f;
  auto group = [&](auto FULL, int j0) __attribute__((always_inline)) {
    constexpr int D = decltype(FULL)::value ? kDepth : kRest;
    PixelRun<V> v[D];
#pragma unroll
    for (int e = 0; e < D; ++e)
      v[e].load(basis + (long)(decltype(FULL)::value || j0 + e < nbasis ? j0 + e : nbasis - 1) * npix + p);
#pragma unroll
    for (int e = 0; e < D; ++e) {
      if (decltype(FULL)::value || j0 + e < nbasis) {
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          if (NS == 1 || s < nsets) {
            const float cj = coeffs[(long)s * nbasis + j0 + e];
#pragma unroll
            for (int q = 0; q < V; ++q) acc[s][q] = fmaf(cj, v[e].v[q], acc[s][q]);
          }
        }
      }
    }
  };
  int j0 = 0;
  for (; j0 + kDepth <= nbasis; j0 += kDepth) group(std::true_type{}, j0);
  for (; j0 < nbasis; j0 += kRest) group(std::false_type{}, j0);
  PixelRun<V> bb{};
  if (base) bb.load(base + p);
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    if (NS > 1 && s >= nsets) break;
    PixelRun<V> r;
#pragma unroll
    for (int q = 0; q < V; ++q) r.v[q] = base ? acc[s][q] + bb.v[q] : acc[s][q];
    r.store(out + (long)s * npix + p);
  }
}

template <int V>
hipError_t eval_basis_go(int nbasis, long npix, int nsets, const float* basis, const float* coeffs,
                         const float* base, float* out, hipStream_t s) {
  const dim3 grid((unsigned)((npix / V + 255) / 256));
  if (nsets == 1) {
    hipLaunchKernelGGL((eval_basis_kernel<1, V>), grid, dim3(256), 0, s, nbasis, npix, 1, basis,
                       coeffs, base, out);
    return hipGetLastError();
  }
  for (int s0 = 0; s0 < nsets; s0 += kSets) {
    const int ns = nsets - s0 < kSets ? nsets - s0 : kSets;
    hipLaunchKernelGGL((eval_basis_kernel<kSets, V>), grid, dim3(256), 0, s, nbasis, npix, ns, basis,
                       coeffs + (long)s0 * nbasis, base, out + (long)s0 * npix);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_eval_basis(int nbasis, long npix, int nsets, const float* basis,
                             const float* coeffs, const float* base, float* out,
                             hipStream_t s) {
  // 16-byte loads and stores need 16-byte aligned rows
  const bool vec = ((npix & 3) == 0) && ((reinterpret_cast<uintptr_t>(basis) & 15) == 0) &&
                   ((reinterpret_cast<uintptr_t>(out) & 15) == 0) &&
                   (!base || (reinterpret_cast<uintptr_t>(base) & 15) == 0);
  return vec ? eval_basis_go<4>(nbasis, npix, nsets, basis, coeffs, base, out, s)
             : eval_basis_go<1>(nbasis, npix, nsets, basis, coeffs, base, out, s);
}

// ---------------------------------------------------------------------------
// Reductions.  One workgroup per instance sums in a fixed order, so results
// are bit-reproducible (no float atomics).
// ---------------------------------------------------------------------------
constexpr int kRedThreads = 1024;

__global__ void __launch_bounds__(kRedThreads)
power_kernel(long npix, const float2* __restrict__ f, float* __restrict__ out) {
  __shared__ float red[kRedThreads / 64];
  const int b = blockIdx.x;
  const float2* fb = f + (long)b * npix;
  float acc = 0.f;
  for (long p = threadIdx.x; p < npix; p += kRedThreads) {
    const float2 e = fb[p];
    acc = fmaf(e.x, e.x, fmaf(e.y, e.y, acc));
  }
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    float s = 0.f;
    for (int i = 0; i < kRedThreads / 64; ++i) s += red[i];
    out[b] = s;
  }
}

hipError_t launch_power(long npix, int batch, const float2* f, float* out, hipStream_t s) {
  hipLaunchKernelGGL(power_kernel, dim3(batch), dim3(kRedThreads), 0, s, npix, f, out);
  return hipGetLastError();
}

// |E|^2 per pixel, or summed over the batch in index order (deterministic).
__global__ void __launch_bounds__(256)
intensity_kernel(long npix, int batch, const float2* __restrict__ f, int sum_batch,
                 float* __restrict__ out) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= npix) return;
  if (sum_batch) {
    float acc = 0.f;
    for (int b = 0; b < batch; ++b) {
      const float2 e = f[(long)b * npix + p];
      acc += e.x * e.x + e.y * e.y;
    }
    out[p] = acc;
  } else {
    for (int b = 0; b < batch; ++b) {
      const float2 e = f[(long)b * npix + p];
      out[(long)b * npix + p] = e.x * e.x + e.y * e.y;
    }
  }
}

hipError_t launch_intensity(long npix, int batch, const float2* f, int sum_batch, float* out,
                            hipStream_t s) {
  hipLaunchKernelGGL(intensity_kernel, dim3((unsigned)((npix + 255) / 256)), dim3(256), 0, s,
                     npix, batch, f, sum_batch, out);
  return hipGetLastError();
}

// psf[p] (=|+=) sum_b planes[b][p] in index order (deterministic): V pixels and
// 16 planes in flight per lane, then kRest of the rest (one after another they
// cost a full latency each): 7.9 -> 3.1 us at 11 planes of 173^2; 64 planes of
// 256^2 take 4.7 us, 3.6 TB/s (a 256^2 image has only 256 waves of 4 pixels; one
// pixel a lane took 5.2).
template <int V>
__global__ void __launch_bounds__(256)
sum_planes_kernel(long npix, int nplanes, const float* __restrict__ planes, int accumulate,
                  float* __restrict__ psf) {
  constexpr int kRest = 8;
  const long p = ((long)blockIdx.x * blockDim.x + threadIdx.x) * V;
  if (p >= npix) return;
  PixelRun<V> acc{};
  if (accumulate) acc.load(psf + p);
  int b0 = 0;
#pragma unroll 16
  for (; b0 < (nplanes & ~15); ++b0) {
    PixelRun<V> v;
    v.load(planes + (long)b0 * npix + p);
#pragma unroll
    for (int q = 0; q < V; ++q) acc.v[q] += v.v[q];
  }
  for (; b0 < nplanes; b0 += kRest) {
    PixelRun<V> v[kRest];
#pragma unroll
    for (int e = 0; e < kRest; ++e)
      v[e].load(planes + (long)(b0 + e < nplanes ? b0 + e : nplanes - 1) * npix + p);
#pragma unroll
    for (int e = 0; e < kRest; ++e) {
      if (b0 + e < nplanes) {
#pragma unroll
        for (int q = 0; q < V; ++q) acc.v[q] += v[e].v[q];
      }
    }
  }
  acc.store(psf + p);
}

hipError_t launch_sum_planes(long npix, int nplanes, const float* planes, int accumulate,
                             float* psf, hipStream_t s) {
  const bool vec = ((npix & 3) == 0) && ((reinterpret_cast<uintptr_t>(planes) & 15) == 0) &&
                   ((reinterpret_cast<uintptr_t>(psf) & 15) == 0);
  if (vec)
    hipLaunchKernelGGL(sum_planes_kernel<4>, dim3((unsigned)((npix / 4 + 255) / 256)), dim3(256), 0,
                       s, npix, nplanes, planes, accumulate, psf);
  else
    hipLaunchKernelGGL(sum_planes_kernel<1>, dim3((unsigned)((npix + 255) / 256)), dim3(256), 0, s,
                       npix, nplanes, planes, accumulate, psf);
  return hipGetLastError();
}

}  // namespace dlx
