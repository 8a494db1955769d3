// Centred 2-D FFT (dLux's FFT propagator) and the angular-spectrum propagator
// on gfx950.
//
// dLux: out = fftshift(fft2(ifftshift(pad(x)))) / M      (utils/propagation.py:52-64)
//       inverse: fftshift(ifft2(ifftshift(pad(x)))) * M  (= conj-sign DFT / M)
//
// A 2-D transform is two launches of one kernel, templated on log2 M, the rows
// per workgroup and the pass, so the index arithmetic folds.  A workgroup runs
// a Stockham auto-sort FFT (stages of radix 16 and 8) on R rows of length M:
// the first stage reads its butterflies straight from memory -- the zero pad
// and ifftshift as an index map -- the stages between go through LDS, and the
// last one writes straight to memory, or through LDS where the rows are stored
// TRANSPOSED.  The second launch of a transform therefore reads the first's
// columns as rows and its transposed write restores the orientation; that
// write also applies fftshift and the 1/M scale.  HBM traffic is one read and
// one write of the M x M complex64 array per launch.  The angular-spectrum
// method takes three launches instead of four (launch_asm): the y transforms
// of its forward and inverse 2-D transforms, with the transfer function
// between them in the registers of the forward's last stage, run back to back.
#include <cmath>

#include "dlx_internal.h"

namespace dlx {
namespace {

// One 8-byte store of a complex64 (the compiler may otherwise split a float2
// store into two 4-byte stores, doubling the write requests of the transposed
// store's short runs).
typedef float cplx_v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void store_c64(float2* p, float2 v) {
  *(cplx_v*)p = cplx_v{v.x, v.y};
}

__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
  return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
// (a) * (sgn i)
__device__ __forceinline__ float2 mul_si(float2 a, float sgn) {
  return make_float2(-sgn * a.y, sgn * a.x);
}

// cos and sin of 2 pi K / 16
constexpr double kC16 = 0.92387953251128674, kS16 = 0.38268343236508977, kH16 = 0.70710678118654752;
constexpr double kCos16[10] = {1.0, kC16, kH16, kS16, 0.0, -kS16, -kH16, -kC16, -1.0, -kC16};
constexpr double kSin16[10] = {0.0, kS16, kH16, kC16, 1.0, kC16, kH16, kS16, 0.0, -kS16};

// In-register DFT of size RAD: y_q = sum_r x_r exp(sgn 2 pi i r q / RAD).
template <int RAD>
__device__ __forceinline__ void dft_reg(float2 (&x)[RAD], float sgn);

template <>
__device__ __forceinline__ void dft_reg<2>(float2 (&x)[2], float) {
  const float2 a = x[0], b = x[1];
  x[0] = make_float2(a.x + b.x, a.y + b.y);
  x[1] = make_float2(a.x - b.x, a.y - b.y);
}

template <>
__device__ __forceinline__ void dft_reg<4>(float2 (&x)[4], float sgn) {
  const float2 a0 = make_float2(x[0].x + x[2].x, x[0].y + x[2].y);
  const float2 a1 = make_float2(x[0].x - x[2].x, x[0].y - x[2].y);
  const float2 a2 = make_float2(x[1].x + x[3].x, x[1].y + x[3].y);
  const float2 a3 = mul_si(make_float2(x[1].x - x[3].x, x[1].y - x[3].y), sgn);
  x[0] = make_float2(a0.x + a2.x, a0.y + a2.y);
  x[2] = make_float2(a0.x - a2.x, a0.y - a2.y);
  x[1] = make_float2(a1.x + a3.x, a1.y + a3.y);
  x[3] = make_float2(a1.x - a3.x, a1.y - a3.y);
}

template <>
__device__ __forceinline__ void dft_reg<8>(float2 (&x)[8], float sgn) {
  float2 e[4] = {x[0], x[2], x[4], x[6]};
  float2 o[4] = {x[1], x[3], x[5], x[7]};
  dft_reg<4>(e, sgn);
  dft_reg<4>(o, sgn);
  const float h = 0.70710678118654752f;
  // o_q * exp(sgn 2 pi i q / 8)
  const float2 o1 = make_float2(h * (o[1].x - sgn * o[1].y), h * (o[1].y + sgn * o[1].x));
  const float2 o2 = mul_si(o[2], sgn);
  const float2 o3 = make_float2(h * (-o[3].x - sgn * o[3].y), h * (-o[3].y + sgn * o[3].x));
  const float2 ot[4] = {o[0], o1, o2, o3};
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    x[q] = make_float2(e[q].x + ot[q].x, e[q].y + ot[q].y);
    x[q + 4] = make_float2(e[q].x - ot[q].x, e[q].y - ot[q].y);
  }
}

// x *= exp(sgn 2 pi i K / 16), the constants as float pairs: two radix-4 steps in
// registers put these factors where a radix-8 stage has one of table and one
// multiplication by sqrt(1/2), and with single floats their roundings, the same at
// every element, cost the transform more than the saved steps gave (2048 points,
// forward and back, relative error in 1e-7: 1.60 in radix-8 stages, 1.66 with
// single constants, 1.51 with pairs).
template <int K>
__device__ __forceinline__ void twist16(float2& x, float sgn) {
  constexpr double cd = kCos16[K], sd = kSin16[K];
  constexpr float c = (float)cd, s = (float)sd, cl = (float)(cd - c), sl = (float)(sd - s);
  const float ss = sgn * s, ssl = sgn * sl;
  x = make_float2(fmaf(x.x, c, fmaf(-x.y, ss, fmaf(x.x, cl, -x.y * ssl))),
                  fmaf(x.x, ss, fmaf(x.y, c, fmaf(x.x, ssl, x.y * cl))));
}

template <>
__device__ __forceinline__ void dft_reg<16>(float2 (&x)[16], float sgn) {
  float2 a[4][4];   // [r1][q2]: DFT over r2 of x[r1 + 4 r2], times W16^(r1 q2)
#pragma unroll
  for (int r = 0; r < 4; ++r) {
#pragma unroll
    for (int q = 0; q < 4; ++q) a[r][q] = x[r + 4 * q];
    dft_reg<4>(a[r], sgn);
  }
  twist16<1>(a[1][1], sgn);
  twist16<2>(a[1][2], sgn);
  twist16<3>(a[1][3], sgn);
  twist16<2>(a[2][1], sgn);
  a[2][2] = mul_si(a[2][2], sgn);
  twist16<6>(a[2][3], sgn);
  twist16<3>(a[3][1], sgn);
  twist16<6>(a[3][2], sgn);
  twist16<9>(a[3][3], sgn);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    float2 y[4] = {a[0][q], a[1][q], a[2][q], a[3][q]};
    dft_reg<4>(y, sgn);
#pragma unroll
    for (int r = 0; r < 4; ++r) x[q + 4 * r] = y[r];
  }
}

// log2 of the radices: three stages up to 4096.  A radix-8 first stage is
// followed by radix 8 and a radix-16 one by radix 16, which the LDS layout
// needs (lin below).  256 points take three stages too: two of radix 16 leave a
// row 16 lanes, each with 16 transfer functions to form one after another, and
// the angular spectrum of eight 128^2 fields took 142 us (131 in stages of radix
// 8 on 512 threads) where these on two rows take 99; eight transforms of 256^2 15.1
// and 12.3 (33.1).
constexpr int log2_rad(int log2m, int st) {
  constexpr int kRad[14][4] = {{},        {1},       {2},       {3},       {4},
                               {3, 2},    {3, 3},    {4, 3},    {3, 3, 2}, {3, 3, 3},
                               {3, 3, 4}, {4, 4, 3}, {4, 4, 4}, {4, 4, 3, 2}};
  return kRad[log2m][st];
}
constexpr int stages(int log2m) {
  int n = 0;
  while (n < 4 && log2_rad(log2m, n) > 0) ++n;
  return n;
}
constexpr int log2_p(int log2m, int st) {   // product of the earlier radices
  int l = 0;
  for (int i = 0; i < st; ++i) l += log2_rad(log2m, i);
  return l;
}

// Twiddles exp(2 pi i r k / (p RAD)) of every stage but the first, in the order
// the stages read them: stage st at p - RAD_0, entry (r - 1) p + k for r = 1 ..
// RAD - 1 (the sizes telescope to M - RAD_0 in all), rounded from double.
template <int LOG2M>
struct Twiddles {
  float v[2 << LOG2M];
};
constexpr double kPi = 3.14159265358979323846;
constexpr double sin_small(double x) {   // |x| <= pi / 4
  const double y = x * x;
  double t = 0.0;
  for (int i = 10; i >= 1; --i) t = (1.0 + t) * (-y / ((2.0 * i) * (2.0 * i + 1.0)));
  return x * (1.0 + t);
}
constexpr double cos_small(double x) {
  const double y = x * x;
  double t = 0.0;
  for (int i = 10; i >= 1; --i) t = (1.0 + t) * (-y / ((2.0 * i - 1.0) * (2.0 * i)));
  return 1.0 + t;
}
template <int LOG2M>
constexpr Twiddles<LOG2M> make_twiddles() {
  constexpr int M = 1 << LOG2M, E = M >= 8 ? M / 8 : 1;   // an octant
  double c[E + 1] = {}, sn[E + 1] = {};
  for (int q = 0; q <= E; ++q) {
    c[q] = cos_small(2.0 * kPi * q / M);
    sn[q] = sin_small(2.0 * kPi * q / M);
  }
  Twiddles<LOG2M> t{};
  int o = 0;
  for (int st = 1; st < stages(LOG2M); ++st) {
    const int p = 1 << log2_p(LOG2M, st), rad = 1 << log2_rad(LOG2M, st);
    for (int r = 1; r < rad; ++r)
      for (int k = 0; k < p; ++k, ++o) {
        const int a = (r * k * (M / (p * rad))) % M;      // M >= 32 where there are two stages
        const int oct = a / E, f = a % E;
        const double x = oct & 1 ? sn[E - f] : c[f], y = oct & 1 ? c[E - f] : sn[f];
        const double u = (oct >> 1) & 1 ? y : x, w = (oct >> 1) & 1 ? x : y;
        t.v[2 * o] = (float)(oct >= 2 && oct < 6 ? -u : u);
        t.v[2 * o + 1] = (float)(oct >= 4 ? -w : w);
      }
  }
  return t;
}
template <int LOG2M>
__device__ constexpr Twiddles<LOG2M> kTwiddles = make_twiddles<LOG2M>();

enum FftPass {
  kFirst = 0,    // padded N x N source, rows stored transposed
  kSecond = 1,   // plain rows, stored transposed with fftshift and the scale
  kMid = 2,      // plain rows (y-lines, row index kx): forward, times H, inverse; plain rows
  kLast = 3,     // rows gathered from columns; plain rows with fftshift and the scale
};

struct FftParams {
  int N, p;         // source side and pad offset (kFirst)
  long in_bstride, out_bstride;
  float scale;
  double asm_z, asm_inv_wl2, asm_df;
  // rows_lo > 0 (kFirst): only the rows that hold the padded field, [0,
  // rows_lo) and [M - rows_lo, M), are transformed (the others are zero rows
  // whose transforms are zero); the launch has 2 rows_lo / R groups.
  // zlo < zhi (kSecond, kMid): positions [zlo, zhi) of every row load as zeros
  // (the columns the previous launch left unwritten).
  int rows_lo, zlo, zhi;
};

// The angular-spectrum transfer function at frequency indices (iy, ix) of the
// centred spectrum (-M/2 .. M/2 - 1 times df), applied to v:
// v exp(2 pi i z sqrt(1/lambda^2 - fx^2 - fy^2)) where the root is real, 0
// elsewhere.  The phase is formed in FP64 turns (tens of thousands of turns at
// millimetre distances), reduced, then taken by the hardware sin / cos
// (turns; max abs error 1.3e-7 on [-1/2, 1/2]).
__device__ __forceinline__ float2 apply_h(float2 v, int iy, int ix, const FftParams& P) {
  const double fy = (double)iy * P.asm_df, fx = (double)ix * P.asm_df;
  const double arg = P.asm_inv_wl2 - fx * fx - fy * fy;
  if (!(arg > 0.0)) return make_float2(0.f, 0.f);
  double t = P.asm_z * sqrt(arg);
  t -= rint(t);
  const float s = __builtin_amdgcn_sinf((float)t), c = __builtin_amdgcn_cosf((float)t);
  return make_float2(v.x * c - v.y * s, v.x * s + v.y * c);
}

// Threads of a workgroup: one radix-16 butterfly each.
constexpr int fft_threads(int log2m, int log2r) {
  const int t = (1 << (log2m + log2r)) / 16;
  return t < 64 ? 64 : t > 1024 ? 1024 : t;
}

// The workgroup's transforms in LDS.  Element x of row rr sits at x with the 5
// bits from bit log2 RAD_0 up XORed into its low 5 and a row term XORed in: a
// bijection on [0, M) for every row that spreads the stages' strided accesses
// and the transposed ones (one column of R rows, M apart) over the 32 8-byte
// LDS banks.  It is linear over XOR, so the positions of a butterfly differ by
// constants.
template <int LOG2M, int LOG2R>
struct RowFft {
  static constexpr int M = 1 << LOG2M, R = 1 << LOG2R, T = fft_threads(LOG2M, LOG2R);
  static constexpr int kStages = stages(LOG2M);
  static constexpr uint32_t lin(uint32_t x) { return x ^ ((x >> log2_rad(LOG2M, 0)) & 31); }
  static __device__ __forceinline__ uint32_t row_off(int rr) {
    return ((uint32_t)rr << LOG2M) | ((uint32_t)(rr * 20) & (M - 1));
  }
  // byte offset of element x of row rr
  static __device__ __forceinline__ uint32_t off(int rr, int x) {
    return (row_off(rr) ^ lin((uint32_t)x)) << 3;
  }
  static __device__ __forceinline__ float2& at(float2* buf, uint32_t byte) {
    return *(float2*)((char*)buf + byte);
  }

  // Stage ST: butterfly j of a row reads x_r = row[j + r M / RAD], twiddles
  // them by exp(sgn 2 pi i r k / (p RAD)) with k = j mod p, transforms, and
  // writes y_q to row[(j - k) RAD + k + q p].  load(v, rr, j) fills a butterfly
  // from elsewhere than LDS (SRC false); post(v, rr, i0) may change it and,
  // returning true, has stored it (element q at i0 + q p).  RFAST: consecutive
  // threads take consecutive rows.
  template <int ST, bool INV, bool SRC, bool DST, bool RFAST, typename Load, typename Post>
  static __device__ __forceinline__ void stage(float2* buf, const float2* tw, Load load, Post post) {
    constexpr float sgn = INV ? 1.f : -1.f;
    constexpr int L = log2_rad(LOG2M, ST), RAD = 1 << L, LP = log2_p(LOG2M, ST), p = 1 << LP;
    constexpr int LJ = LOG2M - L, total = R << LJ;
    constexpr int kItems = total > T ? total / T : 1;
    constexpr bool kAll = total % T == 0;
    float2 v[kItems][RAD];
#pragma unroll
    for (int it = 0; it < kItems; ++it) {
      const int t = threadIdx.x + it * T;
      if (kAll || t < total) {
        const int rr = RFAST ? t & (R - 1) : t >> LJ, j = RFAST ? t >> LOG2R : t & ((1 << LJ) - 1);
        if constexpr (SRC) {
          const uint32_t o = off(rr, j);
#pragma unroll
          for (int r = 0; r < RAD; ++r) v[it][r] = at(buf, o ^ (lin((uint32_t)r << LJ) << 3));
        } else {
          load(v[it], rr, j);
        }
      }
    }
    if constexpr (SRC && DST) __syncthreads();
#pragma unroll
    for (int it = 0; it < kItems; ++it) {
      const int t = threadIdx.x + it * T;
      if (kAll || t < total) {
        const int rr = RFAST ? t & (R - 1) : t >> LJ, j = RFAST ? t >> LOG2R : t & ((1 << LJ) - 1);
        const int k = j & (p - 1);
        if constexpr (ST > 0) {
          const float2* w = tw + (p - (1 << log2_rad(LOG2M, 0))) + k;
#pragma unroll
          for (int r = 1; r < RAD; ++r) {
            const float2 c = w[(r - 1) * p];
            v[it][r] = cmul(v[it][r], make_float2(c.x, sgn * c.y));
          }
        }
        dft_reg<RAD>(v[it], sgn);
        const int i0 = ((j - k) << L) + k;
        post(v[it], rr, i0);
        if constexpr (DST) {
          const uint32_t o = off(rr, i0);
#pragma unroll
          for (int q = 0; q < RAD; ++q) at(buf, o ^ (lin((uint32_t)q << LP) << 3)) = v[it][q];
        }
      }
    }
    if constexpr (DST) __syncthreads();
  }

  // Stages from ST: the first of the transform from `load` unless SRC, the last
  // through `post`, to LDS if DST.
  template <int ST, bool INV, bool SRC, bool DST, bool RFAST, typename Load, typename Post>
  static __device__ __forceinline__ void run(float2* buf, const float2* tw, Load load, Post post) {
    if constexpr (ST + 1 == kStages) {
      stage<ST, INV, SRC || (ST > 0), DST, RFAST && ST == 0>(buf, tw, load, post);
    } else {
      stage<ST, INV, SRC || (ST > 0), true, RFAST && ST == 0>(buf, tw, load,
                                                               [](auto&, int, int) {});
      run<ST + 1, INV, SRC, DST, RFAST>(buf, tw, load, post);
    }
  }
};

// What bounds a launch: LDS and vector work per element beside 16 bytes of HBM
// traffic.  2048^2 angular spectrum of a 1024^2 field, us per launch (first /
// mid / last), radix-8 stages with every stage and both ends through LDS: 15.8 /
// 39.1 / 25.0; this form: 12.3 / 24.5 / 16.2.
template <int LOG2M, int LOG2R, int PASS, bool INV>
__global__ void __launch_bounds__(fft_threads(LOG2M, LOG2R), 4)
fft_rows_kernel(const float2* __restrict__ in, float2* __restrict__ out, FftParams P) {
  using F = RowFft<LOG2M, LOG2R>;
  extern __shared__ float2 lds[];
  constexpr int M = F::M, R = F::R, T = F::T, half_m = M >> 1, kLast_ = F::kStages - 1;
  constexpr int LP = log2_p(LOG2M, kLast_), RADL = 1 << log2_rad(LOG2M, kLast_);
  float2* tw = lds + R * M;
  // consecutive row groups on one XCD (workgroups are dealt to the 8 XCDs
  // round-robin), so the short runs of the transposed stores (and loads) that
  // neighbouring groups access in the same cache lines meet in that XCD's L2
  const int groups = gridDim.x, total_wg = gridDim.x * gridDim.y;
  int id = blockIdx.y * groups + blockIdx.x;
  if (total_wg % 8 == 0) id = (id % 8) * (total_wg / 8) + id / 8;
  const int b = id / groups;
  int r0 = (id - b * groups) * R;
  if (P.rows_lo > 0 && r0 >= P.rows_lo) r0 += M - 2 * P.rows_lo;
  const float2* src = in + (long)b * P.in_bstride;
  float2* dst = out + (long)b * P.out_bstride;

  if constexpr (F::kStages > 1) {   // read after the first stage's barrier
    const float2* g = (const float2*)kTwiddles<LOG2M>.v;
    constexpr int n = M - (1 << log2_rad(LOG2M, 0));
#pragma unroll
    for (int q0 = 0; q0 < n; q0 += T) {
      const int q = q0 + threadIdx.x;
      if (q < n) tw[q] = g[q];
    }
  }

  auto load = [&](auto& v, int rr, int j) __attribute__((always_inline)) {
    constexpr int RAD = sizeof(v) / sizeof(float2), step = M / RAD;
    if constexpr (PASS == kFirst) {
      const int sr = ((r0 + rr + half_m) & (M - 1)) - P.p;
      const bool row_ok = sr >= 0 && sr < P.N;
      const float2* row = src + (long)(row_ok ? sr : 0) * P.N;
#pragma unroll
      for (int r = 0; r < RAD; ++r) {
        const int sc = ((j + r * step + half_m) & (M - 1)) - P.p;
        const bool ok = row_ok && sc >= 0 && sc < P.N;   // loads stay unconditional, in flight
        const float2 x = row[ok ? sc : 0];
        v[r] = ok ? x : make_float2(0.f, 0.f);
      }
    } else if constexpr (PASS == kLast) {
#pragma unroll
      for (int r = 0; r < RAD; ++r) v[r] = src[(long)(j + r * step) * M + r0 + rr];
    } else {
      const float2* row = src + (long)(r0 + rr) * M;
#pragma unroll
      for (int r = 0; r < RAD; ++r) {
        const int y = j + r * step;
        const bool ok = y < P.zlo || y >= P.zhi;
        const float2 x = row[ok ? y : 0];
        v[r] = ok ? x : make_float2(0.f, 0.f);
      }
    }
  };
  auto none = [](auto&, int, int) {};
  if constexpr (PASS == kMid) {
    F::template run<0, false, false, true, false>(
        lds, tw, load, [&](auto& v, int rr, int i0) __attribute__((always_inline)) {
          const int ix = ((r0 + rr + half_m) & (M - 1)) - half_m;
#pragma unroll
          for (int q = 0; q < RADL; ++q)
            v[q] = apply_h(v[q], ((i0 + (q << LP) + half_m) & (M - 1)) - half_m, ix, P);
        });
    F::template run<0, true, true, false, false>(
        lds, tw, load, [&](auto& v, int rr, int i0) __attribute__((always_inline)) {
#pragma unroll
          for (int q = 0; q < RADL; ++q)
            store_c64(dst + (long)(r0 + rr) * M + i0 + (q << LP), v[q]);
        });
  } else if constexpr (PASS == kLast) {
    F::template run<0, INV, false, false, true>(
        lds, tw, load, [&](auto& v, int rr, int i0) __attribute__((always_inline)) {
          const int oy = (r0 + rr + half_m) & (M - 1);
#pragma unroll
          for (int q = 0; q < RADL; ++q) {
            const int ox = (i0 + (q << LP) + half_m) & (M - 1);
            store_c64(dst + (long)oy * M + ox, make_float2(v[q].x * P.scale, v[q].y * P.scale));
          }
        });
  } else {
    F::template run<0, INV, false, true, false>(lds, tw, load, none);
    // transposed store: out[k][row] (consecutive lanes -> consecutive rows)
    constexpr int kPer = R * M > T ? R * M / T : 1;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int t = threadIdx.x + i * T;
      if (R * M % T == 0 || t < R * M) {
        const int k = t >> LOG2R, rr = t & (R - 1), row = r0 + rr;
        float2 v = F::at(lds, F::off(rr, k));
        if constexpr (PASS == kFirst) {
          store_c64(dst + (long)k * M + row, v);
        } else {
          const int oy = (k + half_m) & (M - 1), ox = (row + half_m) & (M - 1);
          store_c64(dst + (long)oy * M + ox, make_float2(v.x * P.scale, v.y * P.scale));
        }
      }
    }
  }
}

// log2 of the rows per workgroup for length-M rows: within the 160 KiB of LDS
// beside the twiddles, enough for long runs in the transposed accesses while
// that leaves one workgroup per CU.  2048^2, us at 2 / 4 / 8 rows: kFirst (1024
// rows) 14.4 / 11.8 / 12.0, kLast 20.3 / 17.0 / 15.6; kMid has no transposed
// access, and two workgroups on a CU overlap: 26.4 / 24.2 at 2 / 4 (1: 31.4).
// 64 transforms of 256^2, us at 1 / 2 rows: 55.2 / 35.9.
constexpr int log2_rows(int log2m, int pass) {
  return log2m <= 7 ? 0 : log2m <= 9 ? 1 : log2m == 11 && pass != kMid ? 3 : log2m <= 12 ? 2 : 0;
}

template <int LOG2M, int LOG2R, int PASS, bool INV>
hipError_t launch_rows_r(const float2* in, float2* out, int batch, const FftParams& P,
                         hipStream_t s) {
  constexpr size_t lds = ((size_t)(1 << (LOG2M + LOG2R)) + (1 << LOG2M)) * sizeof(float2);
  if constexpr (lds > 64 * 1024) {
    // Opt in to more than 64 KiB of dynamic LDS (gfx950 has 160 KiB per CU).
    (void)hipFuncSetAttribute((const void*)fft_rows_kernel<LOG2M, LOG2R, PASS, INV>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    (void)hipGetLastError();
  }
  const int rows = P.rows_lo > 0 ? 2 * P.rows_lo : 1 << LOG2M;
  hipLaunchKernelGGL((fft_rows_kernel<LOG2M, LOG2R, PASS, INV>), dim3(rows >> LOG2R, batch),
                     dim3(fft_threads(LOG2M, LOG2R)), lds, s, in, out, P);
  return hipGetLastError();
}

template <int PASS, bool INV, int LOG2M = 1>
hipError_t launch_rows(int log2m, const float2* in, float2* out, int batch, const FftParams& P,
                       hipStream_t s) {
  if constexpr (LOG2M > 13) {
    return hipErrorInvalidValue;
  } else {
    if (log2m != LOG2M) return launch_rows<PASS, INV, LOG2M + 1>(log2m, in, out, batch, P, s);
    constexpr int R = log2_rows(LOG2M, PASS);
    if constexpr (PASS == kFirst && R > 0) {
      // a launch over the field's rows alone has fewer groups: halve the rows per
      // group while there are fewer than 256
      int r = R;
      if (P.rows_lo > 0)
        while (r > 0 && ((2 * P.rows_lo) >> r < 256 || P.rows_lo % (1 << r))) --r;
      if constexpr (R > 2)
        if (r == 2) return launch_rows_r<LOG2M, 2, PASS, INV>(in, out, batch, P, s);
      if constexpr (R > 1)
        if (r == 1) return launch_rows_r<LOG2M, 1, PASS, INV>(in, out, batch, P, s);
      if (r == 0) return launch_rows_r<LOG2M, 0, PASS, INV>(in, out, batch, P, s);
    }
    return launch_rows_r<LOG2M, R, PASS, INV>(in, out, batch, P, s);
  }
}

int ilog2(int m) {
  int l = 0;
  while ((1 << l) < m) ++l;
  return l;
}

}  // namespace

// Maximum transform side (one row + twiddles fit in LDS).
constexpr int kMaxFftSide = 8192;

bool fft_supported(int m) { return m >= 2 && m <= kMaxFftSide && (m & (m - 1)) == 0; }

// A launch over the rows of an N x N field padded to M x M (ifftshifted):
// the rows that hold the field are [0, N/2) and [M - N/2, M); transform only
// those when N/2 is a multiple of the middle pass's rows per workgroup.  The launch after it
// reads, in each of its rows, the positions the others would have written as
// zeros.
static FftParams first_params(int N, int M) {
  FftParams A{};
  A.N = N;
  A.p = (M - N) / 2;
  A.in_bstride = (long)N * N;
  A.out_bstride = (long)M * M;
  const int half = N / 2;
  A.rows_lo = N < M && half > 0 && half % (1 << log2_rows(ilog2(M), kMid)) == 0 ? half : 0;
  return A;
}
static FftParams next_params(const FftParams& A, int M) {
  FftParams B = A;
  B.rows_lo = 0;
  B.in_bstride = (long)M * M;
  B.zlo = A.rows_lo;
  B.zhi = A.rows_lo > 0 ? M - A.rows_lo : 0;
  return B;
}

// Full centred 2-D transform of `batch` N x N fields, padded to M x M.
// tmp: batch * M * M complex64 scratch.
hipError_t launch_fft2_centred(const float2* in, int N, int M, int batch, int inverse,
                               float scale, float2* tmp, float2* out, hipStream_t s) {
  const int l = ilog2(M);
  const FftParams A = first_params(N, M);
  hipError_t e = inverse ? launch_rows<kFirst, true>(l, in, tmp, batch, A, s)
                         : launch_rows<kFirst, false>(l, in, tmp, batch, A, s);
  if (e != hipSuccess) return e;
  FftParams B = next_params(A, M);
  B.scale = scale;
  return inverse ? launch_rows<kSecond, true>(l, tmp, out, batch, B, s)
                 : launch_rows<kSecond, false>(l, tmp, out, batch, B, s);
}

// Angular-spectrum propagation of one N x N field padded to M x M:
// out = fftshift(ifft2(fft2(ifftshift(pad x)) H')) with H' the transfer
// function at the natural-order frequencies -- the centred forward and
// inverse transforms with their fftshift / ifftshift pairs cancelled between
// them.  Three launches: x transforms of the padded field (transposed store);
// per y-line (fixed kx) the forward y transform, H', and the inverse y
// transform; the inverse x transforms of rows gathered from columns, stored
// with fftshift and the 1/M^2 scale.
hipError_t launch_asm(const float2* in, int N, int M, double z, double wavelength, double dx,
                      float2* tmp, float2* tmp2, float2* out, hipStream_t s) {
  const int l = ilog2(M);
  const FftParams A = first_params(N, M);
  hipError_t e = launch_rows<kFirst, false>(l, in, tmp, 1, A, s);
  if (e != hipSuccess) return e;
  FftParams B = next_params(A, M);
  B.asm_z = z;
  B.asm_inv_wl2 = 1.0 / (wavelength * wavelength);
  B.asm_df = 1.0 / ((double)M * dx);
  e = launch_rows<kMid, false>(l, tmp, tmp2, 1, B, s);
  if (e != hipSuccess) return e;
  B.scale = (float)(1.0 / ((double)M * M));
  return launch_rows<kLast, true>(l, tmp2, out, 1, B, s);
}

}  // namespace dlx

using namespace dlx;

extern "C" size_t dlx_fft2_workspace_size(int32_t n, int32_t m, int32_t batch) {
  (void)n;
  if (m <= 0 || batch <= 0) return 0;
  return align_up((size_t)batch * m * m * sizeof(float2));
}

extern "C" int dlx_fft2(int32_t n, int32_t m, int32_t batch, int32_t inverse, const void* in,
                        void* out, void* workspace, size_t workspace_bytes, void* stream) {
  clear_error();
  DLX_CHECK_ARG(n > 0 && m >= n && batch >= 0, "need 0 < n <= m and batch >= 0");
  DLX_CHECK_ARG(batch <= 65535, "batch must be <= 65535, got %d", batch);
  DLX_CHECK_ARG(((m - n) % 2) == 0, "m - n must be even (centre-preserving pad)");
  if (batch == 0) return DLX_OK;
  DLX_CHECK_ARG(in && out, "null argument to dlx_fft2");
  if (!fft_supported(m)) {
    set_error("dlx_fft2 supports power-of-two sides up to %d, got %d", kMaxFftSide, m);
    return DLX_ERR_UNSUPPORTED;
  }
  const size_t need = dlx_fft2_workspace_size(n, m, batch);
  if (!workspace || workspace_bytes < need) {
    set_error("dlx_fft2 workspace too small: need %zu bytes, got %zu", need, workspace_bytes);
    return DLX_ERR_WORKSPACE;
  }
  DLX_HIP(launch_fft2_centred((const float2*)in, n, m, batch, inverse, 1.0f / (float)m,
                              (float2*)workspace, (float2*)out, (hipStream_t)stream));
  return DLX_OK;
}

extern "C" size_t dlx_asm_workspace_size(int32_t n, int32_t m, int32_t batch) {
  if (m <= 0 || batch <= 0) return 0;
  return 2 * dlx_fft2_workspace_size(n, m, batch);
}

extern "C" int dlx_asm_prop(int32_t n, int32_t m, int32_t batch, const double* wavelength,
                            double pixel_scale, double distance, const void* in, void* out,
                            void* workspace, size_t workspace_bytes, void* stream) {
  clear_error();
  DLX_CHECK_ARG(n > 0 && m >= n && batch >= 0, "need 0 < n <= m and batch >= 0");
  DLX_CHECK_ARG(batch <= 65535, "batch must be <= 65535, got %d", batch);
  DLX_CHECK_ARG(((m - n) % 2) == 0, "m - n must be even (centre-preserving pad)");
  if (batch == 0) return DLX_OK;
  DLX_CHECK_ARG(in && out && wavelength, "null argument to dlx_asm_prop");
  DLX_CHECK_ARG(std::isfinite(pixel_scale) && pixel_scale > 0, "pixel_scale must be > 0");
  DLX_CHECK_ARG(std::isfinite(distance), "distance must be finite");
  if (!fft_supported(m)) {
    set_error("dlx_asm_prop supports power-of-two padded sides up to %d, got %d", kMaxFftSide,
              m);
    return DLX_ERR_UNSUPPORTED;
  }
  const size_t need = dlx_asm_workspace_size(n, m, batch);
  if (!workspace || workspace_bytes < need) {
    set_error("dlx_asm_prop workspace too small: need %zu bytes, got %zu", need,
              workspace_bytes);
    return DLX_ERR_WORKSPACE;
  }
  hipStream_t s = (hipStream_t)stream;
  const size_t slab = dlx_fft2_workspace_size(n, m, batch);
  float2* tmp = (float2*)workspace;
  float2* spec = (float2*)((char*)workspace + slab);
  for (int b = 0; b < batch; ++b) {
    DLX_CHECK_ARG(std::isfinite(wavelength[b]) && wavelength[b] > 0,
                  "wavelength[%d] must be > 0", b);
    DLX_HIP(launch_asm((const float2*)in + (long)b * n * n, n, m, distance, wavelength[b],
                       pixel_scale, tmp + (long)b * m * m, spec + (long)b * m * m,
                       (float2*)out + (long)b * m * m, s));
  }
  return DLX_OK;
}
