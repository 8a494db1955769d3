// The folded MFT's kernels (dlx_fold.h): cosine / sine tables, the pupil and
// field loaders, and the two contractions with their epilogues, in complex64
// (v_mfma_f32_32x32x2_f32) and split-BF16x3 form (v_mfma_f32_32x32x16_bf16,
// hi*hi + hi*lo + lo*hi), on one tile geometry: both forms hold 4 bytes per
// real, so a stage of 16 k is 64 bytes of every tile row -- four 16-byte
// pieces, of which a lane's half (lane / 32) takes two:
//   split-BF16x3  [hi k 0-7][lo k 0-7][hi k 8-15][lo k 8-15]
//   float32       [k 0-3][k 4-7][k 8-11][k 12-15]; MFMA e pairs k = e and 8 + e
// Tile row r keeps piece p at slot p ^ ((r >> 2) & 3), so 16 consecutive rows
// reading one piece touch all 16 bank groups of 16 bytes.
#include "dlx_fold.h"

#include <type_traits>

#include "dlx_phasor.h"
#include "dlx_split.h"

namespace dlx {
namespace {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16_t;
typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t u32x4_t;
typedef __attribute__((address_space(3))) void lds_void_t;
typedef const __attribute__((address_space(1))) void gbl_void_t;

constexpr int kThreads = 256;   // 4 waves
constexpr int kStageK = 16;     // k per stage
constexpr int kRow = 64;        // bytes of a tile row per stage
constexpr int kXcds = 8;

// Hardware workgroup id -> logical id such that consecutive logical ids land
// on the same XCD (hardware deals workgroups round-robin over 8 XCDs).
__device__ __forceinline__ int xcd_order(int hw, int total) {
  const int per = total / kXcds;
  if (hw >= per * kXcds) return hw;   // tail that does not fill all XCDs evenly
  return (hw % kXcds) * per + hw / kXcds;
}

__device__ __forceinline__ float quad_swap1(float v) {   // the value of lane ^ 1
  return __uint_as_float(quad_xor<1>(__float_as_uint(v)));
}

// ---------------------------------------------------------------------------
// tiles
// ---------------------------------------------------------------------------

// Direct-to-LDS loader of a ROWS-row tile: one wave instruction fills 16 rows
// (1 KiB); each thread's source pointers are formed once and advance by one
// stage.
template <int ROWS>
struct TileRows {
  const uint8_t* p[ROWS / 64];
  template <typename F>
  __device__ __forceinline__ void init(F row_ptr) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int piece = (lane & 3) ^ ((lane >> 4) & 3);
#pragma unroll
    for (int q = 0; q < ROWS / 64; ++q)
      p[q] = row_ptr(64 * q + 16 * wave + (lane >> 2)) + piece * 16;
  }
  __device__ __forceinline__ void issue(uint8_t* tile, int s) const {
    const int wave = threadIdx.x >> 6;
#pragma unroll
    for (int q = 0; q < ROWS / 64; ++q)
      __builtin_amdgcn_global_load_lds((gbl_void_t*)(p[q] + (long)s * kRow),
                                       (lds_void_t*)(tile + (64 * q + 16 * wave) * kRow), 16, 0, 0);
  }
};

// A lane's two pieces of tile row row0 + lane % 32 (row0 a multiple of 32).
__device__ __forceinline__ void read_frag(u32x4_t (&f)[2], const uint8_t* tile, int row0) {
  const int lane = threadIdx.x & 63, lr = lane & 31, lk = lane >> 5;
  const uint8_t* r = tile + (row0 + lr) * kRow;
#pragma unroll
  for (int j = 0; j < 2; ++j) f[j] = *(const u32x4_t*)(r + (((2 * lk + j) ^ ((lr >> 2) & 3)) << 4));
}

// acc[i][j] += sum over the stage's 16 k of a_i(m) b_j(n): lane holds column
// n = lane % 32, register r row m = 8 (r / 4) + 4 (lane / 32) + r % 4.
template <bool BF, int NI, int NJ>
__device__ __forceinline__ void mma_stage(f32x16_t (&acc)[NI][NJ], const u32x4_t (&a)[NI][2],
                                          const u32x4_t (&b)[NJ][2]) {
  if constexpr (BF) {
    // lo*hi, hi*lo, hi*hi: the small terms first
#pragma unroll
    for (int t = 0; t < 3; ++t)
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              __builtin_bit_cast(bf16x8_t, a[i][t == 0 ? 1 : 0]),
              __builtin_bit_cast(bf16x8_t, b[j][t == 1 ? 1 : 0]), acc[i][j], 0, 0, 0);
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(
              __uint_as_float(a[i][e >> 2][e & 3]), __uint_as_float(b[j][e >> 2][e & 3]),
              acc[i][j], 0, 0, 0);
  }
}

template <int NI, int NJ>
__device__ __forceinline__ void zero_acc(f32x16_t (&acc)[NI][NJ]) {
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
}

// Four consecutive k (k4 .. k4 + 3 of a 16-k stage, k4 a multiple of 4) of one
// row: the piece and byte they occupy.
template <bool BF>
__device__ __forceinline__ void put4(uint8_t* row, int quad, int f, const float (&v)[4]) {
  if constexpr (BF) {
    uint32_t h[2], l[2];
    split2_bf16(v[0], v[1], h[0], l[0]);
    split2_bf16(v[2], v[3], h[1], l[1]);
    const int p = quad & 2, o = (quad & 1) * 8;
    *(uint2*)(row + ((p ^ f) << 4) + o) = make_uint2(h[0], h[1]);
    *(uint2*)(row + (((p + 1) ^ f) << 4) + o) = make_uint2(l[0], l[1]);
  } else {
    *(float4*)(row + ((quad ^ f) << 4)) = make_float4(v[0], v[1], v[2], v[3]);
  }
}

// ---------------------------------------------------------------------------
// Field loaders.  Thread t of a workgroup takes row py = t / 8 of a 32-row
// tile, its mirror side t % 2 and four k of the stage ((t / 2) % 4): it loads
// both mirrored runs of its row, folds along x, and folds along y with lane
// t ^ 1, which leaves it the parts of beta = t % 2.
// ---------------------------------------------------------------------------
struct FoldPart {
  float v[2][2][4];   // [alpha][c][k]
};

// x and y folds; vp / vm: the values at k+ and k- of the thread's own row.
__device__ __forceinline__ void fold_x(const float2 (&vp)[4], const float2 (&vm)[4], FoldPart& o) {
#pragma clang fp contract(off)
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    o.v[0][0][e] = vp[e].x + vm[e].x;
    o.v[0][1][e] = vp[e].y + vm[e].y;
    o.v[1][0][e] = vp[e].x - vm[e].x;
    o.v[1][1][e] = vp[e].y - vm[e].y;
  }
}
__device__ __forceinline__ void fold_y(FoldPart& o, int beta) {
  const float sg = beta ? -1.f : 1.f;   // lane beta = 1 (row y-): v(y+) - v(y-)
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        o.v[a][c][e] = __builtin_fmaf(o.v[a][c][e], sg, quad_swap1(o.v[a][c][e]));
}

// The pupil loader of one thread.  VEC: n a multiple of 8 and 16-byte aligned
// planes (float4 loads; a run of four is whole or absent).
template <bool VEC>
struct PupilLoad {
  const float *opd, *amp, *phase;   // rows, or null
  int n, kh, quad, x0i;     // x0i = n / 2: the first positive column
  bool row_ok, tilted;
  double inv_wl, tx, tyY, dx, x0;
  float scale;
  float4 op, om, ap, am;    // plus and minus runs; minus in memory order (VEC) / reversed index

  __device__ __forceinline__ void init(const FoldPupil& p, int n_, int py, int beta, int quad_,
                                       double inv) {
    n = n_; kh = (n + 1) >> 1; quad = quad_; x0i = n >> 1;
    row_ok = py < kh;
    const int yp = x0i + (row_ok ? py : 0);
    const int y = beta ? n - 1 - yp : yp;
    opd = p.opd ? p.opd + (long)y * n : nullptr;
    amp = p.amp ? p.amp + (long)y * n : nullptr;
    phase = p.phase ? p.phase + (long)y * n : nullptr;
    inv_wl = inv; tx = p.tx; dx = p.dx; x0 = p.x0; scale = p.scale;
    tilted = p.tx != 0.0 || p.ty != 0.0;
    tyY = p.ty * pupil_coord(y, p.dx, p.x0);
  }
  __device__ __forceinline__ void raw(int s) {
    int p = s * kStageK + quad * 4;
    if constexpr (VEC) {
      p = p < kh ? p : 0;
      const int xp = x0i + p, xm = x0i - 4 - p;
      op = opd ? *(const float4*)(opd + xp) : make_float4(0.f, 0.f, 0.f, 0.f);
      om = opd ? *(const float4*)(opd + xm) : make_float4(0.f, 0.f, 0.f, 0.f);
      ap = amp ? *(const float4*)(amp + xp) : make_float4(1.f, 1.f, 1.f, 1.f);
      am = amp ? *(const float4*)(amp + xm) : make_float4(1.f, 1.f, 1.f, 1.f);
    } else {
      int xp[4], xm[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int pc = p + e < kh ? p + e : kh - 1;
        xp[e] = x0i + pc;
        xm[e] = n - 1 - xp[e];
      }
      op = opd ? make_float4(opd[xp[0]], opd[xp[1]], opd[xp[2]], opd[xp[3]])
               : make_float4(0.f, 0.f, 0.f, 0.f);
      om = opd ? make_float4(opd[xm[3]], opd[xm[2]], opd[xm[1]], opd[xm[0]])
               : make_float4(0.f, 0.f, 0.f, 0.f);
      ap = amp ? make_float4(amp[xp[0]], amp[xp[1]], amp[xp[2]], amp[xp[3]])
               : make_float4(1.f, 1.f, 1.f, 1.f);
      am = amp ? make_float4(amp[xm[3]], amp[xm[2]], amp[xm[1]], amp[xm[0]])
               : make_float4(1.f, 1.f, 1.f, 1.f);
    }
  }
  __device__ __forceinline__ void part(int s, int beta, FoldPart& o) const {
    const int p = s * kStageK + quad * 4;
    const float vop[4] = {op.x, op.y, op.z, op.w}, vom[4] = {om.w, om.z, om.y, om.x};
    const float vap[4] = {ap.x, ap.y, ap.z, ap.w}, vam[4] = {am.w, am.z, am.y, am.x};
    float2 vp[4], vm[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool ok = row_ok && p + e < kh;
      const int xp = x0i + p + e, xm = n - 1 - xp;
      double tp = 0.0, tm = 0.0;
      if (phase) {   // rare: not prefetched with the others
        tp = ok ? (double)phase[xp] * 0.15915494309189535 : 0.0;   // 1 / (2 pi)
        tm = ok ? (double)phase[xm] * 0.15915494309189535 : 0.0;
      }
      double pp = (double)vop[e], pm = (double)vom[e];
      if (tilted) {
        pp = pupil_path(tx, pupil_coord(xp, dx, x0), tyY, pp);
        pm = pupil_path(tx, pupil_coord(xm, dx, x0), tyY, pm);
      }
      vp[e] = pupil_phasor(pp, inv_wl, tp, scale * vap[e]);
      vm[e] = pupil_phasor(pm, inv_wl, tm, scale * vam[e]);
      if (!ok) vp[e] = vm[e] = make_float2(0.f, 0.f);
    }
    fold_x(vp, vm, o);
    fold_y(o, beta);
  }
};

// exp(2 pi i t), t in turns (any size): max abs error 1.3e-7.
__device__ __forceinline__ float2 turn(double t) {
  t -= rint(t);
  return make_float2(__builtin_amdgcn_cosf((float)t), __builtin_amdgcn_sinf((float)t));
}
__device__ __forceinline__ float2 cmul(float2 a, float2 w) {
  return make_float2(a.x * w.x - a.y * w.y, a.x * w.y + a.y * w.x);
}

// The complex64 field loader of one thread.  VEC as above.  The phase is
// formed from its FP64 coefficients as the field is folded: the x factor on
// the loaded values (its linear part is conjugate at k-), the y factor, one
// per thread, between the x and the y fold.
template <bool VEC>
struct FieldLoad {
  const float2* row;
  double c2, cx, o;     // o: the centred index of the first positive column
  float2 ry;
  int n, kh, quad, x0i;
  bool row_ok, phased;
  float4 fp[2], fm[2];  // plus run (k ascending), minus run in memory order

  __device__ __forceinline__ void init(const uint8_t* src, const FoldPhase& ph, int n_, int py,
                                       int beta, int quad_) {
    n = n_; kh = (n + 1) >> 1; quad = quad_; x0i = n >> 1;
    row_ok = py < kh;
    const int pc = row_ok ? py : 0;
    const int yp = x0i + pc;
    row = (const float2*)src + (long)(beta ? n - 1 - yp : yp) * n;
    c2 = ph.c2; cx = ph.cx;
    phased = ph.c2 != 0.0 || ph.cx != 0.0 || ph.cy != 0.0;
    o = (n & 1) ? 0.0 : 0.5;
    const double u = beta ? -((double)pc + o) : (double)pc + o;
    ry = turn(fma(c2 * u, u, ph.cy * u));
  }
  __device__ __forceinline__ void raw(int s) {
    int p = s * kStageK + quad * 4;
    if constexpr (VEC) {
      p = p < kh ? p : 0;
      const float2 *a = row + x0i + p, *b = row + x0i - 4 - p;
      fp[0] = *(const float4*)a; fp[1] = *(const float4*)(a + 2);
      fm[0] = *(const float4*)b; fm[1] = *(const float4*)(b + 2);
    } else {
      float2 a[4], b[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int pc = p + e < kh ? p + e : kh - 1;
        a[e] = row[x0i + pc];
        b[3 - e] = row[n - 1 - x0i - pc];
      }
      fp[0] = make_float4(a[0].x, a[0].y, a[1].x, a[1].y);
      fp[1] = make_float4(a[2].x, a[2].y, a[3].x, a[3].y);
      fm[0] = make_float4(b[0].x, b[0].y, b[1].x, b[1].y);
      fm[1] = make_float4(b[2].x, b[2].y, b[3].x, b[3].y);
    }
  }
  __device__ __forceinline__ void part(int s, int beta, FoldPart& out) const {
    const int p = s * kStageK + quad * 4;
    float2 vp[4] = {{fp[0].x, fp[0].y}, {fp[0].z, fp[0].w}, {fp[1].x, fp[1].y}, {fp[1].z, fp[1].w}};
    float2 vm[4] = {{fm[1].z, fm[1].w}, {fm[1].x, fm[1].y}, {fm[0].z, fm[0].w}, {fm[0].x, fm[0].y}};
    if (phased) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const double u = (double)(p + e) + o;
        const float2 w = turn(fma(c2 * u, u, cx * u));
        vp[e] = cmul(vp[e], w);
        vm[e] = cmul(vm[e], c2 != 0.0 ? turn(fma(c2 * u, u, -cx * u)) : make_float2(w.x, -w.y));
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (!(row_ok && p + e < kh)) vp[e] = vm[e] = make_float2(0.f, 0.f);
    fold_x(vp, vm, out);
    if (phased) {
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float2 w = cmul(make_float2(out.v[a][0][e], out.v[a][1][e]), ry);
          out.v[a][0][e] = w.x;
          out.v[a][1][e] = w.y;
        }
    }
    fold_y(out, beta);
  }
};

// ---------------------------------------------------------------------------
// Row store of a 32 x 32 block whose lane holds folded row lane % 32 and whose
// registers run along k: assembled in a wave-private LDS patch (rows 144 bytes
// apart) and written as 128-byte row runs, 16 bytes a lane (a lane's own
// 8- and 16-byte pieces of 32 rows would each be a request of their own).
// k beyond kvalid is written as zero.
// ---------------------------------------------------------------------------
constexpr int kPatchRow = 144, kPatch = 32 * kPatchRow;

template <bool BF>
__device__ __forceinline__ void store_block(uint8_t* patch, const f32x16_t& acc, int kvalid,
                                            uint8_t* out, long row_bytes, int rows) {
  const int lane = threadIdx.x & 63, lr = lane & 31, lk = lane >> 5;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int k = 8 * q + 4 * lk;
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = k + e < kvalid ? acc[4 * q + e] : 0.f;
    uint8_t* d = patch + lr * kPatchRow + q * 32;
    if constexpr (BF) {
      uint32_t h[2], l[2];
      split2_bf16(v[0], v[1], h[0], l[0]);
      split2_bf16(v[2], v[3], h[1], l[1]);
      *(uint2*)(d + lk * 8) = make_uint2(h[0], h[1]);
      *(uint2*)(d + 16 + lk * 8) = make_uint2(l[0], l[1]);
    } else {
      *(float4*)(d + lk * 16) = make_float4(v[0], v[1], v[2], v[3]);
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int r = 8 * t + (lane >> 3), piece = lane & 7;
    const uint4 v = *(const uint4*)(patch + r * kPatchRow + piece * 16);
    if (r < rows) *(uint4*)(out + (long)r * row_bytes + piece * 16) = v;
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---------------------------------------------------------------------------
// Stage 1: U[(beta, alpha, c), qx][py] = sum_px T_alpha[qx][px] P[(alpha, beta, c), py][px].
// A workgroup takes 32 rows py of all eight (alpha, beta, c) parts -- the four
// mirrored pixels of a loaded quad feed both alphas -- and BNQ outputs qx: at
// 128 the field is formed once per 128-column tile (256 outputs), each wave
// holds eight 32 x 32 blocks (12 fragment reads per 24 MFMAs of a split
// stage), and two workgroups share a CU.  Launches with fewer tiles take 64 or
// 32 columns.
// ---------------------------------------------------------------------------
struct Stage1Prob {
  const uint8_t* src;
  const uint8_t* table;
  uint8_t* out;
  int n, m;
};

template <bool BF, int LOAD, bool VEC, int BNQ>
__device__ __forceinline__ void stage1_tile(uint8_t* lds, const Stage1Prob& g, const FoldPupil& pup,
                                            double inv_wl, const FoldPhase& ph, int py0, int q0) {
  constexpr int kA = 256 * kRow, kBuf = kA + 2 * BNQ * kRow;
  constexpr int NI = BNQ >= 64 ? 4 : 2, NJ = BNQ >= 64 ? BNQ / 64 : 1;
  const int kh = (g.n + 1) >> 1, mh = (g.m + 1) >> 1;
  const int mhp = fold_pad(mh);
  const long rb = 4L * fold_pad(kh);
  const int nst = (kh + kStageK - 1) / kStageK;
  const int wave = threadIdx.x >> 6, alpha = wave >> 1;
  const int arow = alpha * 128 + (BNQ >= 64 ? 0 : (wave & 1) * 64);
  const int brow = alpha * BNQ + (BNQ >= 64 ? (wave & 1) * (BNQ / 2) : 0);

  f32x16_t acc[NI][NJ];
  zero_acc(acc);
  TileRows<2 * BNQ> bt;
  bt.init([&](int r) {
    const int a = r / BNQ, q = q0 + r % BNQ;
    return g.table + (long)(a * mhp + (q < mhp ? q : mhp - 1)) * rb;
  });
  TileRows<256> at;
  PupilLoad<VEC> pl;
  FieldLoad<VEC> fl;
  const int py = threadIdx.x >> 3, beta = threadIdx.x & 1, quad = (threadIdx.x >> 1) & 3;
  if constexpr (LOAD == FOLD_MEM) {
    at.init([&](int r) {
      const int y = py0 + (r & 31);
      return g.src + (long)((r >> 5) * kh + (y < kh ? y : kh - 1)) * rb;
    });
  } else if constexpr (LOAD == FOLD_PUPIL) {
    pl.init(pup, g.n, py0 + py, beta, quad, inv_wl);
  } else {
    fl.init(g.src, ph, g.n, py0 + py, beta, quad);
  }
  auto raw = [&](int s) {
    if constexpr (LOAD == FOLD_PUPIL) pl.raw(s);
    if constexpr (LOAD == FOLD_FIELD) fl.raw(s);
  };
  auto convert = [&](int s) {
    if constexpr (LOAD != FOLD_MEM) {
      FoldPart o;
      if constexpr (LOAD == FOLD_PUPIL) pl.part(s, beta, o);
      else fl.part(s, beta, o);
      uint8_t* buf = lds + (s & 1) * kBuf;
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int c = 0; c < 2; ++c)
          put4<BF>(buf + (((a * 2 + beta) * 2 + c) * 32 + py) * kRow, quad, (py >> 2) & 3, o.v[a][c]);
    }
  };
  auto issue = [&](int s) {
    uint8_t* buf = lds + (s & 1) * kBuf;
    if constexpr (LOAD == FOLD_MEM) at.issue(buf, s);
    bt.issue(buf + kA, s);
  };

  raw(0);
  issue(0);
  convert(0);
  for (int s = 0; s < nst; ++s) {
    __builtin_amdgcn_s_waitcnt(0);   // this wave's part of stage s is in LDS
    __syncthreads();                 // every wave's is; stage s - 1 has been read
    const uint8_t* la = lds + (s & 1) * kBuf;
    u32x4_t fa[NI][2], fb[NJ][2];
#pragma unroll
    for (int j = 0; j < NJ; ++j) read_frag(fb[j], la + kA, brow + 32 * j);
#pragma unroll
    for (int i = 0; i < NI; ++i) read_frag(fa[i], la, arow + 32 * i);
    const bool more = s + 1 < nst;
    if (more) {
      raw(s + 1);
      issue(s + 1);
    }
    __builtin_amdgcn_s_setprio(1);
    mma_stage<BF, NI, NJ>(acc, fa, fb);
    __builtin_amdgcn_s_setprio(0);
    if (more) convert(s + 1);
  }
  __syncthreads();
  uint8_t* patch = lds + wave * kPatch;
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      // A rows run (beta, c) within alpha
      const int bc = BNQ >= 64 ? i : (wave & 1) * 2 + i;
      const int comp = ((bc >> 1) * 2 + alpha) * 2 + (bc & 1);
      const int q = q0 + (brow - alpha * BNQ) + 32 * j;
      if (q < mh)
        store_block<BF>(patch, acc[i][j], kh - py0, g.out + (long)(comp * mh + q) * rb + 4L * py0,
                        rb, mh - q);
    }
}

template <bool BF, int LOAD, bool VEC, int BNQ>
__global__ void __launch_bounds__(kThreads, 2)
fold_stage1_kernel(FoldStage1 a) {
  constexpr int kBuf = (256 + 2 * BNQ) * kRow;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[2 * kBuf];
  const int tq = (fold_half(a.m) + BNQ - 1) / BNQ, tp = (fold_half(a.n) + 31) / 32;
  const int id = xcd_order(blockIdx.x, tq * tp * a.batch);
  const int b = id / (tq * tp), t = id - b * (tq * tp);
  Stage1Prob g;
  g.src = a.src ? a.src + (long)b * a.src_stride : nullptr;
  g.table = a.table + (long)b * a.table_stride;
  g.out = a.out + (long)b * a.out_stride;
  g.n = a.n;
  g.m = a.m;
  stage1_tile<BF, LOAD, VEC, BNQ>(lds, g, a.pupil, a.inv_wl[b], a.phase[b], (t / tq) * 32,
                                  (t % tq) * BNQ);
}

// ---------------------------------------------------------------------------
// Stage 2: F[(beta, alpha, c)][qy][qx] = sum_py T_beta[qy][py] U[(beta, alpha, c), qx][py],
// then the four mirrored outputs.  A workgroup takes BQ rows qy and 32 columns
// qx of all eight parts; wave (beta, h) holds the four (alpha, c) blocks of BQ / 2
// rows, combines along x in registers, and trades one sign of x with the wave
// of the other beta through LDS, after which wave beta holds both signs of y at
// its sign of x.  With NB stage buffers the loads run NB - 1 stages ahead
// (counted vmcnt waits; one LDS object per buffer, so that the compiler's own
// wait before a fragment read covers that buffer's loads alone).
// ---------------------------------------------------------------------------
template <int N>
using IC = std::integral_constant<int, N>;

// The value the partner wave (wave ^ 2) sent: blocks of 1024 floats.
__device__ __forceinline__ void put_block(uint8_t* x, const f32x16_t& v) {
  float4* d = (float4*)(x + (threadIdx.x >> 6) * 4096) + (threadIdx.x & 63);
#pragma unroll
  for (int q = 0; q < 4; ++q)
    d[64 * q] = make_float4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
}
__device__ __forceinline__ void get_block(const uint8_t* x, f32x16_t& v) {
  const float4* d = (const float4*)(x + ((threadIdx.x >> 6) ^ 2) * 4096) + (threadIdx.x & 63);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float4 t = d[64 * q];
    v[4 * q] = t.x; v[4 * q + 1] = t.y; v[4 * q + 2] = t.z; v[4 * q + 3] = t.w;
  }
}

struct Stage2Prob {
  const uint8_t *table, *mid;
  void* out;
  float* out2;
  const float* G;
  FoldPupil pupil;
  FoldPhase phase;
  double inv_wl;
  float alpha;
  int n, m, inverse;
};

template <bool BF, int EPI, int BQ, int NB>
__device__ __forceinline__ void stage2_tile(const Stage2Prob& a, int qy0, int qx0) {
  constexpr int kA = 2 * BQ * kRow, kBuf = kA + 256 * kRow;
  constexpr int NI = BQ / 64;
  constexpr int kLoads = (2 * BQ + 256) / 64;   // global_load_lds per wave and stage
  constexpr bool SWAP = EPI == FOLD_VJP;        // lanes run along qy, registers along qx
  __shared__ __attribute__((aligned(1024))) uint8_t buf0[kBuf], buf1[kBuf];
  __shared__ __attribute__((aligned(1024))) uint8_t buf2[NB > 2 ? kBuf : 16];
  __shared__ __attribute__((aligned(1024))) uint8_t buf3[NB > 3 ? kBuf : 16];
  auto buf = [&](auto J) __attribute__((always_inline)) -> uint8_t* {
    if constexpr (decltype(J)::value == 0) return buf0;
    else if constexpr (decltype(J)::value == 1) return buf1;
    else if constexpr (decltype(J)::value == 2) return buf2;
    else return buf3;
  };

  const int kh = fold_half(a.n), mh = fold_half(a.m), mhp = fold_pad(mh);
  const long rb = 4L * fold_pad(kh);
  const uint8_t *table = a.table, *mid = a.mid;
  const int nst = (kh + kStageK - 1) / kStageK;
  const int lane = threadIdx.x & 63, lr = lane & 31, lk = lane >> 5;
  const int wave = threadIdx.x >> 6, beta = wave >> 1, h = wave & 1;

  TileRows<2 * BQ> at;
  at.init([&](int r) {
    const int bt = r / BQ, q = qy0 + r % BQ;
    return table + (long)(bt * mhp + (q < mhp ? q : mhp - 1)) * rb;
  });
  TileRows<256> bt;
  bt.init([&](int r) {
    const int q = qx0 + (r & 31);
    return mid + (long)((r >> 5) * mh + (q < mh ? q : mh - 1)) * rb;
  });
  f32x16_t acc[NI][4];
  zero_acc(acc);

  auto issue = [&](auto J, int s) __attribute__((always_inline)) {
    at.issue(buf(J), s);
    bt.issue(buf(J) + kA, s);
  };
  // FULL: every stage the step waits past and issues exists (no branches, so
  // the compiler's counts stay exact across the loop's back edge)
  auto step = [&](auto J, auto FULL, int s) __attribute__((always_inline)) {
    constexpr bool full = decltype(FULL)::value;
    if (full || s + NB - 2 < nst)
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kLoads * (NB - 2)) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const uint8_t* la = buf(J);
    u32x4_t fa[NI][2], fb[4][2];
#pragma unroll
    for (int i = 0; i < NI; ++i) read_frag(fa[i], la, beta * BQ + h * (BQ / 2) + 32 * i);
#pragma unroll
    for (int j = 0; j < 4; ++j) read_frag(fb[j], la + kA, (beta * 4 + j) * 32);
    if (full || s + NB - 1 < nst) issue(IC<(decltype(J)::value + NB - 1) % NB>{}, s + NB - 1);
    __builtin_amdgcn_s_setprio(1);
    if constexpr (!SWAP) {
      mma_stage<BF, NI, 4>(acc, fa, fb);
    } else {
      // the same sums with the operands' roles exchanged
      if constexpr (BF) {
#pragma unroll
        for (int t3 = 0; t3 < 3; ++t3)
#pragma unroll
          for (int i = 0; i < NI; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                  __builtin_bit_cast(bf16x8_t, fb[j][t3 == 1 ? 1 : 0]),
                  __builtin_bit_cast(bf16x8_t, fa[i][t3 == 0 ? 1 : 0]), acc[i][j], 0, 0, 0);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
          for (int i = 0; i < NI; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(
                  __uint_as_float(fb[j][e >> 2][e & 3]), __uint_as_float(fa[i][e >> 2][e & 3]),
                  acc[i][j], 0, 0, 0);
      }
    }
    __builtin_amdgcn_s_setprio(0);
  };
  issue(IC<0>{}, 0);
  if constexpr (NB > 2) { if (nst > 1) issue(IC<1>{}, 1); }
  if constexpr (NB > 3) { if (nst > 2) issue(IC<2>{}, 2); }
  int s = 0;
  for (; s + 2 * NB - 1 <= nst; s += NB) {
    step(IC<0>{}, std::true_type{}, s);
    step(IC<1>{}, std::true_type{}, s + 1);
    if constexpr (NB > 2) step(IC<2>{}, std::true_type{}, s + 2);
    if constexpr (NB > 3) step(IC<3>{}, std::true_type{}, s + 3);
  }
  for (; s < nst; s += NB) {
    step(IC<0>{}, std::false_type{}, s);
    if (s + 1 < nst) step(IC<1>{}, std::false_type{}, s + 1);
    if constexpr (NB > 2) { if (s + 2 < nst) step(IC<2>{}, std::false_type{}, s + 2); }
    if constexpr (NB > 3) { if (s + 3 < nst) step(IC<3>{}, std::false_type{}, s + 3); }
  }

  // ---- the mirrored outputs ----
  const float sg = a.inverse ? -1.f : 1.f;
  const float alpha = a.alpha;
  const float ks = beta ? -sg : sg;
  const int m = a.m, half = m >> 1;
  // this wave's sign of x: + for beta = 0, - for beta = 1
  auto col = [&](int qx) { return beta ? m - 1 - half - qx : half + qx; };
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    // F(., x+-) = F_e -+ i s F_o; beta = 1 carries the factor -i s of the y sine
    f32x16_t kr, ki, sr, si;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float er = acc[i][0][r], ei = acc[i][1][r], orr = acc[i][2][r], oi = acc[i][3][r];
      kr[r] = er + ks * oi; ki[r] = ei - ks * orr;
      sr[r] = er - ks * oi; si[r] = ei + ks * orr;
    }
    if (beta) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float x = kr[r], y = sr[r];
        kr[r] = sg * ki[r]; ki[r] = -sg * x;
        sr[r] = sg * si[r]; si[r] = -sg * y;
      }
    }
    __syncthreads();
    put_block(buf0, sr);
    put_block(buf1, si);
    __syncthreads();
    get_block(buf0, sr);
    get_block(buf1, si);
    // y+: sum; y-: difference (the beta = 0 value first)
    const float d = beta ? -1.f : 1.f;
    const int q0 = qy0 + h * (BQ / 2) + 32 * i;
    if constexpr (EPI == FOLD_INTENSITY || EPI == FOLD_STORE || EPI == FOLD_GRAD) {
      const int qx = qx0 + lr;
      if (qx < mh) {
        const int x = col(qx);
        FoldPhase ph{};
        double tx0 = 0.0;
        bool phased = false;
        if constexpr (EPI == FOLD_STORE) {
          ph = a.phase;
          phased = ph.c2 != 0.0 || ph.cx != 0.0 || ph.cy != 0.0 || ph.c0 != 0.0;
          const double u = (double)x - 0.5 * (m - 1);
          tx0 = fma(ph.c2 * u, u, fma(ph.cx, u, ph.c0));
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int qy = q0 + 8 * (r >> 2) + 4 * lk + (r & 3);
          if (qy < mh) {
            const int yp = half + qy, ym = m - 1 - yp;
            const float pr = alpha * (kr[r] + sr[r]), pi = alpha * (ki[r] + si[r]);
            const float mr = alpha * (d * (kr[r] - sr[r])), mi = alpha * (d * (ki[r] - si[r]));
            const long op = (long)yp * m + x, om = (long)ym * m + x;
            if constexpr (EPI == FOLD_INTENSITY) {
              float* out = (float*)a.out;
              out[op] = pr * pr + pi * pi;
              out[om] = mr * mr + mi * mi;
            } else if constexpr (EPI == FOLD_STORE) {
              float2* out = (float2*)a.out;
              float2 vp = make_float2(pr, pi), vm = make_float2(mr, mi);
              if (phased) {
                const double v = (double)yp - 0.5 * (m - 1), q = fma(ph.c2 * v, v, tx0);
                vp = cmul(vp, turn(fma(ph.cy, v, q)));
                vm = cmul(vm, turn(fma(-ph.cy, v, q)));
              }
              out[op] = vp;
              out[om] = vm;
            } else {
              // the pupil's phasor at both pixels
              const double tX = a.pupil.tx, inv = a.inv_wl;
#pragma unroll
              for (int e = 0; e < 2; ++e) {
                const int y = e ? ym : yp;
                const long o = e ? om : op;
                const float gr = e ? mr : pr, gi = e ? mi : pi;
                const double path =
                    pupil_path(tX, pupil_coord(x, a.pupil.dx, a.pupil.x0),
                               a.pupil.ty * pupil_coord(y, a.pupil.dx, a.pupil.x0),
                               a.pupil.opd ? (double)a.pupil.opd[o] : 0.0);
                const double t0 = a.pupil.phase ? (double)a.pupil.phase[o] * 0.15915494309189535 : 0.0;
                const float2 u = pupil_phasor(path, inv, t0, a.pupil.scale);
                const float am = a.pupil.amp ? a.pupil.amp[o] : 1.0f;
                ((float*)a.out)[o] = am * (u.x * gi - u.y * gr);
                if (a.out2) a.out2[o] = u.x * gr + u.y * gi;
              }
            }
          }
        }
      }
    } else {
      // Ebar = 2 G alpha E at this wave's column sign, folded along y, then
      // (trading the other beta) along x
      const int qy = q0 + lr;
      const int yp = half + (qy < mh ? qy : 0), ym = m - 1 - yp;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int qx = qx0 + 8 * (r >> 2) + 4 * lk + (r & 3);
        const int x = col(qx < mh ? qx : 0);
        const float gp = 2.f * alpha * a.G[(long)yp * m + x], gm = 2.f * alpha * a.G[(long)ym * m + x];
        const float pr = gp * (kr[r] + sr[r]), pi = gp * (ki[r] + si[r]);
        const float mr = gm * (d * (kr[r] - sr[r])), mi = gm * (d * (ki[r] - si[r]));
        // keep the part of this wave's beta, send the other
        kr[r] = pr + d * mr; ki[r] = pi + d * mi;
        sr[r] = pr - d * mr; si[r] = pi - d * mi;
      }
      __syncthreads();
      put_block(buf0, sr);
      put_block(buf1, si);
      __syncthreads();
      get_block(buf0, sr);
      get_block(buf1, si);
      __syncthreads();
      uint8_t* patch = buf0 + wave * kPatch;
      uint8_t* out = (uint8_t*)a.out;
      const long orb = 4L * mhp;
#pragma unroll
      for (int c = 0; c < 4; ++c) {   // (alpha, c)
        f32x16_t v;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float k = (c & 1) ? ki[r] : kr[r], o = (c & 1) ? si[r] : sr[r];
          v[r] = c < 2 ? k + o : d * (k - o);   // x+ minus x-
        }
        const int comp = ((c >> 1) * 2 + beta) * 2 + (c & 1);
        if (q0 < mh)
          store_block<BF>(patch, v, mh - qx0, out + (long)(comp * mh + q0) * orb + 4L * qx0, orb,
                          mh - q0);
      }
    }
  }
}

template <bool BF, int EPI, int BQ, int NB>
__global__ void __launch_bounds__(kThreads, NB * (2 * BQ + 256) * kRow <= 80 * 1024 ? 2 : 1)
fold_stage2_kernel(FoldStage2 a) {
  const int mh = fold_half(a.m), tx = (mh + 31) / 32, ty = (mh + BQ - 1) / BQ;
  const int id = xcd_order(blockIdx.x, tx * ty * a.batch);
  const int b = id / (tx * ty), t = id - b * (tx * ty);
  constexpr int kElem = EPI == FOLD_STORE ? 8 : EPI == FOLD_VJP ? 1 : 4;
  Stage2Prob g;
  g.table = a.table + (long)b * a.table_stride;
  g.mid = a.mid + (long)b * a.mid_stride;
  g.out = (uint8_t*)a.out + (long)b * a.out_stride * kElem;
  g.out2 = a.out2 ? a.out2 + (long)b * a.out_stride : nullptr;
  g.G = a.G;
  g.pupil = a.pupil;
  g.phase = a.phase[b];
  g.inv_wl = a.inv_wl[b];
  g.alpha = a.alpha[b];
  g.n = a.n;
  g.m = a.m;
  g.inverse = a.inverse;
  stage2_tile<BF, EPI, BQ, NB>(g, (t / tx) * BQ, (t % tx) * 32);
}

// ---------------------------------------------------------------------------
// Uneven batches (split-BF16x3): one workgroup per tile of a problem list.
// Hardware workgroup w runs on XCD w % 8 and takes that XCD's tile w / 8, so
// the tiles that share a field, a table or an intermediate meet in one L2.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int group_tile(const FoldGroup& l) {
  const int x = blockIdx.x % kXcds, t = l.xcd[x] + (int)blockIdx.x / kXcds;
  return t < l.xcd[x + 1] ? t : -1;
}

template <bool VEC, int BNQ>
__global__ void __launch_bounds__(kThreads, 2)
fold_group_stage1_kernel(FoldGroup l) {
  __shared__ __attribute__((aligned(1024))) uint8_t lds[2 * (256 + 2 * BNQ) * kRow];
  const int t = group_tile(l);
  if (t < 0) return;
  const FoldProblem& p = l.probs[l.map[t]];
  Stage1Prob g;
  g.src = p.src;
  g.table = p.table;
  g.out = p.mid;
  g.n = p.n;
  g.m = p.m;
  const FoldPhase ph = {0.0, p.cx, p.cy, 0.0};
  const int tq = (fold_half(g.m) + BNQ - 1) / BNQ, local = t - p.tile1;
  stage1_tile<true, FOLD_FIELD, VEC, BNQ>(lds, g, FoldPupil{}, 0.0, ph, (local / tq) * 32,
                                          (local % tq) * BNQ);
}

__global__ void __launch_bounds__(kThreads, 2)
fold_group_stage2_kernel(FoldGroup l) {
  const int t = group_tile(l);
  if (t < 0) return;
  const FoldProblem& p = l.probs[l.map[t]];
  Stage2Prob g{};
  g.table = p.table;
  g.mid = p.mid;
  g.out = p.out;
  g.alpha = p.alpha;
  g.n = p.n;
  g.m = p.m;
  g.inverse = p.inverse;
  const int tx = (fold_half(g.m) + 31) / 32, local = t - p.tile2;
  stage2_tile<true, FOLD_INTENSITY, kFoldTileQy, 3>(g, (local / tx) * kFoldTileQy, (local % tx) * 32);
}

// ---------------------------------------------------------------------------
// Tables and the pupil in memory
// ---------------------------------------------------------------------------

// One table: four consecutive k of a row of both the cosine and the sine per
// thread.  Hardware sin / cos take turns (max abs error 1.3e-7, below the split
// pair's 2^-17); the float32 form takes the library's functions.
template <bool BF>
__device__ __forceinline__ void table_entry(int t, double step, int n, int m,
                                            uint8_t* __restrict__ out) {
  const int kh = fold_half(n), mh = fold_half(m), kp = fold_pad(kh), mhp = fold_pad(mh);
  const int quads = kp >> 2;
  if (t >= mhp * quads) return;
  const int q = t / quads, k0 = (t - q * quads) * 4;
  const double on = (n & 1) ? 0.0 : 0.5, om = (m & 1) ? 0.0 : 0.5;
  const double u = step * ((double)q + om);
  float c[4], s[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int p = k0 + e;
    c[e] = s[e] = 0.f;
    if (p < kh && q < mh) {
      double ph = u * ((double)p + on);
      ph -= rint(ph);
      if constexpr (BF) {
        s[e] = __builtin_amdgcn_sinf((float)ph);
        c[e] = __builtin_amdgcn_cosf((float)ph);
      } else {
        sincospif(2.0f * (float)ph, &s[e], &c[e]);
      }
      if (p == 0 && (n & 1)) c[e] *= 0.5f;   // the centre, folded onto itself
    }
  }
  const long rb = 4L * kp;
  uint8_t* cr = out + (long)q * rb + (k0 >> 4) * kRow;
  put4<BF>(cr, (k0 >> 2) & 3, 0, c);
  put4<BF>(cr + (long)mhp * rb, (k0 >> 2) & 3, 0, s);
}

template <bool BF>
__global__ void __launch_bounds__(256)
fold_table_kernel(FoldSteps st, int n, int m, uint8_t* __restrict__ out, long stride) {
  table_entry<BF>(blockIdx.x * blockDim.x + threadIdx.x, st.step[blockIdx.y], n, m,
                  out + (long)blockIdx.y * stride);
}

__global__ void __launch_bounds__(256)
fold_group_table_kernel(const FoldTableJob* __restrict__ jobs) {
  const FoldTableJob j = jobs[blockIdx.x];
  table_entry<true>(blockIdx.y * blockDim.x + threadIdx.x, j.step, j.n, j.m, j.out);
}

constexpr int kPupilWl = 16;   // wavelengths per thread: the planes are read once for them

template <bool BF, bool VEC>
__global__ void __launch_bounds__(256)
fold_pupil_kernel(FoldPupil pup, FoldSteps wl, int nb, int n,
                  uint8_t* __restrict__ out, long stride) {
  const int kh = fold_half(n);
  const long rb = fold_row_bytes(n);
  const int py = blockIdx.x * 32 + (threadIdx.x >> 3);
  const int beta = threadIdx.x & 1, quad = (threadIdx.x >> 1) & 3, s = blockIdx.y;
  PupilLoad<VEC> pl;
  pl.init(pup, n, py, beta, quad, 0.0);
  pl.raw(s);
  const int b0 = blockIdx.z * kPupilWl, b1 = b0 + kPupilWl < nb ? b0 + kPupilWl : nb;
  for (int b = b0; b < b1; ++b) {
    pl.inv_wl = wl.step[b];
    FoldPart o;
    pl.part(s, beta, o);
    if (py >= kh) continue;
    uint8_t* d = out + (long)b * stride + (long)s * kRow;
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int c = 0; c < 2; ++c)
        put4<BF>(d + (long)(((a * 2 + beta) * 2 + c) * kh + py) * rb, quad, 0, o.v[a][c]);
  }
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

template <bool BF, int LOAD, bool VEC>
hipError_t stage1_width(const FoldStage1& a, hipStream_t s) {
  const int mh = fold_half(a.m), tp = (fold_half(a.n) + 31) / 32;
  auto tiles = [&](int w) { return (long)((mh + w - 1) / w) * tp * a.batch; };
  if (mh > 64 && tiles(128) >= 256) {
    hipLaunchKernelGGL((fold_stage1_kernel<BF, LOAD, VEC, 128>), dim3((unsigned)tiles(128)),
                       dim3(kThreads), 0, s, a);
  } else if (mh > 32 && tiles(64) >= 256) {
    hipLaunchKernelGGL((fold_stage1_kernel<BF, LOAD, VEC, 64>), dim3((unsigned)tiles(64)),
                       dim3(kThreads), 0, s, a);
  } else {
    hipLaunchKernelGGL((fold_stage1_kernel<BF, LOAD, VEC, 32>), dim3((unsigned)tiles(32)),
                       dim3(kThreads), 0, s, a);
  }
  return hipGetLastError();
}

template <bool BF>
hipError_t stage1_load(const FoldStage1& a, FoldLoad load, hipStream_t s) {
  if (load == FOLD_MEM) return stage1_width<BF, FOLD_MEM, true>(a, s);
  if (load == FOLD_PUPIL) {
    const bool vec = a.n % 8 == 0 && aligned16(a.pupil.opd) && aligned16(a.pupil.amp);
    return vec ? stage1_width<BF, FOLD_PUPIL, true>(a, s) : stage1_width<BF, FOLD_PUPIL, false>(a, s);
  }
  const bool vec = a.n % 8 == 0 && aligned16(a.src) && a.src_stride % 16 == 0;
  return vec ? stage1_width<BF, FOLD_FIELD, true>(a, s) : stage1_width<BF, FOLD_FIELD, false>(a, s);
}

template <bool BF, int EPI>
hipError_t stage2_size(const FoldStage2& a, hipStream_t s) {
  const int mh = fold_half(a.m), tx = (mh + 31) / 32;
  auto tiles = [&](int q) { return (long)tx * ((mh + q - 1) / q) * a.batch; };
  hipLaunchKernelGGL((fold_stage2_kernel<BF, EPI, 64, 3>), dim3((unsigned)tiles(64)), dim3(kThreads),
                     0, s, a);
  return hipGetLastError();
}

template <bool BF>
hipError_t stage2_epi(const FoldStage2& a, FoldEpilogue epi, hipStream_t s) {
  switch (epi) {
    case FOLD_INTENSITY: return stage2_size<BF, FOLD_INTENSITY>(a, s);
    case FOLD_STORE: return stage2_size<BF, FOLD_STORE>(a, s);
    case FOLD_VJP: return stage2_size<BF, FOLD_VJP>(a, s);
    default: return stage2_size<BF, FOLD_GRAD>(a, s);
  }
}

}  // namespace

hipError_t launch_fold_tables(const double* step, int nb, int n, int m, bool split, bool adjoint,
                              uint8_t* out, long stride, hipStream_t s) {
  for (int b0 = 0; b0 < nb; b0 += FoldSteps::kMax) {
    const int k = nb - b0 < FoldSteps::kMax ? nb - b0 : FoldSteps::kMax;
    FoldSteps st;
    for (int i = 0; i < k; ++i) st.step[i] = step[b0 + i];
    for (int adj = 0; adj < (adjoint ? 2 : 1); ++adj) {
      const int kn = adj ? m : n, km = adj ? n : m;
      uint8_t* o = out + (long)b0 * stride + (adj ? fold_table_bytes(n, m) : 0);
      const int work = fold_pad(fold_half(km)) * (fold_pad(fold_half(kn)) / 4);
      const dim3 grid((unsigned)((work + 255) / 256), k);
      if (split)
        hipLaunchKernelGGL(fold_table_kernel<true>, grid, dim3(256), 0, s, st, kn, km, o, stride);
      else
        hipLaunchKernelGGL(fold_table_kernel<false>, grid, dim3(256), 0, s, st, kn, km, o, stride);
      const hipError_t e = hipGetLastError();
      if (e != hipSuccess) return e;
    }
  }
  return hipSuccess;
}

hipError_t launch_fold_stage1(const FoldStage1& a, FoldLoad load, bool split, hipStream_t s) {
  if (a.batch <= 0) return hipSuccess;
  if (a.batch > FoldStage1::kMaxBatch) return hipErrorInvalidValue;
  return split ? stage1_load<true>(a, load, s) : stage1_load<false>(a, load, s);
}

hipError_t launch_fold_stage2(const FoldStage2& a, FoldEpilogue epi, bool split, hipStream_t s) {
  if (a.batch <= 0) return hipSuccess;
  if (a.batch > FoldStage2::kMaxBatch) return hipErrorInvalidValue;
  return split ? stage2_epi<true>(a, epi, s) : stage2_epi<false>(a, epi, s);
}

hipError_t launch_fold_pupil(const FoldPupil& p, const double* inv_wl, int nb, int n, bool split,
                             uint8_t* out, long stride, hipStream_t s) {
  const bool vec = n % 8 == 0 && aligned16(p.opd) && aligned16(p.amp);
  for (int b0 = 0; b0 < nb; b0 += FoldSteps::kMax) {
    const int k = nb - b0 < FoldSteps::kMax ? nb - b0 : FoldSteps::kMax;
    FoldSteps wl;
    for (int i = 0; i < k; ++i) wl.step[i] = inv_wl[b0 + i];
    const dim3 grid((fold_half(n) + 31) / 32, fold_pad(fold_half(n)) / kStageK,
                    (k + kPupilWl - 1) / kPupilWl);
    uint8_t* o = out + (long)b0 * stride;
    if (split && vec) hipLaunchKernelGGL((fold_pupil_kernel<true, true>), grid, dim3(256), 0, s, p, wl, k, n, o, stride);
    else if (split) hipLaunchKernelGGL((fold_pupil_kernel<true, false>), grid, dim3(256), 0, s, p, wl, k, n, o, stride);
    else if (vec) hipLaunchKernelGGL((fold_pupil_kernel<false, true>), grid, dim3(256), 0, s, p, wl, k, n, o, stride);
    else hipLaunchKernelGGL((fold_pupil_kernel<false, false>), grid, dim3(256), 0, s, p, wl, k, n, o, stride);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

int fold_group_width(int m) {
  const int mh = fold_half(m);
  return mh > 64 ? 128 : mh > 32 ? 64 : 32;
}

hipError_t launch_fold_group_tables(const FoldTableJob* jobs, int njobs, long most, hipStream_t s) {
  hipLaunchKernelGGL(fold_group_table_kernel, dim3(njobs, (unsigned)((most + 255) / 256)), dim3(256),
                     0, s, jobs);
  return hipGetLastError();
}

static unsigned group_grid(const FoldGroup& g) {
  int most = 0;
  for (int x = 0; x < kXcds; ++x) most = std::max(most, g.xcd[x + 1] - g.xcd[x]);
  return (unsigned)(kXcds * most);
}

hipError_t launch_fold_group_stage1(const FoldGroup& g, int width, bool vec, hipStream_t s) {
  const dim3 grid(group_grid(g)), block(kThreads);
  if (grid.x == 0) return hipSuccess;
  auto go = [&](auto V) {
    constexpr bool v = decltype(V)::value;
    if (width == 128) hipLaunchKernelGGL((fold_group_stage1_kernel<v, 128>), grid, block, 0, s, g);
    else if (width == 64) hipLaunchKernelGGL((fold_group_stage1_kernel<v, 64>), grid, block, 0, s, g);
    else hipLaunchKernelGGL((fold_group_stage1_kernel<v, 32>), grid, block, 0, s, g);
  };
  if (vec) go(std::true_type{});
  else go(std::false_type{});
  return hipGetLastError();
}

hipError_t launch_fold_group_stage2(const FoldGroup& g, hipStream_t s) {
  const dim3 grid(group_grid(g));
  if (grid.x == 0) return hipSuccess;
  hipLaunchKernelGGL(fold_group_stage2_kernel, grid, dim3(kThreads), 0, s, g);
  return hipGetLastError();
}

bool fold_pupil_in_loader(int m) { return fold_half(m) <= 256; }

}  // namespace dlx
