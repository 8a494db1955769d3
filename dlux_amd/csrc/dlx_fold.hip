// The folded MFT's kernels (dlx_fold.h): cosine / sine tables, the pupil and
// field loaders, and the two contractions with their epilogues, in complex64
// (v_mfma_f32_32x32x2_f32) and split-BF16x3 form (v_mfma_f32_32x32x16_bf16,
// lo*lo + lo*hi + hi*lo + hi*hi), on one tile geometry: both forms hold 4 bytes per
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

// Global accesses through pointers that may come from descriptors in memory,
// whose address space the compiler does not see: as flat accesses they would
// count with the LDS ones, and every wait for LDS would wait for memory (48
// sources of 256^2 to 1024^2, with the branch-free steps: 728 -> 675 us).
__device__ __forceinline__ u32x4_t load_global(const void* p) {
  return *(const __attribute__((address_space(1))) u32x4_t*)p;
}
__device__ __forceinline__ void store_global(void* p, u32x4_t v) {
  *(__attribute__((address_space(1))) u32x4_t*)p = v;
}

template <int N>
using IC = std::integral_constant<int, N>;

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
// `odd`: the rows are parts of beta = 1 as a loader writes them (part_row).
__device__ __forceinline__ void read_frag(u32x4_t (&f)[2], const uint8_t* tile, int row0,
                                          int odd = 0) {
  const int lane = threadIdx.x & 63, lr = lane & 31, lk = lane >> 5;
  const uint8_t* r = tile + (row0 + (lr ^ (2 * odd))) * kRow;
#pragma unroll
  for (int j = 0; j < 2; ++j)
    f[j] = *(const u32x4_t*)(r + (((2 * lk + j) ^ ((lr >> 2) & 3) ^ odd) << 4));
}

// A table's pieces in the order MFMAs take them: per 32 rows and stage, 2 KiB
// = two runs of 64 lanes x 16 bytes.  No two waves of a workgroup need the same
// rows, so the fragments go straight from memory to registers, a kilobyte per
// load.
__device__ __forceinline__ long table_block(int part, int rows_pad, int kp, int row_blk) {
  return ((long)part * (rows_pad >> 5) + row_blk) * (kp >> 4) * 2048;
}
__device__ __forceinline__ void load_frag(u32x4_t (&f)[2], const uint8_t* blk, int s) {
  const uint8_t* p = blk + (long)s * 2048 + (threadIdx.x & 63) * 16;
  f[0] = load_global(p);
  f[1] = load_global(p + 1024);
}

// acc[i][j] += sum over the stage's 16 k of a_i(m) b_j(n): lane holds column
// n = lane % 32, register r row m = 8 (r / 4) + 4 (lane / 32) + r % 4.
template <bool BF, int NI, int NJ>
__device__ __forceinline__ void mma_stage(f32x16_t (&acc)[NI][NJ], const u32x4_t (&a)[NI][2],
                                          const u32x4_t (&b)[NJ][2]) {
  if constexpr (BF) {
    // lo*lo, lo*hi, hi*lo, hi*hi: the small terms first
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              __builtin_bit_cast(bf16x8_t, a[i][t < 2 ? 1 : 0]),
              __builtin_bit_cast(bf16x8_t, b[j][t & 1 ? 0 : 1]), acc[i][j], 0, 0, 0);
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

// Where a loader puts row py of a part: the lanes of beta = 1 write beside those
// of beta = 0, whose banks they would otherwise share.
__device__ __forceinline__ int part_row(int py, int beta) { return py ^ (2 * beta); }
__device__ __forceinline__ int part_slot(int py, int beta) { return ((py >> 2) & 3) ^ beta; }

__device__ __forceinline__ float2 cmul(float2 a, float2 w) {
  return make_float2(a.x * w.x - a.y * w.y, a.x * w.y + a.y * w.x);
}
// exp(2 pi i t), t in turns (any size): max abs error 1.3e-7.
__device__ __forceinline__ float2 turn(double t) {
  t -= rint(t);
  return make_float2(__builtin_amdgcn_cosf((float)t), __builtin_amdgcn_sinf((float)t));
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

// x and y folds; vp / vm: the values at k+ and k- of the thread's own row, times
// -1 in the lanes of row y- (beta = 1): then own + other's * (beta ? 1 : -1) is
// the even part in one lane and the odd part in the other, one instruction a
// value (a swap, a copy and a multiply-add before: 64 of 423 vector
// instructions of two split stages).
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
  const float sg = beta ? 1.f : -1.f;
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    float(&x)[4] = o.v[a][0], (&y)[4] = o.v[a][1];
    // x = x of lane ^ 1 * sg + x; a DPP operand is read two states after its write
#define DLX_FOLD(i) "v_fmac_f32_dpp %" #i ", %" #i ", %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
    asm("s_nop 1\n\t" DLX_FOLD(0) DLX_FOLD(1) DLX_FOLD(2) DLX_FOLD(3) DLX_FOLD(4) DLX_FOLD(5)
            DLX_FOLD(6) DLX_FOLD(7)
        : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3]), "+v"(y[0]), "+v"(y[1]), "+v"(y[2]),
          "+v"(y[3])
        : "v"(sg));
#undef DLX_FOLD
  }
}

// The pupil loader of one thread.  VEC: n a multiple of 8 and 16-byte aligned
// planes (float4 loads; a run of four is whole or absent).  ANY: any of the
// planes may be missing, there may be a phase plane and a tilt, tested as they
// are read; otherwise the amplitude or the OPD is there, no phase is, a tilt
// is if TILT, and every load is unconditional (a missing plane reads the other
// one, and its constant comes in through the coefficients), so that the loads
// stay in flight over a stage and the phasors can be scheduled among products.
template <bool VEC, bool TILT, bool ANY>
struct PupilLoad {
  const float *opd, *amp, *phase;   // rows
  int n, kh, quad, x0i;             // x0i = n / 2: the first positive column
  bool has_opd, has_amp, has_phase;
  double inv_wl, tx, tyY, dx, x0, co;   // co: 1 if there is an OPD, else 0
  float ca, cb;                     // amplitude = ca * value + cb, signed; zero outside the rows
  struct Runs { float4 op, om, ap, am; };   // plus runs (k ascending), minus runs (descending)
  struct AnyRuns : Runs { float4 pp, pm; };
  using Raw = std::conditional_t<ANY, AnyRuns, Runs>;

  __device__ __forceinline__ void init(const FoldPupil& p, int n_, int py, int beta, int quad_,
                                       double inv) {
    n = n_; kh = (n + 1) >> 1; quad = quad_; x0i = n >> 1;
    const bool row_ok = py < kh;
    const int yp = x0i + (row_ok ? py : 0);
    const int y = beta ? n - 1 - yp : yp;
    has_opd = p.opd != nullptr; has_amp = p.amp != nullptr; has_phase = p.phase != nullptr;
    opd = (has_opd ? p.opd : p.amp) + (long)y * n;
    amp = (has_amp ? p.amp : p.opd) + (long)y * n;
    if constexpr (ANY) phase = p.phase + (long)y * n;
    co = has_opd ? 1.0 : 0.0;
    inv_wl = TILT || ANY ? inv : has_opd ? inv : 0.0;
    tx = p.tx; dx = p.dx; x0 = p.x0;
    tyY = p.ty * pupil_coord(y, p.dx, p.x0);
    const float sc = !row_ok ? 0.f : beta ? -p.scale : p.scale;   // the y fold's sign
    ca = has_amp ? sc : 0.f;
    cb = has_amp ? 0.f : sc;
  }
  __device__ __forceinline__ float4 run_up(const float* row, int p) const {
    if constexpr (VEC) return *(const float4*)(row + x0i + (p < kh ? p : 0));
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = row[x0i + (p + e < kh ? p + e : kh - 1)];
    return make_float4(v[0], v[1], v[2], v[3]);
  }
  __device__ __forceinline__ float4 run_down(const float* row, int p) const {
    if constexpr (VEC) return *(const float4*)(row + x0i - 4 - (p < kh ? p : 0));
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = row[n - 1 - x0i - (p + e < kh ? p + e : kh - 1)];
    return make_float4(v[3], v[2], v[1], v[0]);
  }
  __device__ __forceinline__ void raw(int s, Raw& r) const {
    const int p = s * kStageK + quad * 4;
    if (!ANY || has_opd) { r.op = run_up(opd, p); r.om = run_down(opd, p); }
    if (!ANY || has_amp) { r.ap = run_up(amp, p); r.am = run_down(amp, p); }
    if constexpr (ANY)
      if (has_phase) { r.pp = run_up(phase, p); r.pm = run_down(phase, p); }
  }
  __device__ __forceinline__ void part(int s, int beta, const Raw& r, FoldPart& o) const {
    const int p = s * kStageK + quad * 4;
    const float vo[2][4] = {{r.op.x, r.op.y, r.op.z, r.op.w}, {r.om.w, r.om.z, r.om.y, r.om.x}};
    const float va[2][4] = {{r.ap.x, r.ap.y, r.ap.z, r.ap.w}, {r.am.w, r.am.z, r.am.y, r.am.x}};
    float vt[2][4];
    if constexpr (ANY) {
      const float x[2][4] = {{r.pp.x, r.pp.y, r.pp.z, r.pp.w}, {r.pm.w, r.pm.z, r.pm.y, r.pm.x}};
#pragma unroll
      for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int e = 0; e < 4; ++e) vt[d][e] = x[d][e];
    }
    float2 v[2][4];
    // VEC: the run is whole or absent
    const float ra = !VEC || p < kh ? ca : 0.f, rb = !VEC || p < kh ? cb : 0.f;
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float a = __builtin_fmaf(va[d][e], ra, rb);
        if constexpr (!VEC) a = p + e < kh ? a : 0.f;
        double t = 0.0, path = (double)vo[d][e];
        if constexpr (TILT || ANY) {
          const int pc = p + e < kh ? p + e : kh - 1;
          const int x = d ? n - 1 - x0i - pc : x0i + pc;
          if (ANY && !has_opd) path = 0.0;
          if constexpr (ANY)
            if (has_phase) t = (double)vt[d][e] * 0.15915494309189535;   // 1 / (2 pi)
          if (ANY && !has_amp) a = p + e < kh ? rb : 0.f;
          path = fma(path, co, fma(tx, pupil_coord(x, dx, x0), tyY));   // pupil_path's bits
        }
        v[d][e] = pupil_phasor(path, inv_wl, t, a);
      }
    fold_x(v[0], v[1], o);
    fold_y(o, beta);
  }
};

// The complex64 field loader of one thread.  VEC as above.  A phase's x factor
// multiplies the loaded values (w: its values at k+ and k- of the four k, from
// the stage's window in LDS); the y factor is applied to the stage's results.
template <bool VEC>
struct FieldLoad {
  const float2* row;
  int n, kh, quad, x0i;
  bool row_ok;
  struct Raw { float4 fp[2], fm[2]; };   // plus run (k ascending), minus run in memory order

  __device__ __forceinline__ void init(const uint8_t* src, int n_, int py, int beta, int quad_) {
    n = n_; kh = (n + 1) >> 1; quad = quad_; x0i = n >> 1;
    row_ok = py < kh;
    const int yp = x0i + (row_ok ? py : 0);
    row = (const float2*)src + (long)(beta ? n - 1 - yp : yp) * n;
  }
  __device__ __forceinline__ void raw(int s, Raw& r) const {
    int p = s * kStageK + quad * 4;
    if constexpr (VEC) {
      p = p < kh ? p : 0;
      const float2 *a = row + x0i + p, *b = row + x0i - 4 - p;
      r.fp[0] = *(const float4*)a; r.fp[1] = *(const float4*)(a + 2);
      r.fm[0] = *(const float4*)b; r.fm[1] = *(const float4*)(b + 2);
    } else {
      float2 a[4], b[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int pc = p + e < kh ? p + e : kh - 1;
        a[e] = row[x0i + pc];
        b[3 - e] = row[n - 1 - x0i - pc];
      }
      r.fp[0] = make_float4(a[0].x, a[0].y, a[1].x, a[1].y);
      r.fp[1] = make_float4(a[2].x, a[2].y, a[3].x, a[3].y);
      r.fm[0] = make_float4(b[0].x, b[0].y, b[1].x, b[1].y);
      r.fm[1] = make_float4(b[2].x, b[2].y, b[3].x, b[3].y);
    }
  }
  // w: [k][k+, k-] of the stage's phase
  __device__ __forceinline__ void part(int s, int beta, const Raw& r, bool phased, const float4* w,
                                       FoldPart& out) const {
    const float4 *fp = r.fp, *fm = r.fm;
    const int p = s * kStageK + quad * 4;
    float2 vp[4] = {{fp[0].x, fp[0].y}, {fp[0].z, fp[0].w}, {fp[1].x, fp[1].y}, {fp[1].z, fp[1].w}};
    float2 vm[4] = {{fm[1].z, fm[1].w}, {fm[1].x, fm[1].y}, {fm[0].z, fm[0].w}, {fm[0].x, fm[0].y}};
    if (phased) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float4 t = w[quad * 4 + e];
        vp[e] = cmul(vp[e], make_float2(t.x, t.y));
        vm[e] = cmul(vm[e], make_float2(t.z, t.w));
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (!(row_ok && p + e < kh)) vp[e] = vm[e] = make_float2(0.f, 0.f);
      if (beta) {   // the y fold's sign
        vp[e] = make_float2(-vp[e].x, -vp[e].y);
        vm[e] = make_float2(-vm[e].x, -vm[e].y);
      }
    }
    fold_x(vp, vm, out);
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
    const u32x4_t v = *(const u32x4_t*)(patch + r * kPatchRow + piece * 16);
    if (r < rows) store_global(out + (long)r * row_bytes + piece * 16, v);
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// LDS hand-over between the waves of a workgroup: waits for this wave's LDS
// accesses only; global loads stay in flight.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Trading 32 x 32 blocks between waves through LDS: each wave writes its
// 1024 floats, and after a barrier reads those of wave ^ XOR.
__device__ __forceinline__ void put_block(uint8_t* x, const f32x16_t& v) {
  float4* d = (float4*)(x + (threadIdx.x >> 6) * 4096) + (threadIdx.x & 63);
#pragma unroll
  for (int q = 0; q < 4; ++q)
    d[64 * q] = make_float4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
}
template <int XOR>
__device__ __forceinline__ void get_block(const uint8_t* x, f32x16_t& v) {
  const float4* d = (const float4*)(x + ((threadIdx.x >> 6) ^ XOR) * 4096) + (threadIdx.x & 63);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float4 t = d[64 * q];
    v[4 * q] = t.x; v[4 * q + 1] = t.y; v[4 * q + 2] = t.z; v[4 * q + 3] = t.w;
  }
}

// ---------------------------------------------------------------------------
// Stage 1: U[(beta, alpha, c), qx][py] = sum_px T_alpha[qx][px] P[(alpha, beta, c), py][px].
// A workgroup takes 32 rows py of all eight (alpha, beta, c) parts -- the four
// mirrored pixels of a loaded quad feed both alphas -- and BNQ outputs qx: at
// 128 the field is formed once per 128-column tile (256 outputs), each wave
// holds eight 32 x 32 blocks (eight fragment reads from LDS per 32 MFMAs of a
// split stage), and two workgroups share a CU.  Launches with fewer tiles take
// 64 or 32 columns.  Issue bounds the loop: 32 MFMAs and 180 vector instructions
// (phasors, folds, split) per wave and split stage.  64 wavelengths of 512^2 ->
// 256^2: 40-43 us split, 82-90 float32, where the complex contractions took 101 and 332.
// ---------------------------------------------------------------------------
struct Stage1Prob {
  const uint8_t* src;
  const uint8_t* table;
  uint8_t* out;
  int n, m;
};

template <int BNQ>
struct S1 {
  static constexpr int NI = BNQ >= 64 ? 4 : 2, NJ = BNQ >= 64 ? BNQ / 64 : 1;
  // first A row (in (alpha, beta, c, py) order) and first column of a wave
  __device__ static __forceinline__ int arow(int wave) {
    return (wave >> 1) * 128 + (BNQ >= 64 ? 0 : (wave & 1) * 64);
  }
  __device__ static __forceinline__ int beta(int wave, int i) {
    return BNQ >= 64 ? i >> 1 : wave & 1;
  }
  __device__ static __forceinline__ int col(int wave) {
    return BNQ >= 64 ? (wave & 1) * (BNQ / 2) : 0;
  }
};

// The wave's blocks to the stage-1 result.
template <bool BF, int BNQ>
__device__ __forceinline__ void stage1_store(uint8_t* patch, f32x16_t (&acc)[S1<BNQ>::NI][S1<BNQ>::NJ],
                                             int n, int m, uint8_t* out, int py0, int q0) {
  const int kh = (n + 1) >> 1, mh = (m + 1) >> 1, wave = threadIdx.x >> 6;
  const long rb = 4L * fold_pad(kh);
#pragma unroll
  for (int i = 0; i < S1<BNQ>::NI; ++i)
#pragma unroll
    for (int j = 0; j < S1<BNQ>::NJ; ++j) {
      const int bc = BNQ >= 64 ? i : (wave & 1) * 2 + i;   // (beta, c)
      const int comp = ((bc >> 1) * 2 + (wave >> 1)) * 2 + (bc & 1);
      const int q = q0 + S1<BNQ>::col(wave) + 32 * j;
      if (q < mh)
        store_block<BF>(patch, acc[i][j], kh - py0, out + (long)(comp * mh + q) * rb + 4L * py0, rb,
                        mh - q);
    }
}

// The y factor of a field's phase, applied to the wave's blocks: with
// exp(i f) at row y+ (its linear part conjugate at y-), the even and odd parts
// mix as e' = e cos f + i o sin f, o' = o cos f + i e sin f.  `lds`: 32 KiB
// free of readers (32-column tiles, whose waves hold one beta each, trade).
template <int BNQ>
__device__ __forceinline__ void y_phase(uint8_t* lds, f32x16_t (&acc)[S1<BNQ>::NI][S1<BNQ>::NJ],
                                        double c2, double cy, int n, int py0) {
  const int lk = (threadIdx.x >> 5) & 1;
  const double on = (n & 1) ? 0.0 : 0.5;
  f32x16_t other[2];
  if constexpr (BNQ == 32) {
    put_block(lds, acc[0][0]);
    put_block(lds + 16384, acc[1][0]);
    lds_barrier();
    get_block<1>(lds, other[0]);
    get_block<1>(lds + 16384, other[1]);
    lds_barrier();
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const double u = (double)(py0 + 8 * (r >> 2) + 4 * lk + (r & 3)) + on;
    float2 w = turn(cy * u), q = make_float2(1.f, 0.f);
    if (c2 != 0.0) q = turn(c2 * u * u);
    if constexpr (BNQ == 32) {
      const float2 v = cmul(make_float2(acc[0][0][r] * w.x - other[1][r] * w.y,
                                        acc[1][0][r] * w.x + other[0][r] * w.y), q);
      acc[0][0][r] = v.x;
      acc[1][0][r] = v.y;
    } else {
#pragma unroll
      for (int j = 0; j < S1<BNQ>::NJ; ++j) {
        const float er = acc[0][j][r], ei = acc[1][j][r], od = acc[2][j][r], oi = acc[3][j][r];
        const float2 e = cmul(make_float2(er * w.x - oi * w.y, ei * w.x + od * w.y), q);
        const float2 o = cmul(make_float2(od * w.x - ei * w.y, oi * w.x + er * w.y), q);
        acc[0][j][r] = e.x; acc[1][j][r] = e.y; acc[2][j][r] = o.x; acc[3][j][r] = o.y;
      }
    }
  }
}

constexpr int kPupilAny = 3;    // FOLD_PUPIL through the loader that tests for every plane
constexpr int kPupilTilt = 4;   // FOLD_PUPIL with a tilt

// Fields formed by the loader: the next stage's parts are formed after this
// stage's products are issued, from values loaded two stages ahead.
template <bool BF, int LOAD, bool VEC, int BNQ>
__global__ void __launch_bounds__(kThreads, 2)
fold_stage1_kernel(FoldStage1 a) {
  using S = S1<BNQ>;
  constexpr int NI = S::NI, NJ = S::NJ, kBuf = 256 * kRow;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[2 * kBuf];
  __shared__ float4 win[2][kStageK];   // the x phase of a stage's k, at k+ and k-
  const int kh = fold_half(a.n), mh = fold_half(a.m), mhp = fold_pad(mh), kp = fold_pad(kh);
  const int tq = (mh + BNQ - 1) / BNQ, tp = (kh + 31) / 32;
  const int id = xcd_order(blockIdx.x, tq * tp * a.batch);
  const int b = id / (tq * tp), t = id - b * (tq * tp);
  const int py0 = (t / tq) * 32, q0 = (t % tq) * BNQ;
  const int nst = (kh + kStageK - 1) / kStageK;
  const int wave = threadIdx.x >> 6;

  f32x16_t acc[NI][NJ];
  zero_acc(acc);
  const uint8_t* tab[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int blk = (q0 + S::col(wave)) / 32 + j, last = (mhp >> 5) - 1;
    tab[j] = a.table + (long)b * a.table_stride +
             table_block(wave >> 1, mhp, kp, blk < last ? blk : last);
  }
  const int py = threadIdx.x >> 3, beta = threadIdx.x & 1, quad = (threadIdx.x >> 1) & 3;
  std::conditional_t<LOAD == FOLD_FIELD, FieldLoad<VEC>, PupilLoad<VEC, LOAD == kPupilTilt, LOAD == kPupilAny>> ld;
  FoldPhase ph{};
  bool phased = false;
  if constexpr (LOAD != FOLD_FIELD) {
    ld.init(a.pupil, a.n, py0 + py, beta, quad, a.inv_wl[b]);
  } else {
    ld.init(a.src + (long)b * a.src_stride, a.n, py0 + py, beta, quad);
    ph = a.phase[b];
    phased = ph.c2 != 0.0 || ph.cx != 0.0 || ph.cy != 0.0;
  }
  typename decltype(ld)::Raw raw[2];
  const double on = (a.n & 1) ? 0.0 : 0.5;
  auto window = [&](int s) {   // formed two stages ahead of its use's products
    if constexpr (LOAD == FOLD_FIELD) {
      if (threadIdx.x < kStageK) {
        const double u = (double)(s * kStageK + (int)threadIdx.x) + on, q = ph.c2 * u * u;
        const float2 wp = turn(fma(ph.cx, u, q)), wm = turn(fma(-ph.cx, u, q));
        win[s & 1][threadIdx.x] = make_float4(wp.x, wp.y, wm.x, wm.y);
      }
    }
  };
  // whether a field has a phase is asked outside the loop; by the split form's
  // 128-column tiles inside it, as a second loop spills (64 fields 512^2 -> 256^2,
  // shifted: 73.4 us against 71.1; float32 without a shift 126.7 against 138.0)
  constexpr bool kAsk = LOAD == FOLD_FIELD && BF && BNQ == 128;
  auto convert = [&](auto PH, int s, const typename decltype(ld)::Raw& r) __attribute__((always_inline)) {
    FoldPart o;
    if constexpr (LOAD != FOLD_FIELD) ld.part(s, beta, r, o);
    else ld.part(s, beta, r, kAsk ? phased : decltype(PH)::value, win[s & 1], o);
    uint8_t* buf = lds + (s & 1) * kBuf;
    const int pr = part_row(py, beta), fl = part_slot(py, beta);
#pragma unroll
    for (int al = 0; al < 2; ++al)
#pragma unroll
      for (int c = 0; c < 2; ++c)
        put4<BF>(buf + (((al * 2 + beta) * 2 + c) * 32 + pr) * kRow, quad, fl, o.v[al][c]);
  };
  u32x4_t fb[2][NJ][2];
  auto load_tab = [&](auto J, int s) __attribute__((always_inline)) {
    const int sc = s < nst ? s : nst - 1;
#pragma unroll
    for (int j = 0; j < NJ; ++j) load_frag(fb[decltype(J)::value][j], tab[j], sc);
  };
  // one stage: J = s & 1; FULL: there is a next one; PH: the field has a phase
  auto step = [&](auto J, auto FULL, auto PH, int s) __attribute__((always_inline)) {
    constexpr int j0 = decltype(J)::value;
    lds_barrier();   // stage s is in LDS, stage s - 1 has been read
    const uint8_t* la = lds + j0 * kBuf;
    u32x4_t fa[NI][2];
#pragma unroll
    for (int i = 0; i < NI; ++i)
      read_frag(fa[i], la, S::arow(wave) + 32 * i, S::beta(wave, i));
    load_tab(IC<1 - j0>{}, s + 1);
    ld.raw(s + 2, raw[j0]);
    if constexpr (decltype(PH)::value) window(s + 2);
    // one wave per SIMD (small launches) keeps its products ahead of its
    // conversion: 17.0 against 19.5 us at 16 wavelengths of 512^2 -> 128^2; with
    // two, the raised priority cost 90 -> 100 us (float32, 64 of 512^2 -> 256^2)
    if constexpr (BNQ < 128) __builtin_amdgcn_s_setprio(1);
    mma_stage<BF, NI, NJ>(acc, fa, fb[j0]);
    if constexpr (BNQ < 128) __builtin_amdgcn_s_setprio(0);
    if (decltype(FULL)::value || s + 1 < nst) convert(PH, s + 1, raw[1 - j0]);
  };
  auto run = [&](auto PH) __attribute__((always_inline)) {
    load_tab(IC<0>{}, 0);
    ld.raw(0, raw[0]);
    ld.raw(1, raw[1]);
    if constexpr (decltype(PH)::value) {
      window(0);
      window(1);
      lds_barrier();
    }
    convert(PH, 0, raw[0]);
    // whole pairs: no path of the loop skips a load or a part (16 fields 512^2 ->
    // 256^2, float32: 48.0 -> 46.4 us).  At 128 columns only the aligned loader
    // without a tilt has the registers: elsewhere the parts stay in a block of their
    // own (48 pupils of 511^2 -> 257^2, split: 42 spilled registers and 121 us
    // merged, 4 and 97 apart; 512^2 tilted 64.5 and 61.9)
    using Whole = std::bool_constant<(LOAD == FOLD_PUPIL && VEC) || BNQ < 128>;
    int s = 0;
    for (; s + 2 < nst; s += 2) {
      step(IC<0>{}, Whole{}, PH, s);
      step(IC<1>{}, Whole{}, PH, s + 1);
    }
    step(IC<0>{}, std::false_type{}, PH, s);
    if (s + 1 < nst) step(IC<1>{}, std::false_type{}, PH, s + 1);
  };
  if (kAsk || (LOAD == FOLD_FIELD && phased)) run(std::bool_constant<LOAD == FOLD_FIELD>{});
  else if constexpr (!kAsk) run(std::false_type{});
  lds_barrier();
  if constexpr (LOAD == FOLD_FIELD)
    if (phased) y_phase<BNQ>(lds, acc, ph.c2, ph.cy, a.n, py0);
  stage1_store<BF, BNQ>(lds + wave * kPatch, acc, a.n, a.m, a.out + (long)b * a.out_stride, py0, q0);
}

// Launches with few tiles (fold_stage1_kernel at 32 columns leaves compute units
// idle): 16 rows py and 32 columns a workgroup, stages of 32 k in two runs of 16.
// A tile row block is one (alpha, beta) with its real rows 0-15 and imaginary
// rows 16-31; wave (alpha, beta) accumulates it.  Twice the workgroups, half the
// products of a wave and half the stages to step through: a chain of load,
// form, product bounds such launches.  28.6 -> 20.1 us at 2 wavelengths of
// 1024^2 -> 256^2 (split), 39.1 -> 24.1 at one of 1024^2 -> 512^2 (float32),
// 20.2 -> 13.9 at 7 of 333^2 -> 111^2 (split, tilted).
template <bool BF, int LOAD, bool VEC>
__global__ void __launch_bounds__(kThreads, 2)
fold_stage1_small_kernel(FoldStage1 a) {
  constexpr int kRun = 128 * kRow;   // one run of 16 k: 128 tile rows
  __shared__ __attribute__((aligned(1024))) uint8_t lds[4 * kRun];
  __shared__ float4 win[2][2 * kStageK];   // the x phase of a stage's k, at k+ and k-
  const int kh = fold_half(a.n), mh = fold_half(a.m), mhp = fold_pad(mh), kp = fold_pad(kh);
  const int tq = (mh + 31) / 32, tp = (kh + 15) / 16;
  const int id = xcd_order(blockIdx.x, tq * tp * a.batch);
  const int b = id / (tq * tp), t = id - b * (tq * tp);
  const int py0 = (t / tq) * 16, q0 = (t % tq) * 32;
  const int nst = kp / (2 * kStageK);
  const int wave = threadIdx.x >> 6;
  const uint8_t* tab = a.table + (long)b * a.table_stride + table_block(wave >> 1, mhp, kp, q0 / 32);
  const int py = threadIdx.x >> 4, beta = threadIdx.x & 1, quad = (threadIdx.x >> 1) & 3;
  const int run = (threadIdx.x >> 3) & 1;
  std::conditional_t<LOAD == FOLD_FIELD, FieldLoad<VEC>, PupilLoad<VEC, LOAD == kPupilTilt, LOAD == kPupilAny>> ld;
  FoldPhase ph{};
  bool phased = false;
  if constexpr (LOAD != FOLD_FIELD) {
    ld.init(a.pupil, a.n, py0 + py, beta, quad, a.inv_wl[b]);
  } else {
    ld.init(a.src + (long)b * a.src_stride, a.n, py0 + py, beta, quad);
    ph = a.phase[b];
    phased = ph.c2 != 0.0 || ph.cx != 0.0 || ph.cy != 0.0;
  }
  typename decltype(ld)::Raw raw[2];
  const double on = (a.n & 1) ? 0.0 : 0.5;
  auto window = [&](int s) {
    if constexpr (LOAD == FOLD_FIELD) {
      if (threadIdx.x < 2 * kStageK) {
        const double u = (double)(s * 2 * kStageK + (int)threadIdx.x) + on, q = ph.c2 * u * u;
        const float2 wp = turn(fma(ph.cx, u, q)), wm = turn(fma(-ph.cx, u, q));
        win[s & 1][threadIdx.x] = make_float4(wp.x, wp.y, wm.x, wm.y);
      }
    }
  };
  auto convert = [&](auto PH, int s, const typename decltype(ld)::Raw& r) __attribute__((always_inline)) {
    FoldPart o;
    if constexpr (LOAD != FOLD_FIELD) ld.part(2 * s + run, beta, r, o);
    else ld.part(2 * s + run, beta, r, decltype(PH)::value, win[s & 1] + run * kStageK, o);
    uint8_t* buf = lds + ((s & 1) * 2 + run) * kRun;
    const int pr = part_row(py, beta), fl = part_slot(py, beta);
#pragma unroll
    for (int al = 0; al < 2; ++al)
#pragma unroll
      for (int c = 0; c < 2; ++c)
        put4<BF>(buf + ((al * 2 + beta) * 32 + c * 16 + pr) * kRow, quad, fl, o.v[al][c]);
  };
  f32x16_t acc[1][1];
  zero_acc(acc);
  u32x4_t fb[2][2][1][2];   // [stage parity][run]
  auto load_tab = [&](auto J, int s) __attribute__((always_inline)) {
    const int sc = s < nst ? s : nst - 1;
#pragma unroll
    for (int e = 0; e < 2; ++e) load_frag(fb[decltype(J)::value][e][0], tab, 2 * sc + e);
  };
  auto step = [&](auto J, auto FULL, auto PH, int s) __attribute__((always_inline)) {
    constexpr int j0 = decltype(J)::value;
    lds_barrier();   // stage s is in LDS, stage s - 1 has been read
    u32x4_t fa[2][1][2];
#pragma unroll
    for (int e = 0; e < 2; ++e)
      read_frag(fa[e][0], lds + (j0 * 2 + e) * kRun, wave * 32, wave & 1);
    load_tab(IC<1 - j0>{}, s + 1);
    ld.raw(2 * (s + 2) + run, raw[j0]);
    if constexpr (decltype(PH)::value) window(s + 2);
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int e = 0; e < 2; ++e) mma_stage<BF, 1, 1>(acc, fa[e], fb[j0][e]);
    __builtin_amdgcn_s_setprio(0);
    if (decltype(FULL)::value || s + 1 < nst) convert(PH, s + 1, raw[1 - j0]);
  };
  auto loop = [&](auto PH) __attribute__((always_inline)) {
    load_tab(IC<0>{}, 0);
    ld.raw(run, raw[0]);
    ld.raw(2 + run, raw[1]);
    if constexpr (decltype(PH)::value) {
      window(0);
      window(1);
      lds_barrier();
    }
    convert(PH, 0, raw[0]);
    int s = 0;
    for (; s + 2 < nst; s += 2) {
      step(IC<0>{}, std::true_type{}, PH, s);
      step(IC<1>{}, std::true_type{}, PH, s + 1);
    }
    step(IC<0>{}, std::false_type{}, PH, s);
    if (s + 1 < nst) step(IC<1>{}, std::false_type{}, PH, s + 1);
  };
  if (LOAD == FOLD_FIELD && phased) loop(std::bool_constant<LOAD == FOLD_FIELD>{});
  else loop(std::false_type{});
  lds_barrier();
  f32x16_t& v = acc[0][0];
  const int lane = threadIdx.x & 63, lr = lane & 31, lk = lane >> 5;
  if constexpr (LOAD == FOLD_FIELD) {
    if (phased) {   // the y factor, as y_phase
      f32x16_t other;
      put_block(lds, v);
      lds_barrier();
      get_block<1>(lds, other);
      lds_barrier();
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        const double u = (double)(py0 + 8 * (r >> 2) + 4 * lk + (r & 3)) + on;
        const float2 w = turn(ph.cy * u);
        float2 q = make_float2(1.f, 0.f);
        if (ph.c2 != 0.0) q = turn(ph.c2 * u * u);
        const float2 e = cmul(make_float2(v[r] * w.x - other[r + 8] * w.y,
                                          v[r + 8] * w.x + other[r] * w.y), q);
        v[r] = e.x;
        v[r + 8] = e.y;
      }
    }
  }
  // rows of 64 bytes (the 16 k of a component), through a wave-private patch
  constexpr int kSmallRow = 80;
  uint8_t* patch = lds + wave * kRun;
  const long rb = 4L * kp;
  const int kvalid = kh - py0;
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      float x[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = 8 * q + 4 * lk + e < kvalid ? v[8 * c + 4 * q + e] : 0.f;
      uint8_t* d = patch + (c * 32 + lr) * kSmallRow + q * 32;
      if constexpr (BF) {
        uint32_t h[2], l[2];
        split2_bf16(x[0], x[1], h[0], l[0]);
        split2_bf16(x[2], x[3], h[1], l[1]);
        *(uint2*)(d + lk * 8) = make_uint2(h[0], h[1]);
        *(uint2*)(d + 16 + lk * 8) = make_uint2(l[0], l[1]);
      } else {
        *(float4*)(d + lk * 16) = make_float4(x[0], x[1], x[2], x[3]);
      }
    }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  uint8_t* out = a.out + (long)b * a.out_stride + 4L * py0;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int c = e >> 1, r = 16 * (e & 1) + (lane >> 2), piece = lane & 3;
    const uint4 x = *(const uint4*)(patch + (c * 32 + r) * kSmallRow + piece * 16);
    const int comp = ((wave & 1) * 2 + (wave >> 1)) * 2 + c;
    if (q0 + r < mh) *(uint4*)(out + (long)(comp * mh + q0 + r) * rb + piece * 16) = x;
  }
}

// ---------------------------------------------------------------------------
// A ring of NB stage buffers (16 KiB: 256 folded rows) filled straight from
// memory NB - 1 stages ahead, with the table fragments of the same stage in
// registers: the loop of the kernels whose folded operand is in memory.
// Counted vmcnt waits; one LDS object per buffer, so that the compiler's own
// wait before a fragment read covers that buffer's loads alone.
// mma(buffer, fragments) issues one stage's products.
// ---------------------------------------------------------------------------
template <int NB, int NT, typename BufF, typename IssueF, typename MmaF>
__device__ __forceinline__ void ring_loop(int nst, const uint8_t* const (&tab)[NT], BufF buf,
                                          IssueF issue_rows, MmaF mma) {
  constexpr int kPer = 2 * NT + 4;   // loads per wave and stage
  u32x4_t tf[NB][NT][2];
  auto issue = [&](auto J, int s) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NT; ++i) load_frag(tf[decltype(J)::value][i], tab[i], s);
    issue_rows(J, s);
  };
  // FULL: every stage the step waits past and issues exists (no branches, so
  // the compiler's counts stay exact across the loop's back edge)
  auto step = [&](auto J, auto FULL, int s) __attribute__((always_inline)) {
    constexpr bool full = decltype(FULL)::value;
    if (full || s + NB - 2 < nst)
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kPer * (NB - 2)) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    auto next = [&]() __attribute__((always_inline)) {
      if (full || s + NB - 1 < nst) issue(IC<(decltype(J)::value + NB - 1) % NB>{}, s + NB - 1);
    };
    mma(buf(J), tf[decltype(J)::value], next);
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
}

#define DLX_RING_BUFFERS(NB)                                                              \
  __shared__ __attribute__((aligned(1024))) uint8_t buf0[256 * kRow], buf1[256 * kRow];   \
  __shared__ __attribute__((aligned(1024))) uint8_t buf2[NB > 2 ? 256 * kRow : 16];       \
  __shared__ __attribute__((aligned(1024))) uint8_t buf3[NB > 3 ? 256 * kRow : 16];       \
  auto buf = [&](auto J) __attribute__((always_inline)) -> uint8_t* {                     \
    if constexpr (decltype(J)::value == 0) return buf0;                                   \
    else if constexpr (decltype(J)::value == 1) return buf1;                              \
    else if constexpr (decltype(J)::value == 2) return buf2;                              \
    else return buf3;                                                                     \
  }

// Stage 1 of a folded field in memory.
template <bool BF, int BNQ, int NB>
__global__ void __launch_bounds__(kThreads, 2)
fold_stage1_mem_kernel(FoldStage1 a) {
  using S = S1<BNQ>;
  constexpr int NI = S::NI, NJ = S::NJ;
  DLX_RING_BUFFERS(NB);
  const int kh = fold_half(a.n), mh = fold_half(a.m), mhp = fold_pad(mh), kp = fold_pad(kh);
  const int tq = (mh + BNQ - 1) / BNQ, tp = (kh + 31) / 32;
  const int id = xcd_order(blockIdx.x, tq * tp * a.batch);
  const int b = id / (tq * tp), t = id - b * (tq * tp);
  const int py0 = (t / tq) * 32, q0 = (t % tq) * BNQ;
  const int wave = threadIdx.x >> 6;
  const uint8_t* tab[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int blk = (q0 + S::col(wave)) / 32 + j, last = (mhp >> 5) - 1;
    tab[j] = a.table + (long)b * a.table_stride +
             table_block(wave >> 1, mhp, kp, blk < last ? blk : last);
  }
  const uint8_t* src = a.src + (long)b * a.src_stride;
  TileRows<256> at;
  at.init([&](int r) {
    const int y = py0 + (r & 31);
    return src + (long)((r >> 5) * kh + (y < kh ? y : kh - 1)) * 4 * kp;
  });
  f32x16_t acc[NI][NJ];
  zero_acc(acc);
  ring_loop<NB, NJ>(
      (kh + kStageK - 1) / kStageK, tab, buf,
      [&](auto J, int s) __attribute__((always_inline)) { at.issue(buf(J), s); },
      [&](const uint8_t* la, const u32x4_t (&fb)[NJ][2], auto next) __attribute__((always_inline)) {
        u32x4_t fa[NI][2];
#pragma unroll
        for (int i = 0; i < NI; ++i) read_frag(fa[i], la, S::arow(wave) + 32 * i);
        next();
        __builtin_amdgcn_s_setprio(1);
        mma_stage<BF, NI, NJ>(acc, fa, fb);
        __builtin_amdgcn_s_setprio(0);
      });
  __syncthreads();
  stage1_store<BF, BNQ>((wave & 1 ? buf1 : buf0) + (wave >> 1) * kPatch, acc, a.n, a.m,
                        a.out + (long)b * a.out_stride, py0, q0);
}
// ---------------------------------------------------------------------------
// Stage 2: F[(beta, alpha, c)][qy][qx] = sum_py T_beta[qy][py] U[(beta, alpha, c), qx][py],
// then the four mirrored outputs.  A workgroup takes BQ rows qy and 32 columns
// qx of all eight parts.  BQ = 64: wave (beta, h) holds the four (alpha, c)
// blocks of 32 rows, combines along x in registers, and trades one sign of x
// with the wave of the other beta through LDS, after which wave beta holds both
// signs of y at its sign of x.  BQ = 32, for launches that leave compute units
// idle: wave (beta, alpha) holds both components of one part, and two trades
// leave it the outputs of one sign of x (alpha) and one of y (beta).  Reading U
// and the products take similar times: 24-26 us split, 46-50 float32 at 64 wavelengths
// of 512^2 -> 256^2 (64 MB of U; the complex contraction took 50 and 176).
// ---------------------------------------------------------------------------
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
  constexpr int NJ = BQ == 64 ? 4 : 2;
  constexpr bool SWAP = EPI == FOLD_VJP;        // lanes run along qy, registers along qx
  DLX_RING_BUFFERS(NB);
  const int kh = fold_half(a.n), mh = fold_half(a.m), mhp = fold_pad(mh), kp = fold_pad(kh);
  const int lane = threadIdx.x & 63, lr = lane & 31, lk = lane >> 5;
  const int wave = threadIdx.x >> 6, beta = wave >> 1, h = wave & 1;
  const int q0 = qy0 + (BQ == 64 ? h * 32 : 0);   // the wave's rows
  const int blk = q0 / 32, last = (mhp >> 5) - 1;
  const uint8_t* tab[1] = {a.table + table_block(beta, mhp, kp, blk < last ? blk : last)};
  TileRows<256> bt;
  bt.init([&](int r) {
    const int q = qx0 + (r & 31);
    return a.mid + (long)((r >> 5) * mh + (q < mh ? q : mh - 1)) * 4 * kp;
  });
  f32x16_t acc[1][NJ];
  zero_acc(acc);
  ring_loop<NB, 1>(
      (kh + kStageK - 1) / kStageK, tab, buf,
      [&](auto J, int s) __attribute__((always_inline)) { bt.issue(buf(J), s); },
      [&](const uint8_t* lb, const u32x4_t (&fa)[1][2], auto next) __attribute__((always_inline)) {
        u32x4_t fb[NJ][2];
#pragma unroll
        for (int j = 0; j < NJ; ++j)
          read_frag(fb[j], lb, (beta * 4 + (BQ == 64 ? 0 : 2 * h) + j) * 32);
        next();
        __builtin_amdgcn_s_setprio(1);
        if constexpr (!SWAP) {
          mma_stage<BF, 1, NJ>(acc, fa, fb);
        } else {
          f32x16_t(&sw)[NJ][1] = reinterpret_cast<f32x16_t(&)[NJ][1]>(acc);
          mma_stage<BF, NJ, 1>(sw, fb, fa);
        }
        __builtin_amdgcn_s_setprio(0);
      });

  // ---- the mirrored outputs ----
  const float sg = a.inverse ? -1.f : 1.f;
  const float alpha = a.alpha;
  const int m = a.m, half = m >> 1;
  // (r, i) of the wave `XOR` away
  auto trade = [&](auto XOR, const f32x16_t& r, const f32x16_t& i, f32x16_t& tr,
                   f32x16_t& ti) __attribute__((always_inline)) {
    __syncthreads();
    put_block(buf0, r);
    put_block(buf1, i);
    __syncthreads();
    get_block<decltype(XOR)::value>(buf0, tr);
    get_block<decltype(XOR)::value>(buf1, ti);
  };
  // the wave's sign of x: + for 0, - for 1
  const int sx = BQ == 64 ? beta : h;
  auto col = [&](int qx) { return sx ? m - 1 - half - qx : half + qx; };
  const float d = beta ? -1.f : 1.f;

  // kr, ki: E at the wave's sign of x and y+ (BQ = 32: at the y sign of beta);
  // sr, si (BQ = 64): at y-.
  f32x16_t kr, ki, sr, si;
  if constexpr (BQ == 64) {
    // F(., x+-) = F_e -+ i s F_o; beta = 1 carries the factor -i s of the y sine
    const float ks = beta ? -sg : sg;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float er = acc[0][0][r], ei = acc[0][1][r], orr = acc[0][2][r], oi = acc[0][3][r];
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
    f32x16_t tr, ti;
    trade(IC<2>{}, sr, si, tr, ti);
    // y+: sum; y-: difference (the beta = 0 value first)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      sr[r] = d * (kr[r] - tr[r]); si[r] = d * (ki[r] - ti[r]);
      kr[r] += tr[r]; ki[r] += ti[r];
    }
  } else {
    f32x16_t tr, ti;
    trade(IC<1>{}, acc[0][0], acc[0][1], tr, ti);
    const float ks = h ? -sg : sg;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float er = h ? tr[r] : acc[0][0][r], ei = h ? ti[r] : acc[0][1][r];
      const float orr = h ? acc[0][0][r] : tr[r], oi = h ? acc[0][1][r] : ti[r];
      const float x = er + ks * oi, y = ei - ks * orr;
      kr[r] = beta ? sg * y : x;
      ki[r] = beta ? -sg * x : y;
    }
    trade(IC<2>{}, kr, ki, tr, ti);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      kr[r] = tr[r] + d * kr[r];
      ki[r] = ti[r] + d * ki[r];
    }
  }

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
      auto emit = [&](int y, float re, float im) __attribute__((always_inline)) {
        re *= alpha;
        im *= alpha;
        const long o = (long)y * m + x;
        if constexpr (EPI == FOLD_INTENSITY) {
          ((__attribute__((address_space(1))) float*)a.out)[o] = re * re + im * im;
        } else if constexpr (EPI == FOLD_STORE) {
          float2 v = make_float2(re, im);
          if (phased) {
            const double w = (double)y - 0.5 * (m - 1);
            v = cmul(v, turn(fma(ph.cy, w, fma(ph.c2 * w, w, tx0))));
          }
          ((float2*)a.out)[o] = v;
        } else {
          // the pupil's phasor at the pixel
          const double path = pupil_path(a.pupil.tx, pupil_coord(x, a.pupil.dx, a.pupil.x0),
                                         a.pupil.ty * pupil_coord(y, a.pupil.dx, a.pupil.x0),
                                         a.pupil.opd ? (double)a.pupil.opd[o] : 0.0);
          const double t0 = a.pupil.phase ? (double)a.pupil.phase[o] * 0.15915494309189535 : 0.0;
          const float2 u = pupil_phasor(path, a.inv_wl, t0, a.pupil.scale);
          const float am = a.pupil.amp ? a.pupil.amp[o] : 1.0f;
          ((float*)a.out)[o] = am * (u.x * im - u.y * re);
          if (a.out2) a.out2[o] = u.x * re + u.y * im;
        }
      };
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int qy = q0 + 8 * (r >> 2) + 4 * lk + (r & 3);
        if (qy < mh) {
          const int yp = half + qy, ym = m - 1 - yp;
          if constexpr (BQ == 64) {
            emit(yp, kr[r], ki[r]);
            emit(ym, sr[r], si[r]);
          } else {
            emit(beta ? ym : yp, kr[r], ki[r]);
          }
        }
      }
    }
  } else {
    // Ebar = 2 G alpha E, folded along y, then along x (the wave keeps the part
    // of its beta, and with BQ = 32 of its alpha)
    const int qy = q0 + lr;
    const int yp = half + (qy < mh ? qy : 0), ym = m - 1 - yp;
    uint8_t* patch = (wave & 1 ? buf1 : buf0) + (wave >> 1) * kPatch;
    uint8_t* out = (uint8_t*)a.out;
    const long orb = 4L * mhp;
    f32x16_t tr, ti;
    if constexpr (BQ == 64) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int qx = qx0 + 8 * (r >> 2) + 4 * lk + (r & 3);
        const int x = col(qx < mh ? qx : 0);
        const float gp = 2.f * alpha * a.G[(long)yp * m + x], gm = 2.f * alpha * a.G[(long)ym * m + x];
        const float pr = gp * kr[r], pi = gp * ki[r], mr = gm * sr[r], mi = gm * si[r];
        // keep the part of this wave's beta, send the other
        kr[r] = pr + d * mr; ki[r] = pi + d * mi;
        sr[r] = pr - d * mr; si[r] = pi - d * mi;
      }
      trade(IC<2>{}, sr, si, tr, ti);
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int qx = qx0 + 8 * (r >> 2) + 4 * lk + (r & 3);
        const int x = col(qx < mh ? qx : 0);
        const float g = 2.f * alpha * a.G[(long)(beta ? ym : yp) * m + x];
        kr[r] *= g;
        ki[r] *= g;
      }
      trade(IC<2>{}, kr, ki, tr, ti);
#pragma unroll
      for (int r = 0; r < 16; ++r) {   // y+ plus or minus y-
        kr[r] = tr[r] + d * kr[r];
        ki[r] = ti[r] + d * ki[r];
      }
      trade(IC<1>{}, kr, ki, tr, ti);
    }
    __syncthreads();
    const float dx = sx ? -1.f : 1.f;
#pragma unroll
    for (int c = 0; c < NJ; ++c) {   // (alpha, c), or the wave's alpha's c
      f32x16_t v;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float k = (c & 1) ? ki[r] : kr[r], o = (c & 1) ? ti[r] : tr[r];
        if constexpr (BQ == 64) v[r] = c < 2 ? k + o : d * (k - o);   // x+ plus or minus x-
        else v[r] = o + dx * k;
      }
      const int comp = ((BQ == 64 ? c >> 1 : h) * 2 + beta) * 2 + (c & 1);
      if (q0 < mh)
        store_block<BF>(patch, v, mh - qx0, out + (long)(comp * mh + q0) * orb + 4L * qx0, orb,
                        mh - q0);
    }
  }
}

template <bool BF, int EPI, int BQ, int NB>
__global__ void __launch_bounds__(kThreads, 2)
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

// Stage 1 of an uneven batch, from pre-folded float fields (rows (beta, py) of
// [px][e re, e im, o re, o im], fold_group_fields): a workgroup takes 32 rows
// py of one field and L = 128 / BNQ tiles of BNQ columns, each of any instance
// of that field.  The values loaded for a stage serve all L: per tile the
// instance's x shift rotates the even and odd parts (e' = e cos f + i o sin f,
// o' = o cos f + i e sin f; cos and sin of the stage's k from a window in LDS),
// the parts are split, and the tile's products run; the y shift is applied to
// the results.  768 instances of 256^2 to 1024^2 take 228 + 164 + 119 us in the
// three widths and 184 in stage 2 traced one by one, 610 in a row (the complex
// contractions 1360 in all); issue bounds it as the stage above.
template <int BNQ>
__global__ void __launch_bounds__(kThreads, 2)
fold_group_stage1_kernel(FoldGroup g) {
  using S = S1<BNQ>;
  constexpr int NI = S::NI, NJ = S::NJ, L = 128 / BNQ, kBuf = 256 * kRow;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[2 * kBuf];
  __shared__ float2 win[2][L][kStageK];
  const int t = group_tile(g);
  if (t < 0) return;
  const FoldRowTile rt = g.rows[t];
  const FoldColumns& cg = g.cols[rt.cols];
  const int n = cg.n, kh = fold_half(n), kp = fold_pad(kh), count = cg.count;
  const int py0 = (int)rt.row;
  const int nst = (kh + kStageK - 1) / kStageK, wave = threadIdx.x >> 6;
  const int quad = threadIdx.x & 3, beta = (threadIdx.x >> 2) & 1, py = threadIdx.x >> 3;
  const float4* row;
  {
    const int y = py0 + py < kh ? py0 + py : kh - 1;
    row = (const float4*)cg.src + ((long)beta * kh + y) * kp + quad * 4;
  }
  const uint8_t* tab[L][NJ];
#pragma unroll
  for (int l = 0; l < L; ++l) {
    const FoldColumns::Tile& c = cg.tile_of[l < count ? l : 0];
    const int mhp = fold_pad(fold_half(c.m)), last = (mhp >> 5) - 1;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int blk = (c.q0 + S::col(wave)) / 32 + j;
      tab[l][j] = c.table + table_block(wave >> 1, mhp, kp, blk < last ? blk : last);
    }
  }
  f32x16_t acc[L][NI][NJ];
#pragma unroll
  for (int l = 0; l < L; ++l) zero_acc(acc[l]);
  const double on = (n & 1) ? 0.0 : 0.5;
  const int wl = threadIdx.x / kStageK, we = threadIdx.x % kStageK;   // window entry of a thread
  const double wcx = wl < L ? cg.tile_of[wl < count ? wl : 0].cx : 0.0;
  auto window = [&](int s) {
    if (wl < L) win[s & 1][wl][we] = turn(wcx * ((double)(s * kStageK + we) + on));
  };
  float4 raw[2][4];
  auto load_raw = [&](auto J, int s) __attribute__((always_inline)) {
    const int sc = s < nst ? s : nst - 1;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      raw[decltype(J)::value][e] = __builtin_bit_cast(float4, load_global(row + sc * kStageK + e));
  };
  auto convert = [&](int s, int l, int slot, const float4 (&r)[4]) __attribute__((always_inline)) {
    float v[2][2][4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float2 w = win[s & 1][l][quad * 4 + e];
      v[0][0][e] = r[e].x * w.x - r[e].w * w.y;
      v[0][1][e] = r[e].y * w.x + r[e].z * w.y;
      v[1][0][e] = r[e].z * w.x - r[e].y * w.y;
      v[1][1][e] = r[e].w * w.x + r[e].x * w.y;
    }
    uint8_t* buf = lds + slot * kBuf;
    const int pr = part_row(py, beta), fl = part_slot(py, beta);
#pragma unroll
    for (int al = 0; al < 2; ++al)
#pragma unroll
      for (int c = 0; c < 2; ++c)
        put4<true>(buf + (((al * 2 + beta) * 2 + c) * 32 + pr) * kRow, quad, fl, v[al][c]);
  };
  u32x4_t fb[2][NJ][2];
  auto load_tab = [&](auto J, const uint8_t* const (&tb)[NJ], int s) __attribute__((always_inline)) {
    const int sc = s < nst ? s : nst - 1;
#pragma unroll
    for (int j = 0; j < NJ; ++j) load_frag(fb[decltype(J)::value][j], tb[j], sc);
  };
  // step (s, l): P = s & 1; slot and fragment set (s L + l) & 1.  ALL: the group
  // has L tiles; MORE: there is a next stage -- then no branch splits the step.
  auto step = [&](auto P, auto LL, auto ALL, auto MORE, int s) __attribute__((always_inline)) {
    constexpr bool all = decltype(ALL)::value, more = decltype(MORE)::value;
    constexpr int p = decltype(P)::value, l = decltype(LL)::value;
    constexpr int k = (p * L + l) & 1, ln = (l + 1) % L;
    lds_barrier();
    const int sn = l + 1 < L ? s : s + 1;   // the next step's stage
    u32x4_t fa[NI][2];
    if (all || l < count) {
#pragma unroll
      for (int i = 0; i < NI; ++i)
        read_frag(fa[i], lds + k * kBuf, S::arow(wave) + 32 * i, S::beta(wave, i));
    }
    load_tab(IC<1 - k>{}, tab[ln], sn);
    if constexpr (l == 0) {
      // L = 1 converts the next stage from raw[1 - p] in this step: two ahead
      if constexpr (L == 1) load_raw(P, s + 2);
      else load_raw(IC<1 - p>{}, s + 1);
      // the window of stage s is still read by this stage's converts if L > 1
      window(L == 1 ? s + 2 : s + 1);
    }
    if (all || l < count) mma_stage<true, NI, NJ>(acc[l], fa, fb[k]);
    if ((l + 1 < L || more || sn < nst) && (all || ln < count)) {
      if constexpr (l + 1 < L) convert(sn, ln, 1 - k, raw[p]);
      else convert(sn, ln, 1 - k, raw[1 - p]);
    }
  };
  auto stage = [&](auto P, auto ALL, auto MORE, int s) __attribute__((always_inline)) {
    step(P, IC<0>{}, ALL, MORE, s);
    if constexpr (L > 1) step(P, IC<1>{}, ALL, MORE, s);
    if constexpr (L > 2) {
      step(P, IC<2>{}, ALL, MORE, s);
      step(P, IC<3>{}, ALL, MORE, s);
    }
  };
  auto run = [&](auto ALL) __attribute__((always_inline)) {
    int s = 0;
    for (; s + 2 < nst; s += 2) {
      stage(IC<0>{}, ALL, std::true_type{}, s);
      stage(IC<1>{}, ALL, std::true_type{}, s + 1);
    }
    stage(IC<0>{}, ALL, std::false_type{}, s);
    if (s + 1 < nst) stage(IC<1>{}, ALL, std::false_type{}, s + 1);
  };
  load_tab(IC<0>{}, tab[0], 0);
  load_raw(IC<0>{}, 0);
  if constexpr (L == 1) load_raw(IC<1>{}, 1);
  window(0);
  if constexpr (L == 1) window(1);
  lds_barrier();
  convert(0, 0, 0, raw[0]);
  if (L == 1 || count == L) run(std::true_type{});
  else run(std::false_type{});
#pragma unroll
  for (int l = 0; l < L; ++l) {
    if (l >= count) break;
    const FoldColumns::Tile& c = cg.tile_of[l];
    lds_barrier();
    if (c.cy != 0.0) y_phase<BNQ>(lds, acc[l], 0.0, c.cy, n, py0);
    lds_barrier();
    stage1_store<true, BNQ>(lds + wave * kPatch, acc[l], n, c.m, c.mid, py0, c.q0);
  }
}

// A distinct field of the batch folded along both axes, once for all its
// instances: float rows (beta, py) of [px][e re, e im, o re, o im].
__global__ void __launch_bounds__(256)
fold_group_field_kernel(const FoldFieldJob* __restrict__ jobs) {
  const FoldFieldJob j = jobs[blockIdx.z];
  const int n = j.n, kh = fold_half(n), kp = fold_pad(kh);
  const int py = blockIdx.y, px = blockIdx.x * blockDim.x + threadIdx.x;
  if (py >= kh || px >= kp) return;
  float4 e = make_float4(0.f, 0.f, 0.f, 0.f), o = e;
  if (px < kh) {
    const int xp = (n >> 1) + px, xm = n - 1 - xp, yp = (n >> 1) + py, ym = n - 1 - yp;
    const float2 *rp = j.in + (long)yp * n, *rm = j.in + (long)ym * n;
    const float2 a = rp[xp], b = rp[xm], c = rm[xp], d = rm[xm];
    const float2 pe = {a.x + b.x, a.y + b.y}, po = {a.x - b.x, a.y - b.y};
    const float2 me = {c.x + d.x, c.y + d.y}, mo = {c.x - d.x, c.y - d.y};
    e = make_float4(pe.x + me.x, pe.y + me.y, po.x + mo.x, po.y + mo.y);
    o = make_float4(pe.x - me.x, pe.y - me.y, po.x - mo.x, po.y - mo.y);
  }
  float4* out = (float4*)j.out + (long)py * kp + px;
  out[0] = e;
  out[(long)kh * kp] = o;
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
  const int tx = (fold_half(g.m) + 31) / 32, local = t - p.tile;
  stage2_tile<true, FOLD_INTENSITY, kFoldTileQy, 4>(g, (local / tx) * kFoldTileQy, (local % tx) * 32);
}

// ---------------------------------------------------------------------------
// Tables and the pupil in memory
// ---------------------------------------------------------------------------

// One table: `table_quads` runs of four consecutive k of a row of both the cosine
// and the sine per thread, from the library's functions: the hardware's (max abs
// error 1.3e-7) are off alike in every table, which a sum over sources and
// wavelengths does not average out (24 stars of 8 wavelengths, relative error in
// 1e-7: 6.9 with them, 5.7 without).
//
// The split form rounds the 16 k of a stage one after another and adds what the
// pair hi + lo leaves of a value to the next: over neighbouring k, where a field
// varies slowly, the errors cancel.  Each rounded by itself they add coherently
// at the peak: the folds pair k with its mirror, so a table holds a quarter of
// the complex form's independent roundings.  Rms error of six fields 256^2 ->
// 256^2, shifted, in 1e-7 of the field / the intensity: 22.1 / 8.1 so, 12.9 /
// 4.1 with the carry, these functions and the lo * lo products of mma_stage, 20.3 /
// 5.8 in the unfolded complex form of three products; white fields 54.6 / 54.9,
// 52.1 / 52.0 and 54.2 / 54.4.  The fourth product costs 64 wavelengths of 512^2
// -> 256^2 76.6 -> 81.1 us, 768 uneven instances 658 -> 691.
template <bool BF>
__host__ __device__ constexpr int table_quads() { return BF ? 4 : 1; }
// Threads of the table contracting side n into side m.
template <bool BF>
__host__ __device__ inline int table_threads(int n, int m) {
  return fold_pad(fold_half(m)) * (fold_pad(fold_half(n)) / (4 * table_quads<BF>()));
}

template <bool BF>
__device__ __forceinline__ void table_entry(int t, double step, int n, int m,
                                            uint8_t* __restrict__ out) {
  constexpr int Q = table_quads<BF>();
  const int kh = fold_half(n), mh = fold_half(m), kp = fold_pad(kh), mhp = fold_pad(mh);
  if (t >= table_threads<BF>(n, m)) return;
  // consecutive threads take the 32 rows of a block
  const int runs = kp / (4 * Q), q = (t / (32 * runs)) * 32 + (t & 31);
  const int k0 = ((t >> 5) % runs) * 4 * Q;
  const double on = (n & 1) ? 0.0 : 0.5, om = (m & 1) ? 0.0 : 0.5;
  const double u = step * ((double)q + om);
  uint8_t* d[2];   // the stage's rows in the cosine and the sine
#pragma unroll
  for (int part = 0; part < 2; ++part)
    d[part] = out + table_block(part, mhp, kp, q >> 5) + (long)(k0 >> 4) * 2048 + (q & 31) * 16;
  float left[2] = {0.f, 0.f};
#pragma unroll
  for (int i = 0; i < Q; ++i) {
    const int quad = ((k0 >> 2) & 3) + i;
    float v[2][4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int p = k0 + 4 * i + e;
      float c = 0.f, s = 0.f;
      if (p < kh && q < mh) {
        double ph = u * ((double)p + on);
        ph -= rint(ph);
        sincospif(2.0f * (float)ph, &s, &c);
        if (p == 0 && (n & 1)) c *= 0.5f;   // the centre, folded onto itself
      }
      v[0][e] = c;
      v[1][e] = s;
    }
    // the quad's place in its stage: lane half (quad / 2), and, split, the run of
    // hi and of lo pieces with 8 bytes each; float32, one run of 16 bytes
#pragma unroll
    for (int part = 0; part < 2; ++part) {
      uint8_t* o = d[part] + (quad >> 1) * 512;
      if constexpr (BF) {
        uint32_t h[4], lo[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma clang fp contract(off)
          const bool in = k0 + 4 * i + e < kh && q < mh;
          const float x = in ? v[part][e] + left[part] : 0.f;
          h[e] = bf16x2_rne(x, 0.f);
          const float r = x - __uint_as_float(h[e] << 16);
          lo[e] = bf16x2_rne(r, 0.f);
          left[part] = r - __uint_as_float(lo[e] << 16);
        }
        *(uint2*)(o + (quad & 1) * 8) = make_uint2(h[0] | h[1] << 16, h[2] | h[3] << 16);
        *(uint2*)(o + 1024 + (quad & 1) * 8) = make_uint2(lo[0] | lo[1] << 16, lo[2] | lo[3] << 16);
      } else {
        *(float4*)(o + (quad & 1) * 1024) = make_float4(v[part][0], v[part][1], v[part][2], v[part][3]);
      }
    }
  }
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

// Most wavelengths per thread: the planes are read once for them.
constexpr int kPupilWl = 16;

template <bool BF, bool VEC>
__global__ void __launch_bounds__(256)
fold_pupil_kernel(FoldPupil pup, FoldSteps wl, int nb, int per, int n,
                  uint8_t* __restrict__ out, long stride) {
  const int kh = fold_half(n);
  const long rb = fold_row_bytes(n);
  const int py = blockIdx.x * 32 + (threadIdx.x >> 3);
  const int beta = threadIdx.x & 1, quad = (threadIdx.x >> 1) & 3, s = blockIdx.y;
  PupilLoad<VEC, true, true> pl;
  pl.init(pup, n, py, beta, quad, 0.0);
  typename PupilLoad<VEC, true, true>::Raw raw{};
  pl.raw(s, raw);
  const int b0 = blockIdx.z * per, b1 = b0 + per < nb ? b0 + per : nb;
  for (int b = b0; b < b1; ++b) {
    pl.inv_wl = wl.step[b];
    FoldPart o;
    pl.part(s, beta, raw, o);
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
// The pupil's rows can be read in whole runs of four (a missing plane is aligned).
bool pupil_vec(const FoldPupil& p, int n) {
  return n % 8 == 0 && aligned16(p.opd) && aligned16(p.amp) && aligned16(p.phase);
}

template <bool BF, int LOAD, bool VEC, int BNQ>
void stage1_go(const FoldStage1& a, long tiles, hipStream_t s) {
  if constexpr (LOAD == FOLD_MEM)
    hipLaunchKernelGGL((fold_stage1_mem_kernel<BF, BNQ, BNQ == 128 ? 3 : 4>), dim3((unsigned)tiles), dim3(kThreads), 0,
                       s, a);
  else
    hipLaunchKernelGGL((fold_stage1_kernel<BF, LOAD, VEC, BNQ>), dim3((unsigned)tiles),
                       dim3(kThreads), 0, s, a);
}

template <bool BF, int LOAD, bool VEC>
hipError_t stage1_width(const FoldStage1& a, hipStream_t s) {
  const int mh = fold_half(a.m), tp = (fold_half(a.n) + 31) / 32;
  auto tiles = [&](int w) { return (long)((mh + w - 1) / w) * tp * a.batch; };
  // A wider tile forms the field fewer times; a launch of fewer tiles leaves
  // compute units idle.  Measured per launch, us, at 16 / 32 / 64 / 128 columns
  // (16: the 16-row kernel at 32), 512^2 -> 256^2 pupils:
  //   tiles of 64   float32                     split
  //        128      20.0 / 21.4 / 28.1 / 42.7   14.1 / 15.8 / 18.0 / 21.2
  //        192      27.2 / 31.4 / 28.4 / 43.9   18.5 / 22.3 / 19.7 / 22.6
  //        256      33.5 / 32.3 / 29.1 / 44.5   22.2 / 22.9 / 20.8 / 24.0
  //        320      43.4 / 44.2 / 46.6 / 44.7   25.6 / 28.2 / 26.5 / 24.7
  //       1024       115 /  109 / 94.2 / 81.8   68.0 / 67.4 / 51.4 / 40.3
  // and for a folded field in memory, at 32 / 64 / 128:
  //        128      16.6 / 23.7 / 39.1          11.0 / 13.2 / 20.2
  //        256      26.6 / 25.6 / 42.1          17.2 / 16.4 / 22.9
  //       1024      90.6 / 88.7 / 85.9          65.9 / 49.2 / 46.8
  // (measured at this geometry; other sides enter by their tile counts).  Three
  // 64-column tiles leave a quarter of two 128-column ones empty: float32, bound by
  // its products, takes 64 then (24 fields 511^2 -> 257^2, both stages: 145.3 us at
  // 128 columns, 123.8 at 64; 126.3 and 138.0 at 64 of 512^2 -> 256^2; five tiles, 8 of
  // 512^2 -> 620^2, 94.1 and 98.5, eleven, 4 of 512^2 -> 1300^2, 133.9 and 138.6), the
  // split form, bound by forming the parts, does not (62.9 and 68.3).
  const bool whole = BF || (mh + 63) / 64 != 3;
  if (mh > 64 && whole && tiles(64) > 256) stage1_go<BF, LOAD, VEC, 128>(a, tiles(128), s);
  else if (mh > 32 && tiles(64) >= 192) stage1_go<BF, LOAD, VEC, 64>(a, tiles(64), s);
  else if (LOAD != FOLD_MEM && tiles(32) < 384) {
    if constexpr (LOAD != FOLD_MEM)
      hipLaunchKernelGGL((fold_stage1_small_kernel<BF, LOAD, VEC>),
                         dim3((unsigned)((mh + 31) / 32 * ((fold_half(a.n) + 15) / 16) * a.batch)),
                         dim3(kThreads), 0, s, a);
  } else stage1_go<BF, LOAD, VEC, 32>(a, tiles(32), s);
  return hipGetLastError();
}

template <bool BF>
hipError_t stage1_load(const FoldStage1& a, FoldLoad load, hipStream_t s) {
  if (load == FOLD_MEM) return stage1_width<BF, FOLD_MEM, true>(a, s);
  if (load == FOLD_PUPIL && (a.pupil.phase || (!a.pupil.opd && !a.pupil.amp))) {
    // callers write such pupils to memory first where they have the room
    return pupil_vec(a.pupil, a.n) ? stage1_width<BF, kPupilAny, true>(a, s)
                                   : stage1_width<BF, kPupilAny, false>(a, s);
  }
  if (load == FOLD_PUPIL) {
    const bool vec = pupil_vec(a.pupil, a.n);
    if (a.pupil.tx != 0.0 || a.pupil.ty != 0.0)
      return vec ? stage1_width<BF, kPupilTilt, true>(a, s) : stage1_width<BF, kPupilTilt, false>(a, s);
    return vec ? stage1_width<BF, FOLD_PUPIL, true>(a, s) : stage1_width<BF, FOLD_PUPIL, false>(a, s);
  }
  const bool vec = a.n % 8 == 0 && aligned16(a.src) && a.src_stride % 16 == 0;
  return vec ? stage1_width<BF, FOLD_FIELD, true>(a, s) : stage1_width<BF, FOLD_FIELD, false>(a, s);
}

template <bool BF, int EPI>
hipError_t stage2_size(const FoldStage2& a, hipStream_t s) {
  const int mh = fold_half(a.m), tx = (mh + 31) / 32;
  auto tiles = [&](int q) { return (long)tx * ((mh + q - 1) / q) * a.batch; };
  // 32 rows a workgroup where 64 leave half of the compute units idle (or half of
  // the waves, at mh <= 32).  us at 32 / 64 rows, 512^2 -> 256^2, by tiles of 64:
  // 64: 13.8 / 21.9 float32, 8.5 / 11.2 split; 128: 14.4 / 22.2, 9.7 / 12.0; 160:
  // 26.4 / 22.5, 14.6 / 12.5; 512: 50.8 / 45.9, 31.1 / 24.2; one wavelength of 256^2 ->
  // 128^2 (4 tiles) 11.2 / 15.0 float32
  if (mh <= 32 || tiles(64) <= 128)
    hipLaunchKernelGGL((fold_stage2_kernel<BF, EPI, 32, 4>), dim3((unsigned)tiles(32)),
                       dim3(kThreads), 0, s, a);
  else
    hipLaunchKernelGGL((fold_stage2_kernel<BF, EPI, 64, 4>), dim3((unsigned)tiles(64)),
                       dim3(kThreads), 0, s, a);
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
      const int work = split ? table_threads<true>(kn, km) : table_threads<false>(kn, km);
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
  const bool vec = pupil_vec(p, n);
  for (int b0 = 0; b0 < nb; b0 += FoldSteps::kMax) {
    const int k = nb - b0 < FoldSteps::kMax ? nb - b0 : FoldSteps::kMax;
    FoldSteps wl;
    for (int i = 0; i < k; ++i) wl.step[i] = inv_wl[b0 + i];
    // a thread forms its wavelengths one after another: fewer each while the launch
    // has less than a workgroup per compute unit (4 of 512^2
    // with a phase plane onto 256^2: 128 at 16 each; the PSF 37.5 -> 33.9 us)
    const int px = (fold_half(n) + 31) / 32, py = fold_pad(fold_half(n)) / kStageK;
    int per = kPupilWl;
    while (per > 1 && px * py * ((k + per - 1) / per) < 256) per >>= 1;
    const dim3 grid(px, py, (k + per - 1) / per);
    uint8_t* o = out + (long)b0 * stride;
    if (split && vec) hipLaunchKernelGGL((fold_pupil_kernel<true, true>), grid, dim3(256), 0, s, p, wl, k, per, n, o, stride);
    else if (split) hipLaunchKernelGGL((fold_pupil_kernel<true, false>), grid, dim3(256), 0, s, p, wl, k, per, n, o, stride);
    else if (vec) hipLaunchKernelGGL((fold_pupil_kernel<false, true>), grid, dim3(256), 0, s, p, wl, k, per, n, o, stride);
    else hipLaunchKernelGGL((fold_pupil_kernel<false, false>), grid, dim3(256), 0, s, p, wl, k, per, n, o, stride);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

int fold_group_width(int m) {
  const int mh = fold_half(m);
  return mh > 64 ? 128 : mh > 32 ? 64 : 32;
}

int fold_group_table_threads(int n, int m) { return table_threads<true>(n, m); }

hipError_t launch_fold_group_tables(const FoldTableJob* jobs, int njobs, int most, hipStream_t s) {
  hipLaunchKernelGGL(fold_group_table_kernel, dim3(njobs, (unsigned)((most + 255) / 256)), dim3(256),
                     0, s, jobs);
  return hipGetLastError();
}

static unsigned group_grid(const FoldGroup& g) {
  int most = 0;
  for (int x = 0; x < kXcds; ++x) most = std::max(most, g.xcd[x + 1] - g.xcd[x]);
  return (unsigned)(kXcds * most);
}

hipError_t launch_fold_group_stage1(const FoldGroup& g, int width, hipStream_t s) {
  const dim3 grid(group_grid(g)), block(kThreads);
  if (grid.x == 0) return hipSuccess;
  if (width == 128) hipLaunchKernelGGL(fold_group_stage1_kernel<128>, grid, block, 0, s, g);
  else if (width == 64) hipLaunchKernelGGL(fold_group_stage1_kernel<64>, grid, block, 0, s, g);
  else hipLaunchKernelGGL(fold_group_stage1_kernel<32>, grid, block, 0, s, g);
  return hipGetLastError();
}

hipError_t launch_fold_group_fields(const FoldFieldJob* jobs, int njobs, int most, hipStream_t s) {
  const int kh = fold_half(most);
  for (int j0 = 0; j0 < njobs; j0 += 65535) {
    const int k = njobs - j0 < 65535 ? njobs - j0 : 65535;
    hipLaunchKernelGGL(fold_group_field_kernel, dim3((fold_pad(kh) + 255) / 256, kh, k), dim3(256), 0,
                       s, jobs + j0);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_fold_group_stage2(const FoldGroup& g, hipStream_t s) {
  const dim3 grid(group_grid(g));
  if (grid.x == 0) return hipSuccess;
  hipLaunchKernelGGL(fold_group_stage2_kernel, grid, dim3(kThreads), 0, s, g);
  return hipGetLastError();
}

bool fold_pupil_in_loader(const FoldPupil& p, int n, int m) {
  const int mh = fold_half(m);
  if (!p.phase && (p.opd || p.amp)) return mh <= 256;
  return n <= 256 ? mh <= 256 : pupil_vec(p, n) && mh <= 128;
}

}  // namespace dlx
