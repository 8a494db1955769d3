// Folded transforms: the MFT as real cosine / sine contractions.
//
// The grids of a matrix Fourier transform are symmetric about zero, so per axis
//   W[l][k] = exp(-i s 2 pi a_k b_l),  a_{n-1-k} = -a_k,  b_{m-1-l} = -b_l   (s = +-1)
// and with the input's even and odd parts over the mirrored pairs k+, k- = n-1-k+,
//   X_e[p] = x[k+] + x[k-],   X_o[p] = x[k+] - x[k-],   p = 0 .. ceil(n/2) - 1,
// the outputs at the mirrored pair l+-, q = 0 .. ceil(m/2) - 1, are
//   (W x)[l+-] = sum_p C[q][p] X_e[p]  -+  i s sum_p S[q][p] X_o[p],
//   C = cos(2 pi a_p b_q),  S = sin(2 pi a_p b_q).
// On both axes a field becomes four parity parts (beta along y, alpha along x;
// each complex), every contraction is real x complex over half the k and half
// the outputs -- a quarter of the products of the complex form -- and the four
// mirrored outputs come out of one set of sums.  For odd n the centre pairs
// with itself: its fold is 2x and its table column carries 1/2.
//
// Layouts.  A "folded matrix" is real, row-major with k contiguous, k padded
// with zeros to a multiple of 32 (rows start on 128-byte lines); 4 bytes per
// element in both forms: float32, or split-bf16 chunks of 8 k as 16 bytes of
// hi = bf16(x) then 16 bytes of lo = bf16(x - hi).
//   table      [C, S][rows padded to 32][k], in MFMA fragment order
//   field      rows ((alpha * 2 + beta) * 2 + c) * ceil(n/2) + py,   k = px
//   stage-1 out rows ((beta * 2 + alpha) * 2 + c) * ceil(m/2) + qx,  k = py
// with c = 0 real, 1 imaginary.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include "dlx_internal.h"

namespace dlx {

constexpr int kFoldPad = 32;
__host__ __device__ inline int fold_half(int n) { return (n + 1) / 2; }
__host__ __device__ inline int fold_pad(int h) { return (h + kFoldPad - 1) / kFoldPad * kFoldPad; }
// Bytes of one folded row of a side-n axis.
__host__ __device__ inline long fold_row_bytes(int n) { return 4L * fold_pad(fold_half(n)); }
// Bytes of the table contracting a side-n axis into side m.
__host__ __device__ inline long fold_table_bytes(int n, int m) {
  return 2L * fold_pad(fold_half(m)) * fold_row_bytes(n);
}
// Bytes of a folded n x n field, and of the stage-1 result n x n -> n x m.
__host__ __device__ inline long fold_field_bytes(int n) { return 8L * fold_half(n) * fold_row_bytes(n); }
__host__ __device__ inline long fold_mid_bytes(int n, int m) {
  return 8L * fold_half(m) * fold_row_bytes(n);
}

// Phase step of one MFT axis: 2 pi step (p + o_n)(q + o_m), o = 0 (odd) or 1/2
// (even), is the table's angle; turns.
inline double fold_step(const dlx_mft_geom& g, double wavelength, double dx, double p_out) {
  double s = p_out * dx / wavelength;
  if (g.has_focal) s /= (g.focal_length + g.focal_shift);
  return s;
}

struct FoldSteps {
  static constexpr int kMax = 128;
  double step[kMax];
};

// Tables of nb steps, contracting side n into side m (out + b * stride); with
// `adjoint` the tables of the transposed contraction, side m into side n,
// follow each at out + b * stride + fold_table_bytes(n, m).
hipError_t launch_fold_tables(const double* step, int nb, int n, int m, bool split, bool adjoint,
                              uint8_t* out, long stride, hipStream_t s);

// Where stage 1 takes its field from.
enum FoldLoad {
  FOLD_MEM = 0,     // folded rows in memory
  FOLD_PUPIL = 1,   // phasors of amplitude and OPD planes, formed in the loader
  FOLD_FIELD = 2,   // a complex64 field (optionally times a separable phase)
};

// A separable phase over a grid's centred indices u = k - (side - 1) / 2, in turns:
// c2 (ux^2 + uy^2) + cx ux + cy uy + c0.  An output or input shift of the MFT
// is the linear part, the Collins kernel's chirps the quadratic one.
struct FoldPhase {
  double c2, cx, cy, c0;
};

// The pupil of instance b: a(y, x) exp(2 pi i path(y, x) inv_wl[b]),
// path = tx X + ty Y + opd (FP64), a = scale amp, times exp(i phase) (each plane may be null).
struct FoldPupil {
  const float* opd; const float* amp; const float* phase;
  double dx, x0, tx, ty;
  float scale;
};

struct FoldStage1 {
  static constexpr int kMaxBatch = 64;
  int n, m, batch;                     // field side, output side
  const uint8_t* src; long src_stride; // FOLD_MEM / FOLD_FIELD, bytes per instance
  const uint8_t* table; long table_stride;
  uint8_t* out; long out_stride;
  FoldPupil pupil;                     // FOLD_PUPIL
  double inv_wl[kMaxBatch];
  FoldPhase phase[kMaxBatch];          // FOLD_FIELD: multiplies the field
};

enum FoldEpilogue {
  FOLD_INTENSITY = 0,   // out[b](ly, lx) = |alpha E|^2, float
  FOLD_STORE = 1,       // out[b](ly, lx) = alpha E exp(2 pi i phase(ly, lx)), complex64
  FOLD_VJP = 2,         // folded rows ((alpha, beta, c), qy), k = qx, of 2 G alpha E
  FOLD_GRAD = 3,        // out[b](y, x) = Im(conj(P) alpha E), out2 (optional) = Re(conj(U) alpha E)
};

struct FoldStage2 {
  static constexpr int kMaxBatch = 64;
  int n, m, batch;                     // contracted side (the field's), output side
  int inverse;                         // s = -1
  const uint8_t* table; long table_stride;
  const uint8_t* mid; long mid_stride; // stage-1 result
  void* out; long out_stride;          // elements (INTENSITY, STORE, GRAD) or bytes (VJP)
  float alpha[kMaxBatch];
  const float* G;                      // VJP: dL/dPSF, m x m
  float* out2;                         // GRAD
  FoldPupil pupil;                     // GRAD: P, U = P / a at amplitude scale
  double inv_wl[kMaxBatch];
  FoldPhase phase[kMaxBatch];          // STORE: multiplies the result
};

hipError_t launch_fold_stage1(const FoldStage1& a, FoldLoad load, bool split, hipStream_t s);
hipError_t launch_fold_stage2(const FoldStage2& a, FoldEpilogue epi, bool split, hipStream_t s);

// Uneven batches (split form): |alpha W_y P W_x^T|^2 of many (field, sides,
// step, shift) instances into float planes; descriptors in device memory.
// Stage 2: one problem per instance, whose tiles are [tile, ...) of the list,
// numbered column-fastest.
struct FoldProblem {
  const uint8_t* table;
  const uint8_t* mid;
  float* out;
  float alpha;
  int n, m, inverse, tile, pad_;
};
// Stage 1: up to 128 / width column tiles, of any instances of one pre-folded
// field, worked through by one workgroup per 32 rows.  cx, cy: the turns per
// index of an instance's shift.
struct FoldColumns {
  const uint8_t* src;
  int n, count;
  struct Tile {
    const uint8_t* table;
    uint8_t* mid;
    double cx, cy;
    int q0, m;
  } tile_of[4];
};
struct FoldRowTile {
  uint32_t cols, row;   // column group, first row
};
// A launch over a tile list: stage-1 tiles of column groups (rows), or
// stage-2 tiles' problems (map); XCD x runs [xcd[x], xcd[x + 1]).
struct FoldGroup {
  const FoldProblem* probs;
  const FoldColumns* cols;
  const FoldRowTile* rows;
  const uint32_t* map;
  int xcd[9];
};
struct FoldTableJob {
  uint8_t* out;
  double step;
  int n, m;
};
struct FoldFieldJob {
  const float2* in;
  uint8_t* out;        // fold_field_bytes(n)
  int n, pad_;
};
// Output columns per stage-1 tile for an output side m (32, 64 or 128), and
// the rows and columns of the tiles.
int fold_group_width(int m);
constexpr int kFoldTileQy = 64, kFoldTileQx = 32, kFoldTilePy = 32;
// `most`: fold_group_table_threads of the largest table.
int fold_group_table_threads(int n, int m);
hipError_t launch_fold_group_tables(const FoldTableJob* jobs, int njobs, int most, hipStream_t s);
// `most`: the largest field's side.
hipError_t launch_fold_group_fields(const FoldFieldJob* jobs, int njobs, int most, hipStream_t s);
hipError_t launch_fold_group_stage1(const FoldGroup& g, int width, hipStream_t s);
hipError_t launch_fold_group_stage2(const FoldGroup& g, hipStream_t s);

// The folded pupil written to memory (FOLD_MEM rows), bit for bit what
// FOLD_PUPIL forms.
hipError_t launch_fold_pupil(const FoldPupil& p, const double* inv_wl, int nb, int n, bool split,
                             uint8_t* out, long stride, hipStream_t s);

// True where forming the pupil in the loader beats writing it first.  Each
// 128-column tile forms the pupil again.  With a phase plane, or no plane, the
// loader tests for every plane: up to two of 64 columns that costs less than a launch
// that writes the pupil where it loads whole runs (16 wavelengths of 512^2 -> 128^2
// 31.7 against 40.1 us split, 41.9 against 47.7 float32; 4 of 1024^2 -> 512^2 72.0
// against 55.3), single values only on small pupils (5 of 300^2 -> 101^2 26.2 against
// 27.2; 11 of 401^2 -> 173^2 38.1 against 35.2).
bool fold_pupil_in_loader(const FoldPupil& p, int n, int m);

}  // namespace dlx
