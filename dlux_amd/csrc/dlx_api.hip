// extern "C" entry points of libdlux_amd (declared in include/dlux_amd.h):
// argument validation, workspace carving and kernel orchestration.
#include <cstdarg>
#include <cmath>
#include <cstdlib>
#include <mutex>
#include <vector>

#include "dlx_fold.h"
#include "dlx_internal.h"

namespace dlx {

namespace {
thread_local std::string g_err;
}

void set_error(const char* fmt, ...) {
  char buf[1024];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_err = buf;
}
void clear_error() { g_err.clear(); }

namespace {

// Instances per fused launch of the polychromatic PSF (bounds the workspace).
constexpr int kWlChunk = 64;

// The pupil generated in stage 1's loader (default); DLUX_AMD_PUPIL_PROLOGUE=0
// writes it with the pupil kernel instead (read at every call, for
// comparisons).
bool pupil_prologue_enabled() {
  const char* v = getenv("DLUX_AMD_PUPIL_PROLOGUE");
  return !(v && v[0] == '0');
}

// Optional live timing of the two MFT contraction launches of dlx_psf_poly:
// hipEvents recorded on the caller's stream around each launch.
struct ProfSlot {
  hipEvent_t beg, end;
  int stage;
};
constexpr int kProfSlots = 8192;
struct Profiler {
  int enabled = 0;
  int n = 0;
  std::vector<ProfSlot> slots;
} g_prof;

int prof_begin(int stage, hipStream_t s, int* slot) {
  *slot = -1;
  if (!g_prof.enabled || g_prof.n >= kProfSlots) return DLX_OK;
  if ((int)g_prof.slots.size() <= g_prof.n) {
    ProfSlot ps{};
    DLX_HIP(hipEventCreate(&ps.beg));
    DLX_HIP(hipEventCreate(&ps.end));
    g_prof.slots.push_back(ps);
  }
  *slot = g_prof.n++;
  g_prof.slots[*slot].stage = stage;
  DLX_HIP(hipEventRecord(g_prof.slots[*slot].beg, s));
  return DLX_OK;
}

int prof_end(int slot, hipStream_t s) {
  if (slot < 0) return DLX_OK;
  DLX_HIP(hipEventRecord(g_prof.slots[slot].end, s));
  return DLX_OK;
}

int check_geom(const dlx_mft_geom* g) {
  DLX_CHECK_ARG(g != nullptr, "geom is NULL");
  DLX_CHECK_ARG(g->n_in > 0 && g->n_in <= 16384, "n_in must be in [1, 16384], got %d", g->n_in);
  DLX_CHECK_ARG(g->n_out > 0 && g->n_out <= 16384, "n_out must be in [1, 16384], got %d",
                g->n_out);
  if (g->has_focal)
    DLX_CHECK_ARG(std::isfinite(g->focal_length + g->focal_shift) &&
                      (g->focal_length + g->focal_shift) != 0.0,
                  "focal_length + focal_shift must be finite and non-zero");
  return DLX_OK;
}

}  // namespace

size_t mat_bytes(long rows, long k, bool split) {
  return split ? (size_t)rows * ((k + 7) / 8) * 64 : (size_t)rows * k * sizeof(float2);
}

namespace {

// The psf chain's buffers for a chunk of c wavelengths: the tables (used when
// they are not taken from the cache), the stage-1 result, the per-wavelength
// |E|^2 planes and, when `bytes` leaves room for it, the folded pupil.
struct PsfLayout {
  size_t T, U, I, P, total;   // total without P
};
PsfLayout psf_layout(const dlx_mft_geom& g, int c) {
  PsfLayout L;
  L.T = align_up((size_t)c * fold_table_bytes(g.n_in, g.n_out));
  L.U = align_up((size_t)c * fold_mid_bytes(g.n_in, g.n_out));
  L.I = align_up((size_t)c * g.n_out * g.n_out * sizeof(float));
  L.P = align_up((size_t)c * fold_field_bytes(g.n_in));
  L.total = L.T + L.U + L.I;
  return L;
}

// Workspace of the psf chain: a complex pupil, two complex matrices and the
// planes per wavelength (psf_plain_bytes) -- which the folded buffers fit in on
// all but the smallest grids -- so that the limits a caller meets do not depend
// on how the chain lays its buffers out.
size_t psf_plain_bytes(const dlx_mft_geom& g, int c, bool split) {
  return align_up((size_t)c * mat_bytes(g.n_in, g.n_in, split)) +
         2 * align_up((size_t)c * mat_bytes(g.n_out, g.n_in, split)) +
         align_up((size_t)c * g.n_out * g.n_out * sizeof(float));
}
size_t psf_poly_bytes(const dlx_mft_geom& g, int c, bool split) {
  const size_t plain = psf_plain_bytes(g, c, split), fold = psf_layout(g, c).total;
  return plain > fold ? plain : fold;
}

// The cosine / sine tables of nb phase steps contracting side n into side m
// (and, with `adjoint`, of the transposed contraction), from the device cache
// or generated into `ws` when the cache is bypassed.  Equal steps share one table
// (stride 0).
struct FoldTables {
  const uint8_t *fwd, *adj;
  long stride;
};
// What a call leaves in the cache: the PSF's entry holds both directions, for the
// gradient that may follow, and is made on the first sighting of its steps, as a
// field transform's of the forward direction is; a canonical transform's is made on
// the second, as a caller that scans planes or wavelengths never asks for one again.
enum TableUse { TABLES_PSF, TABLES_FIELD, TABLES_LCT };
int fold_tables(int n, int m, const std::vector<double>& steps, bool split, bool adjoint,
                TableUse use, bool use_cache, uint8_t* ws, hipStream_t s, FoldTables* out,
                CacheLease* lease) {
  const long tf = fold_table_bytes(n, m), ta = fold_table_bytes(m, n);
  bool one = true;
  for (double v : steps) one = one && v == steps[0];
  const int nb = one ? 1 : (int)steps.size();
  const bool both = use == TABLES_PSF;
  void* mem = nullptr;
  bool fresh = true;
  if (use_cache) {
    std::vector<double> key = {2001.0, (double)n, (double)m, split ? 1.0 : 0.0, both ? 1.0 : 0.0};
    key.insert(key.end(), steps.begin(), steps.begin() + nb);
    if (int st = cache_acquire_raw(key, (size_t)nb * (both ? tf + ta : tf), s, &mem, &lease->h,
                                   &fresh, use != TABLES_LCT))
      return st;
  }
  uint8_t* base = mem ? (uint8_t*)mem : ws;
  const bool adj = adjoint || (mem && both);
  const long stride = adj ? tf + ta : tf;
  out->stride = one ? 0 : stride;
  out->fwd = base;
  out->adj = base + tf;
  if (fresh) {
    DLX_HIP(launch_fold_tables(steps.data(), nb, n, m, split, adj, base, stride, s));
    if (int st = cache_ready(lease->h, s)) return st;
  }
  return DLX_OK;
}

std::vector<double> psf_steps(const dlx_mft_geom& g, int nb, const double* wl, double dx,
                              double p_out) {
  std::vector<double> st(nb);
  for (int i = 0; i < nb; ++i) st[i] = fold_step(g, wl[i], dx, p_out);
  return st;
}

// The transform of `batch` complex64 fields with per-instance phase steps,
// input and output phases (either may be NULL) and scales: folded stage 1
// loading the fields, stage 2 storing complex64.  `ws`: tables of the batch,
// then the stage-1 results of a chunk (field_transform_bytes).
constexpr int kFieldChunk = FoldStage1::kMaxBatch;
size_t field_transform_bytes(int n, int m, int batch) {
  const int c = batch < kFieldChunk ? batch : kFieldChunk;
  return align_up((size_t)batch * fold_table_bytes(n, m)) +
         align_up((size_t)c * fold_mid_bytes(n, m));
}
int field_transform(int n, int m, int batch, bool inverse, const std::vector<double>& steps,
                    TableUse use, const FoldPhase* pin, const FoldPhase* pout, const double* alpha,
                    const void* in, void* out, bool split, uint8_t* ws, hipStream_t s) {
  CacheLease h(s);
  FoldTables tab;
  if (int st = fold_tables(n, m, steps, split, false, use, true, ws, s, &tab, &h)) return st;
  uint8_t* U = ws + align_up((size_t)batch * fold_table_bytes(n, m));
  for (int b0 = 0; b0 < batch; b0 += kFieldChunk) {
    const int nb = batch - b0 < kFieldChunk ? batch - b0 : kFieldChunk;
    FoldStage1 f{};
    f.n = n; f.m = m; f.batch = nb;
    f.src_stride = 8L * n * n;
    f.src = (const uint8_t*)in + b0 * f.src_stride;
    f.table = tab.fwd + b0 * tab.stride; f.table_stride = tab.stride;
    f.out = U; f.out_stride = fold_mid_bytes(n, m);
    FoldStage2 e{};
    e.n = n; e.m = m; e.batch = nb; e.inverse = inverse;
    e.table = f.table; e.table_stride = tab.stride;
    e.mid = U; e.mid_stride = f.out_stride;
    e.out_stride = (long)m * m;
    e.out = (float2*)out + b0 * e.out_stride;
    for (int i = 0; i < nb; ++i) {
      if (pin) f.phase[i] = pin[b0 + i];
      if (pout) e.phase[i] = pout[b0 + i];
      e.alpha[i] = (float)alpha[b0 + i];
    }
    DLX_HIP(launch_fold_stage1(f, FOLD_FIELD, split, s));
    DLX_HIP(launch_fold_stage2(e, FOLD_STORE, split, s));
  }
  return h.release();
}

// Workspace of the VJP for one chunk of c wavelengths: the tables of both
// directions (used when the cache is bypassed), the stage-1 intermediate of
// either direction, Ebar, and the per-wavelength gradient planes.
struct VjpLayout {
  size_t T, U, Eb, H, P, total;   // P: the folded pupil, where the loader does not form it
};
VjpLayout vjp_layout(const dlx_mft_geom& g, int c) {
  VjpLayout L;
  L.T = align_up((size_t)c * (fold_table_bytes(g.n_in, g.n_out) + fold_table_bytes(g.n_out, g.n_in)));
  const long u = fold_mid_bytes(g.n_in, g.n_out), v = fold_mid_bytes(g.n_out, g.n_in);
  L.U = align_up((size_t)c * (u > v ? u : v));
  L.Eb = align_up((size_t)c * fold_field_bytes(g.n_out));
  L.H = align_up((size_t)c * g.n_in * g.n_in * sizeof(float));
  L.P = align_up((size_t)c * fold_field_bytes(g.n_in));
  L.total = L.T + L.U + L.Eb + 2 * L.H + L.P;
  return L;
}

}  // namespace
}  // namespace dlx

using namespace dlx;

extern "C" {

const char* dlx_version(void) { return "dlux_amd 0.1.0 gfx950"; }

const char* dlx_last_error(void) { return dlx::g_err.c_str(); }

int dlx_transfer_matrix(const dlx_mft_geom* geom, int32_t batch, const double* wavelength,
                        const double* pixel_scale_in, const double* pixel_scale_out,
                        const double* shift, void* out, void* stream) {
  clear_error();
  if (int st = check_geom(geom)) return st;
  DLX_CHECK_ARG(batch >= 0, "batch must be >= 0");
  if (batch == 0) return DLX_OK;
  DLX_CHECK_ARG(wavelength && pixel_scale_in && pixel_scale_out && out,
                "null argument to dlx_transfer_matrix");
  const dlx_mft_geom& g = *geom;
  const long stride = (long)g.n_out * g.n_in;
  for (int b0 = 0; b0 < batch; b0 += DftChunk::kMax) {
    const int n = batch - b0 < DftChunk::kMax ? batch - b0 : DftChunk::kMax;
    DftChunk c;
    for (int i = 0; i < n; ++i) {
      const int b = b0 + i;
      DLX_CHECK_ARG(std::isfinite(wavelength[b]) && wavelength[b] > 0,
                    "wavelength[%d] must be > 0", b);
      DLX_CHECK_ARG(std::isfinite(pixel_scale_in[b]) && pixel_scale_in[b] != 0,
                    "pixel_scale_in[%d] must be non-zero", b);
      DLX_CHECK_ARG(std::isfinite(pixel_scale_out[b]), "pixel_scale_out[%d] must be finite", b);
      const MftInst p = make_inst(g, wavelength[b], pixel_scale_in[b], pixel_scale_out[b],
                                  shift ? shift[b] : 0.0);
      c.a_scale[i] = p.a_scale;
      c.a_off[i] = p.a_off;
      c.b_scale[i] = p.b_scale;
      c.b_off[i] = p.b_off;
    }
    DLX_HIP(launch_dft_chunk(c, n, g.n_in, g.n_out, g.inverse, (float2*)out + (long)b0 * stride,
                             stride, (hipStream_t)stream));
  }
  return DLX_OK;
}

size_t dlx_mft_workspace_size(const dlx_mft_geom* geom, int32_t batch, int32_t precision) {
  if (!geom || batch <= 0) return 0;
  const bool split = precision == DLX_PREC_BF16X3;
  const size_t mat = align_up((size_t)batch * mat_bytes(geom->n_out, geom->n_in, split));
  // three complex matrices per instance (and a converted field), which the
  // folded tables and intermediate fit in on all but the smallest grids
  size_t total = 3 * mat;
  if (split) total += align_up((size_t)batch * mat_bytes(geom->n_in, geom->n_in, true));
  const size_t fold = field_transform_bytes(geom->n_in, geom->n_out, batch);
  return total > fold ? total : fold;
}

int dlx_mft(const dlx_mft_geom* geom, int32_t batch, const void* in, void* out,
            const double* wavelength, const double* pixel_scale_in,
            const double* pixel_scale_out, const double* shift_x, const double* shift_y,
            const double* field_scale, int32_t precision, void* workspace,
            size_t workspace_bytes, void* stream) {
  clear_error();
  if (int st = check_geom(geom)) return st;
  DLX_CHECK_ARG(batch >= 0, "batch must be >= 0");
  if (batch == 0) return DLX_OK;
  DLX_CHECK_ARG(in && out && wavelength && pixel_scale_in && pixel_scale_out,
                "null argument to dlx_mft");
  DLX_CHECK_ARG(precision == DLX_PREC_FP32 || precision == DLX_PREC_BF16X3,
                "unknown precision %d", precision);
  const size_t need = dlx_mft_workspace_size(geom, batch, precision);
  if (!workspace || workspace_bytes < need) {
    set_error("dlx_mft workspace too small: need %zu bytes, got %zu", need, workspace_bytes);
    return DLX_ERR_WORKSPACE;
  }
  const dlx_mft_geom& g = *geom;
  hipStream_t s = (hipStream_t)stream;
  // Per axis W = exp(-2 pi i s a_k b_l) with a_k = (u_k - sh) / N and
  // b_l = (u_l - sh) b: the product splits into the centred kernel and the
  // phases step sh u_k on the input and step (sh u_l - sh^2) on the output,
  // step = b / N; the tables depend on neither shift nor scale.
  std::vector<double> steps(batch), c(batch);
  std::vector<FoldPhase> pin(batch), pout(batch);
  const double sg = g.inverse ? -1.0 : 1.0;
  bool shifted = false;
  for (int b = 0; b < batch; ++b) {
    DLX_CHECK_ARG(std::isfinite(wavelength[b]) && wavelength[b] > 0, "wavelength[%d] must be > 0",
                  b);
    DLX_CHECK_ARG(std::isfinite(pixel_scale_in[b]) && pixel_scale_in[b] != 0,
                  "pixel_scale_in[%d] must be non-zero", b);
    DLX_CHECK_ARG(std::isfinite(pixel_scale_out[b]), "pixel_scale_out[%d] must be finite", b);
    const double st = fold_step(g, wavelength[b], pixel_scale_in[b], pixel_scale_out[b]);
    const double sx = shift_x ? shift_x[b] : 0.0, sy = shift_y ? shift_y[b] : 0.0;
    steps[b] = st;
    pin[b] = {0.0, sg * st * sx, sg * st * sy, 0.0};
    pout[b] = {0.0, sg * st * sx, sg * st * sy, -sg * st * (sx * sx + sy * sy)};
    shifted = shifted || sx != 0.0 || sy != 0.0;
    c[b] = mft_norm(g, wavelength[b], pixel_scale_in[b], pixel_scale_out[b]) *
           (field_scale ? field_scale[b] : 1.0);
  }
  return field_transform(g.n_in, g.n_out, batch, g.inverse != 0, steps, TABLES_FIELD,
                         shifted ? pin.data() : nullptr, shifted ? pout.data() : nullptr, c.data(),
                         in, out, precision == DLX_PREC_BF16X3, (uint8_t*)workspace, s);
}

size_t dlx_lct_workspace_size(int32_t n_in, int32_t n_out, int32_t batch, int32_t precision) {
  if (n_in <= 0 || n_out <= 0 || batch <= 0) return 0;
  const bool split = precision == DLX_PREC_BF16X3;
  size_t total = 2 * align_up((size_t)batch * mat_bytes(n_out, n_in, split));
  const size_t fold = field_transform_bytes(n_in, n_out, batch);
  if (fold > total) total = fold;
  if (split) total += align_up((size_t)batch * mat_bytes(n_in, n_in, true));
  return total;
}

int dlx_lct(int32_t n_in, int32_t n_out, int32_t batch, const double* abcd,
            const double* wavelength, double pixel_scale_in, double center_in,
            double pixel_scale_out, double center_out, const void* in, void* out,
            int32_t precision, void* workspace, size_t workspace_bytes, void* stream) {
  clear_error();
  DLX_CHECK_ARG(n_in > 0 && n_in <= 16384 && n_out > 0 && n_out <= 16384,
                "n_in and n_out must be in [1, 16384], got %d and %d", n_in, n_out);
  DLX_CHECK_ARG(batch >= 0 && batch <= 65535, "batch must be in [0, 65535], got %d", batch);
  if (batch == 0) return DLX_OK;
  DLX_CHECK_ARG(abcd && wavelength && in && out, "null argument to dlx_lct");
  DLX_CHECK_ARG(precision == DLX_PREC_FP32 || precision == DLX_PREC_BF16X3,
                "unknown precision %d", precision);
  const double A = abcd[0], B = abcd[1], D = abcd[3];
  DLX_CHECK_ARG(std::isfinite(A) && std::isfinite(D) && std::isfinite(B) && B != 0.0,
                "the ABCD matrix needs finite A and D and a finite, non-zero B");
  DLX_CHECK_ARG(std::isfinite(pixel_scale_in) && pixel_scale_in > 0 &&
                    std::isfinite(pixel_scale_out) && pixel_scale_out > 0,
                "pixel scales must be > 0");
  DLX_CHECK_ARG(std::isfinite(center_in) && std::isfinite(center_out), "centres must be finite");
  for (int b = 0; b < batch; ++b)
    DLX_CHECK_ARG(std::isfinite(wavelength[b]) && wavelength[b] > 0,
                  "wavelength[%d] must be > 0", b);
  const size_t need = dlx_lct_workspace_size(n_in, n_out, batch, precision);
  if (!workspace || workspace_bytes < need) {
    set_error("dlx_lct workspace too small: need %zu bytes, got %zu", need, workspace_bytes);
    return DLX_ERR_WORKSPACE;
  }
  hipStream_t s = (hipStream_t)stream;
  // Per axis the Collins kernel exp(2 pi i (A x^2 - 2 x x' + D x'^2) / (2 lambda B)
  // -+ i pi / 4), x = xc + u dx, x' = xc' + v dx', is the centred kernel of
  // step dx dx' / (lambda |B|) between the chirps of u and of v.
  const double xc = center_in, xo = center_out, dx = pixel_scale_in, dxo = pixel_scale_out;
  std::vector<double> steps(batch), alpha(batch);
  std::vector<FoldPhase> pin(batch), pout(batch);
  for (int b = 0; b < batch; ++b) {
    const double lb = wavelength[b] * B;
    steps[b] = dx * dxo / std::fabs(lb);
    alpha[b] = dx * dxo / (wavelength[b] * std::fabs(B));
    const double li = (A * xc - xo) / lb * dx, lo = (D * xo - xc) / lb * dxo;
    pin[b] = {A * dx * dx / (2.0 * lb), li, li, 0.0};
    // the constants of both axes: chirps at the centres, the cross term, 1 / (i B)
    pout[b] = {D * dxo * dxo / (2.0 * lb), lo, lo,
               2.0 * ((A * xc * xc - 2.0 * xc * xo + D * xo * xo) / (2.0 * lb)) +
                   (B > 0 ? -0.25 : 0.25)};
  }
  return field_transform(n_in, n_out, batch, B < 0, steps, TABLES_LCT, pin.data(), pout.data(),
                         alpha.data(), in, out, precision == DLX_PREC_BF16X3, (uint8_t*)workspace,
                         s);
}

size_t dlx_lct_fft_workspace_size(int32_t n, int32_t m, int32_t batch) {
  if (n <= 0 || m <= 0 || batch <= 0) return 0;
  return align_up((size_t)batch * n * n * sizeof(float2)) + dlx_fft2_workspace_size(n, m, batch);
}

int dlx_lct_fft(int32_t n, int32_t m, int32_t batch, const double* abcd,
                const double* wavelength, double pixel_scale_in, double center_in,
                double center_out, const void* in, void* out, double* pixel_scale_out,
                void* workspace, size_t workspace_bytes, void* stream) {
  clear_error();
  DLX_CHECK_ARG(n > 0 && m >= n && ((m - n) % 2) == 0,
                "need 0 < n <= m with m - n even, got n = %d, m = %d", n, m);
  DLX_CHECK_ARG(batch >= 0 && batch <= 65535, "batch must be in [0, 65535], got %d", batch);
  if (batch == 0) return DLX_OK;
  DLX_CHECK_ARG(abcd && wavelength && in && out, "null argument to dlx_lct_fft");
  const double A = abcd[0], B = abcd[1], D = abcd[3];
  DLX_CHECK_ARG(std::isfinite(A) && std::isfinite(D) && std::isfinite(B) && B != 0.0,
                "the ABCD matrix needs finite A and D and a finite, non-zero B");
  DLX_CHECK_ARG(std::isfinite(pixel_scale_in) && pixel_scale_in > 0, "pixel_scale_in must be > 0");
  DLX_CHECK_ARG(std::isfinite(center_in) && std::isfinite(center_out), "centres must be finite");
  for (int b = 0; b < batch; ++b)
    DLX_CHECK_ARG(std::isfinite(wavelength[b]) && wavelength[b] > 0,
                  "wavelength[%d] must be > 0", b);
  const size_t need = dlx_lct_fft_workspace_size(n, m, batch);
  if (!workspace || workspace_bytes < need) {
    set_error("dlx_lct_fft workspace too small: need %zu bytes, got %zu", need,
              workspace_bytes);
    return DLX_ERR_WORKSPACE;
  }
  hipStream_t s = (hipStream_t)stream;
  const double sg = B > 0 ? 1.0 : -1.0, dx = pixel_scale_in, M = m;
  // the centred FFT pairs offsets from index m / 2; the grids are symmetric
  // about (m - 1) / 2, de apart
  const double de = (m / 2) - (m - 1) / 2.0;
  float2* C1 = (float2*)workspace;
  uint8_t* fws = (uint8_t*)workspace + align_up((size_t)batch * n * n * sizeof(float2));
  const long nn = (long)n * n, mm = (long)m * m;
  // input chirp (A term), with the linear terms that centre the output on center_out
  for (int b0 = 0; b0 < batch; b0 += LctChirpChunk::kMax) {
    const int nb = batch - b0 < LctChirpChunk::kMax ? batch - b0 : LctChirpChunk::kMax;
    LctChirpChunk c;
    for (int i = 0; i < nb; ++i) {
      const double lb = wavelength[b0 + i] * B;
      c.q2[i] = A / (2.0 * lb);
      c.q1[i] = -center_out / lb - sg * de / (M * dx);
      c.q0[i] = center_out * center_in / lb + sg * de * center_in / (M * dx) + sg * de * de / M;
      c.x0[i] = center_in - (n - 1) / 2.0 * dx;
      c.dx[i] = dx;
    }
    DLX_HIP(launch_lct_chirp(c, nb, n, (const float2*)in + (long)b0 * nn, C1 + (long)b0 * nn,
                             s));
  }
  if (int st = dlx_fft2(n, m, batch, sg < 0, C1, out, fws, dlx_fft2_workspace_size(n, m, batch),
                        stream))
    return st;
  // output chirp (D term), the output-side linear terms and the constant phase
  for (int b0 = 0; b0 < batch; b0 += LctChirpChunk::kMax) {
    const int nb = batch - b0 < LctChirpChunk::kMax ? batch - b0 : LctChirpChunk::kMax;
    LctChirpChunk c;
    for (int i = 0; i < nb; ++i) {
      const double lb = wavelength[b0 + i] * B;
      const double d_out = wavelength[b0 + i] * std::fabs(B) / (M * dx);
      if (pixel_scale_out) pixel_scale_out[b0 + i] = d_out;
      c.q2[i] = D / (2.0 * lb);
      c.q1[i] = -center_in / lb - sg * de / (M * d_out);
      c.q0[i] = sg * de * center_out / (M * d_out) - sg / 8.0;
      c.x0[i] = center_out - (m - 1) / 2.0 * d_out;
      c.dx[i] = d_out;
    }
    DLX_HIP(launch_lct_chirp(c, nb, m, (const float2*)out + (long)b0 * mm,
                             (float2*)out + (long)b0 * mm, s));
  }
  return DLX_OK;
}

int dlx_pupil_field(int32_t n, int32_t batch, const double* wavelength, double pixel_scale,
                    double center, double tilt_x, double tilt_y, const float* amp,
                    const float* opd, const float* phase, double scale, const void* in,
                    void* out, void* stream) {
  clear_error();
  DLX_CHECK_ARG(n > 0, "n must be > 0");
  DLX_CHECK_ARG(batch >= 0, "batch must be >= 0");
  if (batch == 0) return DLX_OK;
  DLX_CHECK_ARG(wavelength && out, "null argument to dlx_pupil_field");
  DLX_CHECK_ARG(std::isfinite(pixel_scale) && std::isfinite(center) && std::isfinite(tilt_x) &&
                    std::isfinite(tilt_y) && std::isfinite(scale),
                "non-finite scalar argument to dlx_pupil_field");
  hipStream_t s = (hipStream_t)stream;
  const long npix = (long)n * n;
  const double x0 = center - (n - 1) / 2.0 * pixel_scale;
  for (int b0 = 0; b0 < batch; b0 += PupilChunk::kMax) {
    const int nb = batch - b0 < PupilChunk::kMax ? batch - b0 : PupilChunk::kMax;
    PupilChunk c;
    for (int i = 0; i < nb; ++i) {
      DLX_CHECK_ARG(std::isfinite(wavelength[b0 + i]) && wavelength[b0 + i] > 0,
                    "wavelength[%d] must be > 0", b0 + i);
      c.inv_wl[i] = 1.0 / wavelength[b0 + i];
    }
    DLX_HIP(launch_pupil_chunk(c, nb, n, pixel_scale, x0, tilt_x, tilt_y, amp, opd, phase,
                               (float)scale, in ? (const float2*)in + b0 * npix : nullptr,
                               (float2*)out + b0 * npix, s));
  }
  return DLX_OK;
}

int dlx_eval_basis(int32_t nbasis, int64_t npix, int32_t nsets, const float* basis,
                   const float* coeffs, const float* base, float* out, void* stream) {
  clear_error();
  DLX_CHECK_ARG(nbasis >= 0 && npix >= 0 && nsets >= 0, "negative size to dlx_eval_basis");
  if (npix == 0 || nsets == 0) return DLX_OK;
  DLX_CHECK_ARG(out && (nbasis == 0 || (basis && coeffs)), "null argument to dlx_eval_basis");
  DLX_HIP(launch_eval_basis(nbasis, npix, nsets, basis, coeffs, base, out,
                            (hipStream_t)stream));
  return DLX_OK;
}

int dlx_power(int64_t npix, int32_t batch, const void* field, float* out, void* stream) {
  clear_error();
  DLX_CHECK_ARG(npix >= 0 && batch >= 0, "negative size to dlx_power");
  if (batch == 0) return DLX_OK;
  DLX_CHECK_ARG(field && out, "null argument to dlx_power");
  DLX_HIP(launch_power(npix, batch, (const float2*)field, out, (hipStream_t)stream));
  return DLX_OK;
}

int dlx_intensity(int64_t npix, int32_t batch, const void* field, int32_t sum_over_batch,
                  float* out, void* stream) {
  clear_error();
  DLX_CHECK_ARG(npix >= 0 && batch >= 0, "negative size to dlx_intensity");
  if (batch == 0 || npix == 0) return DLX_OK;
  DLX_CHECK_ARG(field && out, "null argument to dlx_intensity");
  DLX_HIP(launch_intensity(npix, batch, (const float2*)field, sum_over_batch, out,
                           (hipStream_t)stream));
  return DLX_OK;
}

}  // extern "C"

namespace dlx {
namespace {

int check_psf_poly_args(const dlx_mft_geom* geom, int32_t nwl, const double* wavelength,
                        const double* weight, double pixel_scale_in, double pixel_scale_out,
                        double center, double tilt_x, double tilt_y, double scale, float* psf,
                        int32_t precision) {
  if (int st = check_geom(geom)) return st;
  DLX_CHECK_ARG(nwl > 0, "nwl must be > 0, got %d", nwl);
  DLX_CHECK_ARG(wavelength && weight && psf, "null argument to dlx_psf_poly");
  DLX_CHECK_ARG(precision == DLX_PREC_FP32 || precision == DLX_PREC_BF16X3,
                "unknown precision %d", precision);
  DLX_CHECK_ARG(std::isfinite(pixel_scale_in) && pixel_scale_in != 0.0 &&
                    std::isfinite(pixel_scale_out) && std::isfinite(center) &&
                    std::isfinite(tilt_x) && std::isfinite(tilt_y) && std::isfinite(scale),
                "non-finite scalar argument to dlx_psf_poly");
  for (int l = 0; l < nwl; ++l) {
    DLX_CHECK_ARG(std::isfinite(weight[l]) && weight[l] >= 0, "weight[%d] must be >= 0", l);
    DLX_CHECK_ARG(std::isfinite(wavelength[l]) && wavelength[l] > 0,
                  "wavelength[%d] must be > 0", l);
  }
  return DLX_OK;
}

// The psf chain over chunks of at most c wavelengths in `ws` (psf_poly_bytes(c)
// bytes): tables (from the device cache when `use_cache`, else generated into
// ws), the two folded contractions with the |E|^2 epilogue, and the running
// sum over wavelengths in wavelength order (so the result does not depend on
// c).  With `planes` set, every wavelength's w_l |E_l|^2 plane is written there
// instead (planes + l N_out^2) and nothing is summed.  `prof` records the
// contractions' live timing.
int psf_poly_run(const dlx_mft_geom& g, int32_t nwl, const double* wavelength,
                 const double* weight, double pixel_scale_in, double pixel_scale_out,
                 double center, double tilt_x, double tilt_y, const float* amp,
                 const float* opd, const float* phase, double scale, float* psf, bool split,
                 uint8_t* ws, int c, bool use_cache, bool prof, hipStream_t s,
                 float* planes = nullptr) {
  const PsfLayout L = psf_layout(g, c);
  uint8_t* T_ws = ws;
  uint8_t* U = T_ws + L.T;
  float* I = (float*)(U + L.U);
  uint8_t* P = (uint8_t*)I + L.I;
  const bool room = L.total + L.P <= psf_poly_bytes(g, c, split);
  const long nout2 = (long)g.n_out * g.n_out;
  FoldStage1 f1{};
  f1.n = g.n_in;
  f1.m = g.n_out;
  f1.out = U;
  f1.out_stride = fold_mid_bytes(g.n_in, g.n_out);
  f1.pupil = {opd, amp, phase, pixel_scale_in, center - (g.n_in - 1) / 2.0 * pixel_scale_in, tilt_x,
              tilt_y, (float)scale};
  // the pupil formed in stage 1's loader (no pupil array in HBM), or written
  // first where many column tiles would each form it again
  const bool in_loader =
      !room || (pupil_prologue_enabled() && fold_pupil_in_loader(f1.pupil, g.n_in, g.n_out));
  for (int l0 = 0; l0 < nwl; l0 += c) {
    const int nb = nwl - l0 < c ? nwl - l0 : c;
    // one wavelength is its own sum
    float* Ic = planes ? planes + (long)l0 * nout2 : nwl == 1 ? psf : I;
    CacheLease h(s);
    FoldTables tab;
    if (int st = fold_tables(g.n_in, g.n_out,
                             psf_steps(g, nb, wavelength + l0, pixel_scale_in, pixel_scale_out),
                             split, false, TABLES_PSF, use_cache, T_ws, s, &tab, &h))
      return st;
    f1.batch = nb;
    f1.table = tab.fwd;
    f1.table_stride = tab.stride;
    for (int i = 0; i < nb; ++i) f1.inv_wl[i] = 1.0 / wavelength[l0 + i];
    if (!in_loader) {
      f1.src = P;
      f1.src_stride = fold_field_bytes(g.n_in);
      DLX_HIP(launch_fold_pupil(f1.pupil, f1.inv_wl, nb, g.n_in, split, P, f1.src_stride, s));
    }
    int slot = -1;
    if (prof) { if (int st = prof_begin(1, s, &slot)) return st; }
    DLX_HIP(launch_fold_stage1(f1, in_loader ? FOLD_PUPIL : FOLD_MEM, split, s));
    if (prof) { if (int st = prof_end(slot, s)) return st; }
    // |E_l|^2 = (c_l sqrt(w_l))^2 |W_y P W_x^T|^2: the scale is applied in the
    // stage-2 epilogue, so the tables depend on the geometry only.
    FoldStage2 f2{};
    f2.n = g.n_in;
    f2.m = g.n_out;
    f2.batch = nb;
    f2.inverse = g.inverse;
    f2.table = tab.fwd;
    f2.table_stride = tab.stride;
    f2.mid = U;
    f2.mid_stride = f1.out_stride;
    f2.out = Ic;
    f2.out_stride = nout2;
    for (int i = 0; i < nb; ++i)
      f2.alpha[i] = (float)(mft_norm(g, wavelength[l0 + i], pixel_scale_in, pixel_scale_out) *
                            std::sqrt(weight[l0 + i]));
    if (prof) { if (int st = prof_begin(2, s, &slot)) return st; }
    DLX_HIP(launch_fold_stage2(f2, FOLD_INTENSITY, split, s));
    if (prof) { if (int st = prof_end(slot, s)) return st; }
    if (int st = h.release()) return st;
    if (!planes && nwl > 1) DLX_HIP(launch_sum_planes(nout2, nb, I, l0 > 0, psf, s));
  }
  return DLX_OK;
}

}  // namespace
}  // namespace dlx

extern "C" {

size_t dlx_psf_poly_workspace_size(const dlx_mft_geom* geom, int32_t nwl, int32_t precision) {
  if (!geom || nwl <= 0) return 0;
  return psf_poly_bytes(*geom, nwl < kWlChunk ? nwl : kWlChunk, precision == DLX_PREC_BF16X3);
}

int dlx_psf_poly(const dlx_mft_geom* geom, int32_t nwl, const double* wavelength,
                 const double* weight, double pixel_scale_in, double pixel_scale_out,
                 double center, double tilt_x, double tilt_y, const float* amp,
                 const float* opd, const float* phase, double scale, float* psf,
                 int32_t precision, void* workspace, size_t workspace_bytes, void* stream) {
  clear_error();
  if (int st = check_psf_poly_args(geom, nwl, wavelength, weight, pixel_scale_in,
                                   pixel_scale_out, center, tilt_x, tilt_y, scale, psf,
                                   precision))
    return st;
  const size_t need = dlx_psf_poly_workspace_size(geom, nwl, precision);
  if (!workspace || workspace_bytes < need) {
    set_error("dlx_psf_poly workspace too small: need %zu bytes, got %zu", need,
              workspace_bytes);
    return DLX_ERR_WORKSPACE;
  }
  return psf_poly_run(*geom, nwl, wavelength, weight, pixel_scale_in, pixel_scale_out, center,
                      tilt_x, tilt_y, amp, opd, phase, scale, psf,
                      precision == DLX_PREC_BF16X3, (uint8_t*)workspace,
                      nwl < kWlChunk ? nwl : kWlChunk, true, true, (hipStream_t)stream);
}

size_t dlx_psf_poly_detector_workspace_size(const dlx_mft_geom* geom, int32_t nwl,
                                            int32_t precision, const dlx_detector_op* ops,
                                            int32_t nops) {
  if (!geom || nwl <= 0) return 0;
  const int c = nwl < kWlChunk ? nwl : kWlChunk;
  const size_t planes = align_up((size_t)nwl * geom->n_out * geom->n_out * sizeof(float));
  return psf_poly_bytes(*geom, c, precision == DLX_PREC_BF16X3) + planes +
         detector_ws_bytes(geom->n_out, 1, ops, nops, nwl);
}

int dlx_psf_poly_detector(const dlx_mft_geom* geom, int32_t nwl, const double* wavelength,
                          const double* weight, double pixel_scale_in, double pixel_scale_out,
                          double center, double tilt_x, double tilt_y, const float* amp,
                          const float* opd, const float* phase, double scale,
                          const dlx_detector_op* ops, int32_t nops, float* out,
                          int32_t precision, void* workspace, size_t workspace_bytes,
                          void* stream) {
  clear_error();
  if (int st = check_psf_poly_args(geom, nwl, wavelength, weight, pixel_scale_in,
                                   pixel_scale_out, center, tilt_x, tilt_y, scale, out,
                                   precision))
    return st;
  int32_t side = 0;
  if (int st = dlx_detector_out_side(geom->n_out, ops, nops, &side)) return st;
  const size_t need = dlx_psf_poly_detector_workspace_size(geom, nwl, precision, ops, nops);
  if (!workspace || workspace_bytes < need) {
    set_error("dlx_psf_poly_detector workspace too small: need %zu bytes, got %zu", need,
              workspace_bytes);
    return DLX_ERR_WORKSPACE;
  }
  const bool split = precision == DLX_PREC_BF16X3;
  const int c = nwl < kWlChunk ? nwl : kWlChunk;
  uint8_t* ws = (uint8_t*)workspace;
  const size_t chain = psf_poly_bytes(*geom, c, split);
  float* planes = (float*)(ws + chain);
  const size_t pbytes = align_up((size_t)nwl * geom->n_out * geom->n_out * sizeof(float));
  hipStream_t s = (hipStream_t)stream;
  // every wavelength's w_l |E_l|^2 plane, then the detector chain whose first
  // pass loads the sum over the planes (in wavelength order: the PSF that
  // dlx_psf_poly returns, never written)
  if (int st = psf_poly_run(*geom, nwl, wavelength, weight, pixel_scale_in, pixel_scale_out,
                            center, tilt_x, tilt_y, amp, opd, phase, scale, nullptr, split, ws,
                            c, true, true, s, planes))
    return st;
  return detector_apply_sum(geom->n_out, 1, nwl, (long)geom->n_out * geom->n_out, planes, ops,
                            nops, out, ws + chain + pbytes, workspace_bytes - chain - pbytes, s);
}

size_t dlx_psf_poly_vjp_workspace_size(const dlx_mft_geom* geom, int32_t nwl,
                                       int32_t precision) {
  if (!geom || nwl <= 0) return 0;
  const int c = nwl < kWlChunk ? nwl : kWlChunk;
  // more than the PSF's own workspace: one buffer serves a step's forward and
  // backward calls
  const size_t psf = psf_poly_bytes(*geom, c, precision == DLX_PREC_BF16X3);
  const VjpLayout L = vjp_layout(*geom, c);
  return (L.total > psf ? L.total : psf) + 256;
}

int dlx_psf_poly_vjp(const dlx_mft_geom* geom, int32_t nwl, const double* wavelength,
                     const double* weight, double pixel_scale_in, double pixel_scale_out,
                     double center, double tilt_x, double tilt_y, const float* amp,
                     const float* opd, const float* phase, double scale, const float* dpsf,
                     float* grad_opd, float* grad_phase, float* grad_amp, int32_t precision,
                     void* workspace, size_t workspace_bytes, void* stream) {
  clear_error();
  if (int st = check_geom(geom)) return st;
  DLX_CHECK_ARG(nwl > 0, "nwl must be > 0, got %d", nwl);
  DLX_CHECK_ARG(wavelength && weight && dpsf, "null argument to dlx_psf_poly_vjp");
  DLX_CHECK_ARG(grad_opd || grad_phase || grad_amp,
                "dlx_psf_poly_vjp needs grad_opd, grad_phase or grad_amp");
  DLX_CHECK_ARG(precision == DLX_PREC_FP32 || precision == DLX_PREC_BF16X3,
                "unknown precision %d", precision);
  DLX_CHECK_ARG(std::isfinite(pixel_scale_in) && pixel_scale_in != 0.0 &&
                    std::isfinite(pixel_scale_out) && std::isfinite(center) &&
                    std::isfinite(tilt_x) && std::isfinite(tilt_y) && std::isfinite(scale),
                "non-finite scalar argument to dlx_psf_poly_vjp");
  const size_t need = dlx_psf_poly_vjp_workspace_size(geom, nwl, precision);
  if (!workspace || workspace_bytes < need) {
    set_error("dlx_psf_poly_vjp workspace too small: need %zu bytes, got %zu", need,
              workspace_bytes);
    return DLX_ERR_WORKSPACE;
  }
  for (int l = 0; l < nwl; ++l) {
    DLX_CHECK_ARG(std::isfinite(weight[l]) && weight[l] >= 0, "weight[%d] must be >= 0", l);
    DLX_CHECK_ARG(std::isfinite(wavelength[l]) && wavelength[l] > 0,
                  "wavelength[%d] must be > 0", l);
  }
  const dlx_mft_geom& g = *geom;
  hipStream_t s = (hipStream_t)stream;
  const bool split = precision == DLX_PREC_BF16X3;
  const int c = nwl < kWlChunk ? nwl : kWlChunk;
  const VjpLayout L = vjp_layout(g, c);
  uint8_t* T_ws = (uint8_t*)workspace;
  uint8_t* U = T_ws + L.T;
  uint8_t* Eb = U + L.U;
  float* H = (float*)(Eb + L.Eb);
  float* H2 = grad_amp ? (float*)((uint8_t*)H + L.H) : nullptr;
  uint8_t* P = (uint8_t*)H + 2 * L.H;
  const long nin = g.n_in;
  const FoldPupil pup = {opd, amp, phase, pixel_scale_in,
                         center - (g.n_in - 1) / 2.0 * pixel_scale_in, tilt_x, tilt_y, (float)scale};
  for (int l0 = 0; l0 < nwl; l0 += c) {
    const int nb = nwl - l0 < c ? nwl - l0 : c;
    GradChunk gc;
    CacheLease h(s);
    FoldTables tab;
    if (int st = fold_tables(g.n_in, g.n_out,
                             psf_steps(g, nb, wavelength + l0, pixel_scale_in, pixel_scale_out),
                             split, true, TABLES_PSF, true, T_ws, s, &tab, &h))
      return st;
    FoldStage2 e{}, b{};
    for (int i = 0; i < nb; ++i) {
      e.alpha[i] = b.alpha[i] =
          (float)(mft_norm(g, wavelength[l0 + i], pixel_scale_in, pixel_scale_out) *
                  std::sqrt(weight[l0 + i]));
      gc.kw[i] = (float)(2.0 * M_PI / wavelength[l0 + i]);
      b.inv_wl[i] = 1.0 / wavelength[l0 + i];
    }
    // forward: the pupil through stage 1, then Ebar = 2 G E folded for the way back
    FoldStage1 f{};
    f.n = g.n_in; f.m = g.n_out; f.batch = nb;
    f.table = tab.fwd; f.table_stride = tab.stride;
    f.out = U; f.out_stride = fold_mid_bytes(g.n_in, g.n_out);
    f.pupil = pup;
    for (int i = 0; i < nb; ++i) f.inv_wl[i] = b.inv_wl[i];
    const bool in_loader = fold_pupil_in_loader(pup, g.n_in, g.n_out);
    if (!in_loader) {
      f.src = P;
      f.src_stride = fold_field_bytes(g.n_in);
      DLX_HIP(launch_fold_pupil(pup, f.inv_wl, nb, g.n_in, split, P, f.src_stride, s));
    }
    DLX_HIP(launch_fold_stage1(f, in_loader ? FOLD_PUPIL : FOLD_MEM, split, s));
    e.n = g.n_in; e.m = g.n_out; e.batch = nb; e.inverse = g.inverse;
    e.table = tab.fwd; e.table_stride = tab.stride;
    e.mid = U; e.mid_stride = f.out_stride;
    e.out = Eb; e.out_stride = fold_field_bytes(g.n_out);
    e.G = dpsf;
    DLX_HIP(launch_fold_stage2(e, FOLD_VJP, split, s));
    // adjoint: the same transform with the sides exchanged and the sign
    // flipped; its epilogue multiplies by the pupil's phasor
    FoldStage1 v{};
    v.n = g.n_out; v.m = g.n_in; v.batch = nb;
    v.src = Eb; v.src_stride = e.out_stride;
    v.table = tab.adj; v.table_stride = tab.stride;
    v.out = U; v.out_stride = fold_mid_bytes(g.n_out, g.n_in);
    DLX_HIP(launch_fold_stage1(v, FOLD_MEM, split, s));
    b.n = g.n_out; b.m = g.n_in; b.batch = nb; b.inverse = !g.inverse;
    b.table = tab.adj; b.table_stride = tab.stride;
    b.mid = U; b.mid_stride = v.out_stride;
    b.out = H; b.out_stride = nin * nin; b.out2 = H2;
    b.pupil = pup;
    DLX_HIP(launch_fold_stage2(b, FOLD_GRAD, split, s));
    if (int st = h.release()) return st;
    if (grad_opd || grad_phase)
      DLX_HIP(launch_grad_reduce(gc, nb, nin * nin, H, l0 > 0, grad_opd, grad_phase, s));
    if (grad_amp)   // sum over wavelengths of Re(conj(U) Pbar) = dL/dA
      DLX_HIP(launch_grad_reduce(gc, nb, nin * nin, H2, l0 > 0, nullptr, grad_amp, s));
  }
  return DLX_OK;
}

size_t dlx_project_basis_workspace_size(int32_t nbasis, int64_t npix, int32_t nsets) {
  if (nbasis <= 0 || npix <= 0 || nsets <= 0) return 0;
  return align_up((size_t)nbasis * nsets * project_parts(npix) * sizeof(float));
}

int dlx_project_basis(int32_t nbasis, int64_t npix, int32_t nsets, const float* basis,
                      const float* grad, float* out, void* workspace, size_t workspace_bytes,
                      void* stream) {
  clear_error();
  DLX_CHECK_ARG(nbasis >= 0 && npix >= 0 && nsets >= 0, "negative size to dlx_project_basis");
  DLX_CHECK_ARG(nbasis <= 65535 && nsets <= 65535, "nbasis and nsets must be <= 65535");
  if (nbasis == 0 || nsets == 0) return DLX_OK;
  DLX_CHECK_ARG(basis && grad && out, "null argument to dlx_project_basis");
  hipStream_t s = (hipStream_t)stream;
  const size_t need = dlx_project_basis_workspace_size(nbasis, npix, nsets);
  if (need && (!workspace || workspace_bytes < need)) {
    set_error("dlx_project_basis workspace too small: need %zu bytes, got %zu", need,
              workspace_bytes);
    return DLX_ERR_WORKSPACE;
  }
  DLX_HIP(launch_project_basis(nbasis, npix, nsets, basis, grad, (float*)workspace, out, s));
  return DLX_OK;
}

int dlx_profile_enable(int32_t enable) {
  clear_error();
  g_prof.enabled = enable ? 1 : 0;
  g_prof.n = 0;
  return DLX_OK;
}

int dlx_profile_read(int32_t stage, double* total_ms, int32_t* count) {
  clear_error();
  DLX_CHECK_ARG(total_ms && count, "null argument to dlx_profile_read");
  double t = 0.0;
  int c = 0;
  for (int i = 0; i < g_prof.n; ++i) {
    if (g_prof.slots[i].stage != stage) continue;
    DLX_HIP(hipEventSynchronize(g_prof.slots[i].end));
    float ms = 0.f;
    DLX_HIP(hipEventElapsedTime(&ms, g_prof.slots[i].beg, g_prof.slots[i].end));
    t += ms;
    ++c;
  }
  *total_ms = t;
  *count = c;
  return DLX_OK;
}

}  // extern "C"

// ---------------------------------------------------------------------------
// dlx_psf_poly_noalloc: the psf chain with every buffer in one fixed device
// array of the library, for callers that cannot allocate (code under graph
// capture, serving loops, harnesses that forbid hipMalloc).  The array is a
// file-scope __device__ symbol: each GPU the library runs on holds its own
// copy (allocated when the code object loads there, kept until the process
// ends).  Its device address is looked up once per device with
// hipGetSymbolAddress and only that address is handed to kernels; the array's
// name in host code is a host-side stand-in, not a device pointer.
// ---------------------------------------------------------------------------
namespace dlx {

constexpr size_t kNoallocScratchBytes = (size_t)64 << 20;   // 64 MiB per GPU
// Room beyond it for grids of a few pixels, whose folded buffers pad n to 64:
// with at most 64 MiB of plain buffers the output side is at most 4096, and the
// folded ones exceed them by less than 640 n_out + 8192 bytes.
constexpr size_t kNoallocSlack = (size_t)4 << 20;
static __device__ __align__(256) uint8_t scratch[kNoallocScratchBytes + kNoallocSlack];

namespace {

constexpr int kMaxScratchDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_dev[kMaxScratchDevices] = {};

// The current device's copy of `scratch` (looked up on its first use there).
int scratch_address(void** out) {
  *out = nullptr;
  int dev = 0;
  DLX_HIP(hipGetDevice(&dev));
  DLX_CHECK_ARG(dev >= 0 && dev < kMaxScratchDevices, "device %d beyond the %d supported", dev,
                kMaxScratchDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_dev[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr) {
      (void)hipGetLastError();
      set_error("hipGetSymbolAddress of the scratch array failed on device %d: %s", dev,
                hipGetErrorString(e));
      return DLX_ERR_HIP;
    }
    g_scratch_dev[dev] = p;
  }
  *out = g_scratch_dev[dev];
  return DLX_OK;
}

}  // namespace
}  // namespace dlx

extern "C" {

size_t dlx_psf_poly_noalloc_scratch_bytes(void) { return kNoallocScratchBytes; }

int dlx_psf_poly_noalloc(const dlx_mft_geom* geom, int32_t nwl, const double* wavelength,
                         const double* weight, double pixel_scale_in, double pixel_scale_out,
                         double center, double tilt_x, double tilt_y, const float* amp,
                         const float* opd, const float* phase, double scale, float* psf,
                         int32_t precision, void* stream) {
  clear_error();
  if (int st = check_psf_poly_args(geom, nwl, wavelength, weight, pixel_scale_in,
                                   pixel_scale_out, center, tilt_x, tilt_y, scale, psf,
                                   precision))
    return st;
  const bool split = precision == DLX_PREC_BF16X3;
  const size_t one = psf_plain_bytes(*geom, 1, split);
  if (one > kNoallocScratchBytes) {
    set_error("dlx_psf_poly_noalloc: one wavelength of a %d^2 -> %d^2 PSF needs %zu bytes, "
              "more than the %zu-byte scratch array; use dlx_psf_poly with a workspace",
              geom->n_in, geom->n_out, one, kNoallocScratchBytes);
    return DLX_ERR_INVALID;
  }
  // the largest chunk of wavelengths whose buffers fit the array
  int c = nwl < kWlChunk ? nwl : kWlChunk;
  while (c > 1 && psf_poly_bytes(*geom, c, split) > kNoallocScratchBytes) --c;
  void* ws = nullptr;
  if (int st = scratch_address(&ws)) return st;
  // tables are generated into the array every call: the device cache allocates
  return psf_poly_run(*geom, nwl, wavelength, weight, pixel_scale_in, pixel_scale_out, center,
                      tilt_x, tilt_y, amp, opd, phase, scale, psf, split, (uint8_t*)ws, c,
                      false, false, (hipStream_t)stream);
}

}  // extern "C"
