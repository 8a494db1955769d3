// Uneven batched MFT: many (field, wavelength, shift) instances of different
// pupil and output sizes, computed by grouped persistent launches (gfx950).
//
// One call of dlx_mft_batched_psf runs, whatever the mix of shapes:
//   1. one launch that generates the distinct cosine / sine tables (instances
//      of equal sides and phase step share one), and one that folds each
//      distinct complex64 field;
//   2. one grouped launch per tile width (output sides to 64, to 128, above)
//      of the folded stage 1, whose workgroups take several instances of one
//      field and apply each one's shift as a phase (dlx_fold.h);
//   3. one grouped launch of stage 2 with the |E|^2 epilogue,
//      I_i = |alpha_i W_y,i U_i|^2 (alpha_i = c_i sqrt(weight_i));
//   4. one launch that sums the planes of each output image, in a fixed order.
// Per-instance descriptors live in the caller's workspace; the host fills them
// in a pinned staging slot and copies them with the launches (stream-ordered).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <cstdlib>
#include <map>
#include <mutex>
#include <unordered_map>
#include <vector>

#include "dlx_fold.h"
#include "dlx_internal.h"

namespace dlx {
namespace {

struct SumJob {              // out[p] = sum_{q < count} planes[q * npix + p]
  float* out;
  const float* planes;
  long npix;
  int count, pad_;
};

// One pixel per lane (a wave reads 256 contiguous bytes of a plane), 16 planes
// in flight per lane before the in-order additions.
__global__ void __launch_bounds__(256)
group_sum_kernel(const SumJob* __restrict__ jobs) {
  const SumJob& j = jobs[blockIdx.y];
  for (long p = (long)blockIdx.x * blockDim.x + threadIdx.x; p < j.npix;
       p += (long)gridDim.x * blockDim.x) {
    float acc = 0.f;
    int q = 0;
    for (; q + 16 <= j.count; q += 16) {
      float v[16];
#pragma unroll
      for (int e = 0; e < 16; ++e) v[e] = j.planes[(long)(q + e) * j.npix + p];
#pragma unroll
      for (int e = 0; e < 16; ++e) acc += v[e];
    }
    for (; q < j.count; ++q) acc += j.planes[(long)q * j.npix + p];
    j.out[p] = acc;
  }
}

// ---------------------------------------------------------------------------
// pinned staging slots for descriptor uploads
// ---------------------------------------------------------------------------
struct Slot {
  void* host = nullptr;
  size_t cap = 0;
  hipEvent_t done = nullptr;
  bool used = false;
};

struct Staging {
  std::mutex mu;
  static constexpr int kSlots = 16;
  Slot slots[kSlots];
  int next = 0;
};

Staging& staging() {
  static Staging s;
  return s;
}

__global__ void __launch_bounds__(256)
upload_kernel(const uint4* __restrict__ src, uint4* __restrict__ dst, long n) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[i];
}

// Copy `bytes` (a multiple of 16) of host descriptors to device `dst` on stream
// s through a pinned slot, which a kernel reads over the bus: the descriptors of
// 768 instances hold the stream for 16 us, where hipMemcpyAsync took 27.  The
// slot is reused only after the copy that last used it ran.
int upload(const void* src, size_t bytes, void* dst, hipStream_t s) {
  if (bytes == 0) return DLX_OK;
  Staging& st = staging();
  std::lock_guard<std::mutex> lock(st.mu);
  Slot& sl = st.slots[st.next];
  st.next = (st.next + 1) % Staging::kSlots;
  if (sl.used) DLX_HIP(hipEventSynchronize(sl.done));
  if (sl.cap < bytes) {
    if (sl.host) DLX_HIP(hipHostFree(sl.host));
    sl.host = nullptr;
    sl.cap = 0;
    size_t cap = 1 << 16;
    while (cap < bytes) cap <<= 1;
    DLX_HIP(hipHostMalloc(&sl.host, cap, hipHostMallocMapped | hipHostMallocCoherent |
                                             hipHostMallocPortable));
    sl.cap = cap;
  }
  // the host writes a slot after its event, and reads nothing behind it
  if (!sl.done)
    DLX_HIP(hipEventCreateWithFlags(&sl.done, hipEventDisableTiming | hipEventDisableSystemFence));
  std::memcpy(sl.host, src, bytes);
  void* dev = nullptr;
  DLX_HIP(hipHostGetDevicePointer(&dev, sl.host, 0));
  const long n = (long)(bytes / 16);
  hipLaunchKernelGGL(upload_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s,
                     (const uint4*)dev, (uint4*)dst, n);
  DLX_HIP(hipGetLastError());
  DLX_HIP(hipEventRecord(sl.done, s));
  sl.used = true;
  return DLX_OK;
}

// ---------------------------------------------------------------------------
// planning
// ---------------------------------------------------------------------------
constexpr int kLists = 3;                   // stage-1 lists by tile width
constexpr int kWidth[kLists] = {32, 64, 128};
int list_of(int m) { return fold_group_width(m) == 128 ? 2 : fold_group_width(m) == 64 ? 1 : 0; }

struct Plan {
  // workspace offsets (bytes); descriptors first
  size_t off_tab, off_fld, off_prob, off_cols, off_map1[kLists], off_map2, off_sum, desc;
  size_t off_T, off_P, off_U, off_I, total;
  size_t tab_bytes = 0;
  std::vector<FoldTableJob> tab;
  std::vector<size_t> tab_off;       // of each distinct table, from off_T
  std::vector<int> tab_of;           // instance -> table
  int tab_most = 0;                  // threads of the largest table
  std::vector<FoldFieldJob> fld;     // distinct fields
  std::vector<size_t> fld_off;
  std::vector<int> fld_of;           // instance -> field
  int fld_most = 0;                  // side of the largest field
  std::vector<FoldProblem> prob;     // in launch order
  std::vector<FoldColumns> cols;
  std::vector<FoldRowTile> map1[kLists];
  std::vector<uint32_t> map2;
  int xcd1[kLists][9], xcd2[9];
  std::vector<SumJob> sum;
  std::vector<size_t> U_off, I_off;  // per instance
};

int validate(int n, const dlx_mft_instance* inst, int n_outputs) {
  DLX_CHECK_ARG(n >= 0, "n must be >= 0");
  DLX_CHECK_ARG(n == 0 || inst, "instances is NULL");
  DLX_CHECK_ARG(n_outputs >= 0 && n_outputs <= 65535, "n_outputs must be in [0, 65535]");
  for (int i = 0; i < n; ++i) {
    const dlx_mft_instance& d = inst[i];
    DLX_CHECK_ARG(d.n_in > 0 && d.n_in <= 16384 && d.n_out > 0 && d.n_out <= 16384,
                  "instance %d: n_in and n_out must be in [1, 16384]", i);
    DLX_CHECK_ARG(d.field != nullptr, "instance %d: field is NULL", i);
    DLX_CHECK_ARG(d.out_index >= 0 && d.out_index < n_outputs,
                  "instance %d: out_index %d outside [0, %d)", i, d.out_index, n_outputs);
    DLX_CHECK_ARG(std::isfinite(d.wavelength) && d.wavelength > 0,
                  "instance %d: wavelength must be > 0", i);
    DLX_CHECK_ARG(std::isfinite(d.pixel_scale_in) && d.pixel_scale_in != 0,
                  "instance %d: pixel_scale_in must be non-zero", i);
    DLX_CHECK_ARG(std::isfinite(d.pixel_scale_out), "instance %d: pixel_scale_out", i);
    DLX_CHECK_ARG(std::isfinite(d.shift_x) && std::isfinite(d.shift_y),
                  "instance %d: shifts must be finite", i);
    DLX_CHECK_ARG(std::isfinite(d.weight) && d.weight >= 0, "instance %d: weight must be >= 0",
                  i);
    if (d.has_focal)
      DLX_CHECK_ARG(std::isfinite(d.focal_length + d.focal_shift) &&
                        d.focal_length + d.focal_shift != 0.0,
                    "instance %d: focal_length + focal_shift must be finite and non-zero", i);
  }
  std::vector<int> nout(n_outputs, 0);
  for (int i = 0; i < n; ++i) {
    int& o = nout[inst[i].out_index];
    DLX_CHECK_ARG(o == 0 || o == inst[i].n_out,
                  "instances of output %d have different n_out (%d and %d)",
                  inst[i].out_index, o, inst[i].n_out);
    o = inst[i].n_out;
  }
  return DLX_OK;
}

dlx_mft_geom geom_of(const dlx_mft_instance& d) {
  dlx_mft_geom g{};
  g.n_in = d.n_in;
  g.n_out = d.n_out;
  g.inverse = d.inverse;
  g.has_focal = d.has_focal;
  g.focal_length = d.focal_length;
  g.focal_shift = d.focal_shift;
  return g;
}

struct TableKey {
  int n, m;
  double step;
  bool operator==(const TableKey& o) const {
    return n == o.n && m == o.m && std::memcmp(&step, &o.step, sizeof(double)) == 0;
  }
};
struct TableHash {
  size_t operator()(const TableKey& k) const {
    uint64_t b;
    std::memcpy(&b, &k.step, sizeof(b));
    b ^= ((uint64_t)(uint32_t)k.n << 32 | (uint32_t)k.m) * 0x9E3779B97F4A7C15ull;
    b *= 0xBF58476D1CE4E5B9ull;
    return (size_t)(b ^ (b >> 31));
  }
};

int rows1(int n) { return (fold_half(n) + kFoldTilePy - 1) / kFoldTilePy; }
int cols1(int m) { return (fold_half(m) + fold_group_width(m) - 1) / fold_group_width(m); }
int tiles2(int m) {
  const int mh = fold_half(m);
  return ((mh + kFoldTileQy - 1) / kFoldTileQy) * ((mh + kFoldTileQx - 1) / kFoldTileQx);
}

// Sizes and offsets of the batch's buffers.
int plan_sizes(int n, const dlx_mft_instance* inst, int n_outputs, Plan& P) {
  std::unordered_map<const void*, int> fields;
  size_t plain = 0;      // the unfolded layout's buffers: never asked for less
  size_t fbytes = 0;
  P.fld_of.resize(n);
  for (int i = 0; i < n; ++i) {
    const dlx_mft_instance& d = inst[i];
    if (i > 0 && d.field == inst[i - 1].field) {
      P.fld_of[i] = P.fld_of[i - 1];
    } else {
      auto it = fields.emplace(d.field, (int)P.fld.size());
      P.fld_of[i] = it.first->second;
      if (it.second) {
        P.fld.push_back({(const float2*)d.field, nullptr, d.n_in, 0});
        P.fld_off.push_back(fbytes);
        fbytes += align_up(fold_field_bytes(d.n_in));
        P.fld_most = std::max(P.fld_most, (int)d.n_in);
        plain += align_up(mat_bytes(d.n_in, d.n_in, true));
      }
    }
    if (P.fld[P.fld_of[i]].n != d.n_in) {
      set_error("instance %d: the same field pointer is used with n_in %d and %d", i,
                P.fld[P.fld_of[i]].n, d.n_in);
      return DLX_ERR_INVALID;
    }
  }
  // distinct tables
  std::unordered_map<TableKey, int, TableHash> tables;
  P.tab_of.resize(n);
  for (int i = 0; i < n; ++i) {
    const dlx_mft_instance& d = inst[i];
    const TableKey k = {d.n_in, d.n_out,
                        fold_step(geom_of(d), d.wavelength, d.pixel_scale_in, d.pixel_scale_out)};
    auto it = tables.emplace(k, (int)P.tab.size());
    if (it.second) {
      P.tab.push_back({nullptr, k.step, k.n, k.m});
      P.tab_off.push_back(P.tab_bytes);
      P.tab_bytes += fold_table_bytes(k.n, k.m);
      P.tab_most = std::max(P.tab_most, fold_group_table_threads(k.n, k.m));
    }
    P.tab_of[i] = it.first->second;
  }
  size_t off = 0;
  auto take = [&](size_t bytes) { const size_t o = off; off += align_up(bytes); return o; };
  P.off_tab = take(P.tab.size() * sizeof(FoldTableJob));
  P.off_fld = take(P.fld.size() * sizeof(FoldFieldJob));
  P.off_prob = take((size_t)n * sizeof(FoldProblem));
  // bounds: a column group per column tile
  size_t n1[kLists] = {}, n2 = 0, nc = 0;
  for (int i = 0; i < n; ++i) {
    const int c = cols1(inst[i].n_out);
    n1[list_of(inst[i].n_out)] += (size_t)rows1(inst[i].n_in) * c;
    n2 += tiles2(inst[i].n_out);
    nc += c;
  }
  P.off_cols = take(nc * sizeof(FoldColumns));
  for (int l = 0; l < kLists; ++l) P.off_map1[l] = take(n1[l] * sizeof(FoldRowTile));
  P.off_map2 = take(n2 * sizeof(uint32_t));
  P.off_sum = take((size_t)n_outputs * sizeof(SumJob));
  P.desc = off;
  P.off_T = take(P.tab_bytes);
  P.off_P = take(fbytes);
  P.off_U = off;
  P.U_off.resize(n);
  for (int i = 0; i < n; ++i) {
    P.U_off[i] = take(fold_mid_bytes(inst[i].n_in, inst[i].n_out));
    plain += align_up(mat_bytes(inst[i].n_out, inst[i].n_in, true)) *
             (inst[i].shift_x == inst[i].shift_y ? 2 : 3);
  }
  // planes grouped by output, in instance order within an output
  std::vector<int> count(n_outputs, 0), seen(n_outputs, 0);
  std::vector<size_t> base(n_outputs, 0);
  for (int i = 0; i < n; ++i) ++count[inst[i].out_index];
  P.off_I = off;
  P.I_off.resize(n);
  for (int i = 0; i < n; ++i) {
    const int o = inst[i].out_index;
    const size_t plane = (size_t)inst[i].n_out * inst[i].n_out * sizeof(float);
    if (seen[o] == 0) {
      base[o] = take(count[o] * plane);
      plain += align_up(count[o] * plane);
    }
    P.I_off[i] = base[o] + (size_t)seen[o]++ * plane;
  }
  P.total = std::max(off, P.desc + plain);
  return DLX_OK;
}

// Cut a tile list into 8 runs of equal cost, one per XCD.
void cut_list(const std::vector<float>& cost, int (&xcd)[9]) {
  double total = 0.0, run = 0.0;
  for (float c : cost) total += c;
  int x = 0;
  xcd[0] = 0;
  for (size_t t = 0; t < cost.size(); ++t) {
    while (x < 7 && run >= total * (x + 1) / 8) xcd[++x] = (int)t;
    run += cost[t];
  }
  while (x < 8) xcd[++x] = (int)cost.size();
}

// The descriptors.  A stage-1 list is dealt to the XCDs in units of an eighth
// of a field's row blocks with all its column groups, the costliest unit first
// to the XCD with the least work, and every XCD runs its long tiles first: the
// launch ends evenly (whole fields dealt to XCDs kept 160 of 512 workgroup
// slots busy for 48 sources of 256^2 to 1024^2; a list cut into runs of equal
// cost, an XCD of large fields alone, left a half-empty second round), and the
// workgroups that share field rows share an L2.
void plan_fill(int n, const dlx_mft_instance* inst, int n_outputs, float* const* outs, uint8_t* ws,
               Plan& P) {
  for (size_t q = 0; q < P.tab.size(); ++q) P.tab[q].out = ws + P.off_T + P.tab_off[q];
  for (size_t f = 0; f < P.fld.size(); ++f) P.fld[f].out = ws + P.off_P + P.fld_off[f];
  std::vector<std::vector<int>> members(P.fld.size());
  for (int i = 0; i < n; ++i) members[P.fld_of[i]].push_back(i);
  struct Unit {
    int cols, ncols, row, nrows;
    float cost;   // of one row block
  };
  std::vector<Unit> units;
  for (int l = kLists - 1; l >= 0; --l) {
    const int L = 128 / kWidth[l];
    units.clear();
    for (size_t f = 0; f < members.size(); ++f) {
      const int c0 = (int)P.cols.size(), st = (fold_half(P.fld[f].n) + 15) / 16;
      for (int i : members[f]) {
        const dlx_mft_instance& d = inst[i];
        if (list_of(d.n_out) != l) continue;
        const FoldTableJob& t = P.tab[P.tab_of[i]];
        const double sg = d.inverse ? -1.0 : 1.0;
        for (int c = 0; c < cols1(d.n_out); ++c) {
          if ((int)P.cols.size() == c0 || P.cols.back().count == L) {
            FoldColumns g{};
            g.src = P.fld[f].out;
            g.n = d.n_in;
            P.cols.push_back(g);
          }
          FoldColumns& g = P.cols.back();
          // the input half of the shift (the output half is a phase: no intensity)
          g.tile_of[g.count++] = {t.out, ws + P.U_off[i], sg * t.step * d.shift_x,
                                  sg * t.step * d.shift_y, c * kWidth[l], d.n_out};
        }
      }
      const int nc = (int)P.cols.size() - c0;
      if (nc == 0) continue;
      float cost = 0.f;   // a step's fixed part and its products, and a tile's store
      for (int c = c0; c < c0 + nc; ++c)
        cost += (float)(P.cols[c].count * ((st + 2) * (kWidth[l] + 64) + 256));
      const int rows = rows1(P.fld[f].n), piece = (rows + 7) / 8;
      for (int r = 0; r < rows; r += piece)
        units.push_back({c0, nc, r, std::min(piece, rows - r), cost});
    }
    std::stable_sort(units.begin(), units.end(), [](const Unit& a, const Unit& b) {
      return a.cost * a.nrows > b.cost * b.nrows;
    });
    std::vector<const Unit*> on[8];
    double load[8] = {};
    for (const Unit& u : units) {
      int best = 0;
      for (int x = 1; x < 8; ++x)
        if (load[x] < load[best]) best = x;
      on[best].push_back(&u);
      load[best] += u.cost * u.nrows;
    }
    for (int x = 0; x < 8; ++x) {
      P.xcd1[l][x] = (int)P.map1[l].size();
      std::stable_sort(on[x].begin(), on[x].end(), [](const Unit* a, const Unit* b) {
        return a->cost / a->ncols > b->cost / b->ncols;
      });
      for (const Unit* u : on[x])
        for (int r = u->row; r < u->row + u->nrows; ++r)
          for (int c = u->cols; c < u->cols + u->ncols; ++c)
            P.map1[l].push_back({(uint32_t)c, (uint32_t)(r * kFoldTilePy)});
    }
    P.xcd1[l][8] = (int)P.map1[l].size();
  }
  P.prob.reserve(n);
  std::vector<float> cost2;
  // stage 2: instances of one field (a source's wavelengths) together, in runs
  // of equal cost
  for (const std::vector<int>& run : members)
    for (int i : run) {
      const dlx_mft_instance& d = inst[i];
      const double c = mft_norm(geom_of(d), d.wavelength, d.pixel_scale_in, d.pixel_scale_out);
      FoldProblem p{};
      p.table = P.tab[P.tab_of[i]].out;
      p.mid = ws + P.U_off[i];
      p.out = (float*)(ws + P.I_off[i]);
      p.alpha = (float)(c * std::sqrt(d.weight));
      p.n = d.n_in;
      p.m = d.n_out;
      p.inverse = d.inverse ? 1 : 0;
      p.tile = (int)P.map2.size();
      P.map2.insert(P.map2.end(), tiles2(p.m), (uint32_t)P.prob.size());
      cost2.insert(cost2.end(), tiles2(p.m), (float)((fold_half(p.n) + 15) / 16 + 6));
      P.prob.push_back(p);
    }
  cut_list(cost2, P.xcd2);
  std::vector<int> job(n_outputs, -1);
  for (int i = 0; i < n; ++i) {
    int& j = job[inst[i].out_index];
    if (j < 0) {
      j = (int)P.sum.size();
      P.sum.push_back({outs[inst[i].out_index], (const float*)(ws + P.I_off[i]),
                       (long)inst[i].n_out * inst[i].n_out, 0, 0});
    }
    ++P.sum[j].count;
  }
}

// ---------------------------------------------------------------------------
// launches, eager or as a replayed graph
// ---------------------------------------------------------------------------
// Every launch reads its jobs and problems from the descriptors at the front of
// the workspace; its grid and by-value arguments depend on the plan's shape
// only.  So one captured graph serves every call with the same workspace and
// the same shape, whatever the fields, wavelengths, weights, shifts, outputs
// and table addresses (all uploaded before the launch).
int launch_plan(const Plan& Q, uint8_t* ws, bool with_tables, hipStream_t s) {
  if (with_tables)
    DLX_HIP(launch_fold_group_tables((const FoldTableJob*)(ws + Q.off_tab), (int)Q.tab.size(),
                                     Q.tab_most, s));
  DLX_HIP(launch_fold_group_fields((const FoldFieldJob*)(ws + Q.off_fld), (int)Q.fld.size(),
                                   Q.fld_most, s));
  FoldGroup g{};
  g.probs = (const FoldProblem*)(ws + Q.off_prob);
  g.cols = (const FoldColumns*)(ws + Q.off_cols);
  for (int l = kLists - 1; l >= 0; --l) {   // the largest outputs first
    if (Q.map1[l].empty()) continue;
    g.rows = (const FoldRowTile*)(ws + Q.off_map1[l]);
    std::memcpy(g.xcd, Q.xcd1[l], sizeof(g.xcd));
    DLX_HIP(launch_fold_group_stage1(g, kWidth[l], s));
  }
  g.map = (const uint32_t*)(ws + Q.off_map2);
  std::memcpy(g.xcd, Q.xcd2, sizeof(g.xcd));
  DLX_HIP(launch_fold_group_stage2(g, s));
  if (Q.sum.empty()) return DLX_OK;
  long most = 0;
  for (const SumJob& j : Q.sum) most = j.npix > most ? j.npix : most;
  const unsigned gx = (unsigned)std::min<long>((most + 255) / 256, 256);
  hipLaunchKernelGGL(group_sum_kernel, dim3(gx, (unsigned)Q.sum.size()), dim3(256), 0, s,
                     (const SumJob*)(ws + Q.off_sum));
  return launch_status("group_sum_kernel");
}

// Everything launch_plan's grids and by-value arguments depend on.
std::vector<long> plan_shape(const Plan& Q, const uint8_t* ws, bool fresh, int dev) {
  std::vector<long> k = {(long)dev, (long)(uintptr_t)ws, (long)fresh, (long)Q.off_tab,
                         (long)Q.tab.size(), (long)Q.tab_most, (long)Q.off_fld, (long)Q.fld.size(),
                         (long)Q.fld_most, (long)Q.off_prob, (long)Q.off_cols, (long)Q.off_map2,
                         (long)Q.off_sum, (long)Q.sum.size()};
  for (int l = 0; l < kLists; ++l) {
    k.push_back((long)Q.off_map1[l]);
    k.insert(k.end(), Q.xcd1[l], Q.xcd1[l] + 9);
  }
  k.insert(k.end(), Q.xcd2, Q.xcd2 + 9);
  for (const SumJob& j : Q.sum) k.push_back(j.npix);
  return k;
}

struct GraphEntry {
  hipGraphExec_t exec = nullptr;
  hipEvent_t done = nullptr;     // recorded after the entry's latest launch
  uint64_t tick = 0;
};

struct GraphCache {
  std::mutex mu;
  std::map<std::vector<long>, GraphEntry> map;
  std::map<int, hipStream_t> capture;   // per device: a private stream to capture on
  uint64_t tick = 0, captures = 0, replays = 0;
  int enabled = -1;              // -1: not yet read from the environment
  static constexpr size_t kMax = 64;
};

GraphCache& graphs() {
  static GraphCache c;
  return c;
}

int graphs_on(GraphCache& c) {
  if (c.enabled < 0) {
    // off by default: on ROCm 7.2 a launch of this graph took more host time
    // than its direct launches (50-480 us against 50-380 us per call)
    const char* e = std::getenv("DLUX_AMD_BATCHED_GRAPHS");
    c.enabled = (e && e[0] == '1') ? 1 : 0;
  }
  return c.enabled;
}

void drop_entry(GraphEntry& e) {
  if (e.done) {
    hipEventSynchronize(e.done);   // the exec is destroyed after its last launch ran
    hipEventDestroy(e.done);
  }
  if (e.exec) hipGraphExecDestroy(e.exec);
  e = GraphEntry{};
}

// Launch the plan through the graph cache.  The first sighting of a shape runs
// eagerly (*eager set); the second captures the launches on a private stream
// (capture records and runs nothing), instantiates the graph and launches it
// on `s`; later sightings launch it again.  The caller's stream may be the
// null stream.
int launch_plan_graph(const Plan& Q, uint8_t* ws, bool fresh, hipStream_t s, bool* eager) {
  *eager = true;
  GraphCache& c = graphs();
  std::lock_guard<std::mutex> lock(c.mu);
  if (!graphs_on(c)) return DLX_OK;
  int dev = 0;
  DLX_HIP(hipGetDevice(&dev));
  std::vector<long> key = plan_shape(Q, ws, fresh, dev);
  auto it = c.map.find(key);
  if (it == c.map.end()) {
    if (c.map.size() >= GraphCache::kMax) {
      auto old = c.map.begin();
      for (auto q = c.map.begin(); q != c.map.end(); ++q)
        if (q->second.tick < old->second.tick) old = q;
      drop_entry(old->second);
      c.map.erase(old);
    }
    c.map[key].tick = ++c.tick;
    return DLX_OK;
  }
  GraphEntry& e = it->second;
  e.tick = ++c.tick;
  if (!e.exec) {
    hipStream_t& cs = c.capture[dev];
    if (!cs) DLX_HIP(hipStreamCreateWithFlags(&cs, hipStreamNonBlocking));
    hipGraph_t g = nullptr;
    DLX_HIP(hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal));
    const int st = launch_plan(Q, ws, fresh, cs);
    const hipError_t end = hipStreamEndCapture(cs, &g);
    if (st) {
      if (end == hipSuccess && g) hipGraphDestroy(g);
      return st;
    }
    DLX_HIP(end);
    const hipError_t inst = hipGraphInstantiate(&e.exec, g, nullptr, nullptr, 0);
    hipGraphDestroy(g);
    if (inst != hipSuccess) {
      e.exec = nullptr;
      DLX_HIP(inst);
    }
    DLX_HIP(hipEventCreateWithFlags(&e.done, hipEventDisableTiming));
    ++c.captures;
  }
  DLX_HIP(hipGraphLaunch(e.exec, s));
  DLX_HIP(hipEventRecord(e.done, s));
  ++c.replays;
  *eager = false;
  return DLX_OK;
}

template <typename T>
void put(std::vector<uint8_t>& host, size_t off, const std::vector<T>& v) {
  if (!v.empty()) std::memcpy(host.data() + off, v.data(), v.size() * sizeof(T));
}

}  // namespace
}  // namespace dlx

using namespace dlx;

extern "C" {

size_t dlx_mft_batched_workspace_size(int32_t n, const dlx_mft_instance* instances,
                                      int32_t n_outputs) {
  if (n <= 0 || !instances || n_outputs <= 0) return 0;
  for (int i = 0; i < n; ++i)
    if (instances[i].out_index < 0 || instances[i].out_index >= n_outputs ||
        instances[i].n_in <= 0 || instances[i].n_out <= 0)
      return 0;
  Plan P;
  if (plan_sizes(n, instances, n_outputs, P) != DLX_OK) return 0;
  return P.total;
}

int dlx_mft_batched_psf(int32_t n, const dlx_mft_instance* instances, int32_t n_outputs,
                        float* const* outputs, void* workspace, size_t workspace_bytes,
                        void* stream) {
  clear_error();
  if (int st = validate(n, instances, n_outputs)) return st;
  if (n == 0 || n_outputs == 0) return DLX_OK;
  DLX_CHECK_ARG(outputs != nullptr, "outputs is NULL");
  for (int i = 0; i < n; ++i)
    DLX_CHECK_ARG(outputs[instances[i].out_index] != nullptr, "outputs[%d] is NULL",
                  instances[i].out_index);
  hipStream_t s = (hipStream_t)stream;
  Plan Q;
  if (int st = plan_sizes(n, instances, n_outputs, Q)) return st;
  if (!workspace || workspace_bytes < Q.total) {
    set_error("dlx_mft_batched_psf workspace too small: need %zu bytes, got %zu", Q.total,
              workspace_bytes);
    return DLX_ERR_WORKSPACE;
  }
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  DLX_HIP(hipStreamIsCapturing(s, &cs));
  if (cs != hipStreamCaptureStatusNone) {
    set_error("dlx_mft_batched_psf uploads per-call descriptors and cannot be captured");
    return DLX_ERR_UNSUPPORTED;
  }
  uint8_t* ws = (uint8_t*)workspace;

  // The tables depend only on the instances' sides and phase steps: keep the
  // whole set resident in the device cache and regenerate only on a miss.
  std::vector<double> key;
  key.reserve(1 + Q.tab.size() * 3);
  key.push_back(2002.0);
  for (const FoldTableJob& j : Q.tab) key.insert(key.end(), {(double)j.n, (double)j.m, j.step});
  void* tcache = nullptr;
  CacheLease lease(s);
  bool fresh = true;
  if (int st = cache_acquire_raw(key, Q.tab_bytes, s, &tcache, &lease.h, &fresh)) return st;
  plan_fill(n, instances, n_outputs, outputs, ws, Q);
  if (tcache) {
    const uint8_t* t0 = ws + Q.off_T;
    for (FoldTableJob& j : Q.tab) j.out = (uint8_t*)tcache + (j.out - t0);
    for (FoldProblem& p : Q.prob) p.table = (const uint8_t*)tcache + (p.table - t0);
    for (FoldColumns& g : Q.cols)
      for (int i = 0; i < g.count; ++i)
        g.tile_of[i].table = (const uint8_t*)tcache + (g.tile_of[i].table - t0);
  }
  // all descriptors sit at the front of the workspace: one upload
  std::vector<uint8_t> host(Q.desc, 0);
  put(host, Q.off_tab, Q.tab);
  put(host, Q.off_fld, Q.fld);
  put(host, Q.off_prob, Q.prob);
  put(host, Q.off_cols, Q.cols);
  for (int l = 0; l < kLists; ++l) put(host, Q.off_map1[l], Q.map1[l]);
  put(host, Q.off_map2, Q.map2);
  put(host, Q.off_sum, Q.sum);
  if (int st = upload(host.data(), host.size(), ws, s)) return st;

  // the launches, as a replayed graph when this shape was seen before
  bool eager = true;
  if (int st = launch_plan_graph(Q, ws, fresh, s, &eager)) return st;
  if (eager)
    if (int st = launch_plan(Q, ws, fresh, s)) return st;
  if (fresh)
    if (int st = cache_ready(lease.h, s)) return st;
  return lease.release();
}

int dlx_batched_graph_stats(uint64_t* captures, uint64_t* launches, int32_t* entries) {
  clear_error();
  GraphCache& c = graphs();
  std::lock_guard<std::mutex> lock(c.mu);
  if (captures) *captures = c.captures;
  if (launches) *launches = c.replays;
  if (entries) {
    int n = 0;
    for (auto& kv : c.map) n += kv.second.exec != nullptr;
    *entries = n;
  }
  return DLX_OK;
}

int dlx_batched_graphs(int32_t enable) {
  clear_error();
  GraphCache& c = graphs();
  std::lock_guard<std::mutex> lock(c.mu);
  const int prev = graphs_on(c);
  if (enable >= 0) {
    c.enabled = enable ? 1 : 0;
    if (!c.enabled) {
      for (auto& kv : c.map) drop_entry(kv.second);
      c.map.clear();
    }
  }
  return prev;
}

}  // extern "C"
