// symgs.hip -- multicolor symmetric Gauss-Seidel sweep (the reference's
// SymGSSolver, src/symgs/symgs.h:28; algorithm src/symgs/omp_base.cc:8-39 and
// src/symgs/verifier.cc:50-77), bit-exact with the sequential sweep.
//
// Semantics.  For each color c = 0..C-1, then C-1..0: every row r listed in
// indices[color_offsets[c] .. color_offsets[c+1]) gets
//     rsum = sum over the row's off-diagonal entries, in CSR order, of
//            x[col] * val (product rounded, then added: sequential FP32);
//     diag = the value of the row's LAST entry with column == r (0 if none);
//     x[r] = (b[r] - rsum) / diag   unless diag == 0.
// Rows of one color never reference each other (a proper coloring, checked
// when the plan is built), so updating them in parallel equals the
// reference's sequential loop over the color, bit for bit.
//
// Layout in HBM (built once per plan).  Every color is a contiguous range of
// plan rows, its rows of at most kSeqRow (64) off-diagonal entries first, by
// falling length (in chunks, kSortRows), then its longer rows.
//
// Short rows: slices of up to 64 rows (one wavefront, one lane a row), the
// entries of a slice stored in 16-byte groups across its rows (group k of lane
// l at off + k * rows + l), so a wavefront reads 1 KB of consecutive entries
// with each load and every lane adds its own row in CSR order in a register:
// no LDS, no barrier, no per-row offsets.  A group is two {column, value}
// pairs; where all rows of the slice are of one length and the k-th entry of
// each lies the same number of columns from its row (interior rows of a
// stencil), it is four values, and the distances are stored once a slice.
// Sorting by length keeps the padding to a group a row plus what the few
// slices that straddle a length change hold; a slice of fewer rows is stored
// that narrow, so a color of one row costs one row.
//
// Long rows: CSR, one workgroup each (hub_chain_sum: the workgroup gathers a
// chunk into LDS while one lane adds the previous one in order).
//
// One color = one launch of symgs_color_kernel; the stream orders the colors.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cstring>
#include <vector>

#include "gardenia_hip.h"
#include "gd_common.h"
#include "pull_engine.h"

namespace gd {
namespace {

constexpr int kSgXcds = 8;

// Rows sorted by length together.  A slice of rows far apart gathers from as many
// lines of x as rows, so rows of many lengths are sorted in chunks: 200,000 rows
// of 1 .. 64 entries within 2000 columns, one sweep, all together / in chunks of
// 64 / 256 / 1024: 203 / 115 / 113 / 129 us (LDS row tiles over a CSR 129); 1 M of
// 1 .. 40 540 / 257 / 204 / 261 (267); 1 M of 18 .. 27 310 / 166 / 173 / 210 (265).
// Where nearly all of a color's rows are of one length (large stencils), they
// stay neighbours in either order, and all together leave fewer slices with two
// lengths.  27-point stencils, two sweeps, all together / in chunks of 256: 126^3
// (95 % of the rows inside) 355 / 422 us, 97^3 (94 %) 212 / 189, 80^3 (93 %) 170 /
// 161, 40^3 (86 %) 121 / 115; 1 M rows, three quarters of one length 309 / 173.
constexpr int kSortRows = 256;
constexpr int64_t kSgDeltaMax = (1ll << 31) - 128;  // distances a plan stores at most

// Up to 64 rows of one color.  A general slice (delta < 0) has `n` pairs of
// entries a row at ent[off ...]; a uniform one, where the k-th entry of every
// row lies the same number of columns from its row, `n` float4 of values
// there and the `len` column distances at delta[delta ...].
struct Slice {
  int row0;    // first plan row
  int n_rows;  // 1 .. 64
  int n;
  int len;  // entries of the longest row
  int64_t off;
  int delta;
  int pad;
};

// One plan row.
struct RowRec {
  float diag;
  int orig;  // its matrix row
  int len;   // off-diagonal entries
  int pad;
};
static_assert(sizeof(RowRec) == 16 && sizeof(Slice) == 32, "plan records");

struct SymgsArgs {
  float* x;
  const float* __restrict__ b;
  const RowRec* __restrict__ rows;
  const Slice* __restrict__ slices;
  int n_slices;
  const int4* __restrict__ ent;  // {column, value, column, value} or four values
  const int* __restrict__ delta;
  const Tile* __restrict__ hubs;  // long rows: {plan row, -, first entry, end}
  int n_hubs;
  const int32_t* __restrict__ col;  // long rows
  const float* __restrict__ val;
  int e_max;
};

struct SymgsGather {
  const float* __restrict__ x;
  const float* __restrict__ val;
  // x[j] * Ax[jj] (src/symgs/verifier.cc:61): rounded here, added in order later
  __device__ __forceinline__ float value(int e, int u) const { return x[u] * val[e]; }
};

// if (diag != 0) x[inew] = (b[inew] - rsum) / diag   (verifier.cc:63)
__device__ __forceinline__ void row_update(const SymgsArgs& a, const RowRec& r, float bv,
                                           float rsum) {
  if (r.diag != 0.0f) a.x[r.orig] = (bv - rsum) / r.diag;
}

// One general slice on one wavefront, kP pairs of entries a step, the next
// step's in flight.  Two pairs for rows of up to 12 entries, four for longer ones
// (200,000 rows of 1 .. 64, one sweep: 167 us with two, 113 with four; 50,000 of
// 1 .. 64 121 / 93).  Eight are faster for few rows (92) and slower for many (1 M
// of 1 .. 40 204 us with four, 228 with eight): neighbouring entries of a row
// often share a line of x, which the first load of it must have brought in before
// the next asks.
// The entries a lane reads past its row are the slice's padding or, past the
// slice's end, its last pair again: their terms are replaced by -0.0, which
// changes no sum.
template <int kP>
__device__ __forceinline__ float general_sum(const SymgsArgs& a, const Slice& sl,
                                             const RowRec& r, int lane) {
  const int4* __restrict__ e = a.ent + sl.off + lane;
  const int last = sl.n - 1;
  float sum = 0.0f;
  int4 cur[kP], nxt[kP];
  if (last >= 0) {
#pragma unroll
    for (int j = 0; j < kP; j++) cur[j] = e[(int64_t)min(j, last) * sl.n_rows];
  }
  for (int k = 0; k <= last; k += kP) {
    float v[2 * kP];
#pragma unroll
    for (int j = 0; j < kP; j++) {
      v[2 * j] = a.x[cur[j].x];
      v[2 * j + 1] = a.x[cur[j].z];
    }
#pragma unroll
    for (int j = 0; j < kP; j++) nxt[j] = e[(int64_t)min(k + kP + j, last) * sl.n_rows];
    const int left = r.len - 2 * k;
#pragma unroll
    for (int j = 0; j < kP; j++) {
      const float t0 = v[2 * j] * __int_as_float(cur[j].y);
      const float t1 = v[2 * j + 1] * __int_as_float(cur[j].w);
      sum += 2 * j < left ? t0 : -0.0f;
      sum += 2 * j + 1 < left ? t1 : -0.0f;
    }
#pragma unroll
    for (int j = 0; j < kP; j++) cur[j] = nxt[j];
  }
  return sum;
}

// One uniform slice: 4 bytes an entry instead of 8, the columns from scalar
// registers.  Padding distances are 0.  27-point stencil, two sweeps: 97^3 212
// us (general slices 234, LDS row tiles over a CSR 322), 128^3 382 (499, 598):
// 12.5 MB of values a color at 97^3, most of them from the Infinity Cache, in
// 6.6 us, about 2.5 of which is the launch.  Bound by the gathers of x: two or
// four groups of values a step, in flight together, cost 220 and 226 us.
__device__ __forceinline__ float uniform_sum(const SymgsArgs& a, const Slice& sl,
                                             const RowRec& r, int lane) {
  const float4* __restrict__ e = reinterpret_cast<const float4*>(a.ent) + sl.off + lane;
  const int4* __restrict__ d = reinterpret_cast<const int4*>(a.delta + sl.delta);
  float sum = 0.0f;
  float4 cur = e[0];
  for (int k = 0; k < sl.n; k++) {
    const int4 c = d[k];
    const float x0 = a.x[r.orig + c.x], x1 = a.x[r.orig + c.y], x2 = a.x[r.orig + c.z],
                x3 = a.x[r.orig + c.w];
    const float4 nxt = e[(int64_t)min(k + 1, sl.n - 1) * sl.n_rows];
    const int left = sl.len - 4 * k;
    sum += x0 * cur.x;
    sum += 1 < left ? x1 * cur.y : -0.0f;
    sum += 2 < left ? x2 * cur.z : -0.0f;
    sum += 3 < left ? x3 * cur.w : -0.0f;
    cur = nxt;
  }
  return sum;
}

__device__ __forceinline__ void slice_rows(const SymgsArgs& a, const Slice& sl, int lane) {
  if (lane >= sl.n_rows) return;
  const RowRec r = a.rows[sl.row0 + lane];
  const float bv = a.b[r.orig];
  row_update(a, r, bv,
             sl.delta >= 0 ? uniform_sum(a, sl, r, lane)
             : sl.len > 12 ? general_sum<4>(a, sl, r, lane)
                           : general_sum<2>(a, sl, r, lane));
}

// The slice of workgroup b: the slices in 8 equal runs, one an XCD, since
// neighbouring rows share x lines.
__device__ __forceinline__ int xcd_slice(int b, int n) {
  const int xcd = b % kSgXcds;
  return xcd * (n / kSgXcds) + min(xcd, n % kSgXcds) + b / kSgXcds;
}

// One color in one launch, of wavefront-sized workgroups, one slice each:
// they spread evenly over the SIMDs however few there are (256-thread
// workgroups of four slices: 97^3 274 us, 40^3 173; these: 261 and 106).
__global__ __launch_bounds__(kWave) void symgs_color_kernel(const SymgsArgs a) {
  slice_rows(a, a.slices[xcd_slice(blockIdx.x, a.n_slices)], threadIdx.x);
}

// The same for a color with long rows: workgroups [0, n_hubs) add one long row
// each (hub_chain_sum), the rest take four slices each.  Long rows first: they
// take longest.
__global__ __launch_bounds__(kBlock) void symgs_long_kernel(const SymgsArgs a) {
  __shared__ __align__(16) float buf[2 * kHubChunk + 4];
  const int b = blockIdx.x;
  if (b < a.n_hubs) {
    const Tile t = a.hubs[b];
    const RowRec r = a.rows[t.x];
    const float bv = a.b[r.orig];
    // 16 float4 LDS reads ahead: the chains bound these sweeps (8 ahead: 9% slower)
    const float rsum =
        hub_chain_sum<16, false>(a.col, nullptr, a.e_max, t.z, t.w - t.z,
                                 SymgsGather{a.x, a.val}, 0.0f, buf, buf + kHubChunk,
                                 buf + 2 * kHubChunk);
    if (threadIdx.x == 0) row_update(a, r, bv, rsum);
    return;
  }
  const int s = __builtin_amdgcn_readfirstlane((b - a.n_hubs) * (kBlock / kWave) +
                                               (int)threadIdx.x / kWave);
  if (s < a.n_slices) slice_rows(a, a.slices[s], threadIdx.x % kWave);
}

#define SG_LOOP(i, n) \
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < (n); \
       i += (int64_t)gridDim.x * blockDim.x)

int sg_grid(int64_t n) { return (int)std::max<int64_t>(1, std::min<int64_t>((n + 255) / 256, 8192)); }

// Plan row i = matrix row idx[i]: range check, its color (binary search in
// the color offsets), and each matrix row listed at most once.
__global__ void sg_rows_kernel(int n_p, const int32_t* __restrict__ idx, int m,
                               const int32_t* __restrict__ co, int n_colors,
                               int32_t* __restrict__ color_of, int* __restrict__ bad) {
  SG_LOOP(i, n_p) {
    const int r = idx[i];
    if (r < 0 || r >= m) {
      atomicOr(bad, 1);
      continue;
    }
    const int pos = co[0] + (int)i;
    int lo = 0, hi = n_colors;  // last c with co[c] <= pos
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (co[mid] <= pos)
        lo = mid;
      else
        hi = mid;
    }
    if (atomicCAS(color_of + r, -1, lo) != -1) atomicOr(bad, 2);
  }
}

// Off-diagonal count and last diagonal value of plan input row i; a proper
// coloring joins no two rows of one color by an off-diagonal entry.
__global__ void sg_count_kernel(int n_p, const int32_t* __restrict__ idx,
                                const int32_t* __restrict__ Ap, const int32_t* __restrict__ Aj,
                                const float* __restrict__ Ax,
                                const int32_t* __restrict__ color_of, int32_t* __restrict__ len,
                                float* __restrict__ diag, int* __restrict__ bad) {
  SG_LOOP(i, n_p) {
    const int r = idx[i];
    const int c = color_of[r];
    int n = 0, f = 0;
    float d = 0.0f;
    for (int k = Ap[r]; k < Ap[r + 1]; k++) {
      const int j = Aj[k];
      if (j == r) {
        d = Ax[k];
      } else {
        n++;
        f |= color_of[j] == c;
      }
    }
    len[i] = n;
    diag[i] = d;
    if (f) atomicOr(bad, 4);
  }
}

// Plan row q is input row order[q].
__global__ void sg_rec_kernel(int n_p, const int32_t* __restrict__ order,
                              const int32_t* __restrict__ idx, const int32_t* __restrict__ len,
                              const float* __restrict__ diag, RowRec* __restrict__ rows) {
  SG_LOOP(q, n_p) {
    const int i = order[q];
    rows[q] = RowRec{diag[i], idx[i], len[i], 0};
  }
}

// The off-diagonal entries of matrix row r, in CSR order: next() -> one more.
struct RowEntries {
  const int32_t* __restrict__ Aj;
  const float* __restrict__ Ax;
  int r, k, end;
  __device__ __forceinline__ bool next(int* c, float* v) {
    while (k < end && Aj[k] == r) k++;
    if (k >= end) return false;
    *c = Aj[k];
    *v = Ax[k];
    k++;
    return true;
  }
};

// One wavefront a slice whose rows are all of one length (the others have
// delta < 0 already): uniform, then distances to delta[slices[s].delta ...],
// or delta = -1.
__global__ void sg_uniform_kernel(int n_slices, Slice* __restrict__ slices,
                                  const RowRec* __restrict__ rows, const int32_t* __restrict__ Ap,
                                  const int32_t* __restrict__ Aj, const float* __restrict__ Ax,
                                  int* __restrict__ delta) {
  const int lane = threadIdx.x % kWave;
  for (int64_t s = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kWave; s < n_slices;
       s += (int64_t)gridDim.x * blockDim.x / kWave) {
    const Slice sl = slices[s];
    if (sl.delta < 0) continue;
    const int r = rows[sl.row0 + min(lane, sl.n_rows - 1)].orig;
    RowEntries e{Aj, Ax, r, Ap[r], Ap[r + 1]};
    bool same = true;
    for (int k = 0; k < sl.len; k++) {
      int c = r;
      float v = 0.0f;
      e.next(&c, &v);
      const int d = c - r;
      same = same && d == __builtin_amdgcn_readfirstlane(d);
      if (lane == 0) delta[sl.delta + k] = d;
    }
    if (__ballot(!same) && lane == 0) slices[s].delta = -1;
  }
}

// The entries of slice s, by one wavefront; pads repeat the row's own column.
__global__ void sg_slice_fill_kernel(int n_slices, const Slice* __restrict__ slices,
                                     const RowRec* __restrict__ rows,
                                     const int32_t* __restrict__ Ap,
                                     const int32_t* __restrict__ Aj, const float* __restrict__ Ax,
                                     int4* __restrict__ ent) {
  const int lane = threadIdx.x % kWave;
  for (int64_t s = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kWave; s < n_slices;
       s += (int64_t)gridDim.x * blockDim.x / kWave) {
    const Slice sl = slices[s];
    if (lane >= sl.n_rows) continue;
    const int r = rows[sl.row0 + lane].orig;
    RowEntries e{Aj, Ax, r, Ap[r], Ap[r + 1]};
    for (int p = 0; p < sl.n; p++) {
      int c[4] = {r, r, r, r};
      float v[4] = {};
      const int n = sl.delta >= 0 ? 4 : 2;
#pragma unroll
      for (int h = 0; h < 4; h++)
        if (h < n) e.next(&c[h], &v[h]);
      int4 q = make_int4(c[0], __float_as_int(v[0]), c[1], __float_as_int(v[1]));
      if (n == 4)
        q = make_int4(__float_as_int(v[0]), __float_as_int(v[1]), __float_as_int(v[2]),
                      __float_as_int(v[3]));
      ent[sl.off + (int64_t)p * sl.n_rows + lane] = q;
    }
  }
}

// The entries of the long rows, one thread a row.
__global__ void sg_hub_fill_kernel(int n_hubs, const Tile* __restrict__ hubs,
                                   const RowRec* __restrict__ rows,
                                   const int32_t* __restrict__ Ap,
                                   const int32_t* __restrict__ Aj, const float* __restrict__ Ax,
                                   int32_t* __restrict__ col, float* __restrict__ val) {
  SG_LOOP(h, n_hubs) {
    const int r = rows[hubs[h].x].orig;
    int o = hubs[h].z;
    for (int k = Ap[r]; k < Ap[r + 1]; k++) {
      const int j = Aj[k];
      if (j != r) {
        col[o] = j;
        val[o] = Ax[k];
        o++;
      }
    }
  }
}

}  // namespace
}  // namespace gd

using namespace gd;

struct gd_symgs_plan {
  int m = 0;
  int n_p = 0;  // rows swept (color_offsets[C] - color_offsets[0])
  int64_t nnz_p = 0;  // off-diagonal entries of those rows
  int n_colors = 0;
  int64_t hub_nnz = 0;  // those of the long rows
  double plan_ms = 0.0;
  DeviceBuffer rows, slices, ent, delta, hubs, col, val;
  std::vector<int> slice_begin, hub_begin;  // per color, n_colors + 1 entries
  int max_row_len = 0;
};

namespace {

int read_flag(const DeviceBuffer& b, hipStream_t s, int* h) {
  GD_HIP_TRY(hipMemcpyAsync(h, b.ptr, sizeof(int), hipMemcpyDeviceToHost, s));
  GD_HIP_TRY(hipStreamSynchronize(s));
  return GD_OK;
}

int plan_build(gd_symgs_plan* p, int m, int64_t nnz, const int32_t* d_Ap, const int32_t* d_Aj,
               const float* d_Ax, const int32_t* d_idx, const int32_t* co, int C, hipStream_t s) {
  p->m = m;
  p->n_colors = C;
  const int n_p = co[C] - co[0];
  p->n_p = n_p;
  int rc = check_columns(d_Aj, nnz, m, s);
  if (rc) return rc;
  {  // the matrix offsets must be a CSR prefix sum
    std::vector<int32_t> h(m + 1);
    GD_HIP_TRY(hipMemcpyAsync(h.data(), d_Ap, 4 * ((size_t)m + 1), hipMemcpyDeviceToHost, s));
    GD_HIP_TRY(hipStreamSynchronize(s));
    GD_CHECK_ARG(h[0] == 0 && (int64_t)h[m] == nnz, "Ap[0] must be 0 and Ap[m] must equal nnz");
    for (int i = 0; i < m; i++) GD_CHECK_ARG(h[i + 1] >= h[i], "Ap must be non-decreasing");
  }
  const size_t np = (size_t)std::max(n_p, 1);
  DeviceBuffer d_co, color_of, bad, len, diag, order;
  rc = d_co.alloc(4 * ((size_t)C + 1));
  if (!rc) rc = color_of.alloc(4 * (size_t)std::max(m, 1));
  if (!rc) rc = bad.alloc(sizeof(int));
  if (!rc) rc = len.alloc(4 * np);
  if (!rc) rc = diag.alloc(4 * np);
  if (!rc) rc = order.alloc(4 * np);
  if (!rc) rc = p->rows.alloc(sizeof(RowRec) * np);
  if (rc) return rc;
  GD_HIP_TRY(hipMemcpyAsync(d_co.ptr, co, 4 * ((size_t)C + 1), hipMemcpyHostToDevice, s));
  GD_HIP_TRY(hipMemsetAsync(color_of.ptr, 0xff, 4 * (size_t)std::max(m, 1), s));  // -1
  GD_HIP_TRY(hipMemsetAsync(bad.ptr, 0, sizeof(int), s));
  int h_bad = 0;
  std::vector<int32_t> h_len(n_p);
  const int32_t* idx = n_p > 0 ? d_idx + co[0] : nullptr;
  if (n_p > 0) {
    hipLaunchKernelGGL(sg_rows_kernel, dim3(sg_grid(n_p)), dim3(256), 0, s, n_p, idx, m,
                       d_co.as<int32_t>(), C, color_of.as<int32_t>(), bad.as<int>());
    GD_HIP_TRY(hipGetLastError());
    rc = read_flag(bad, s, &h_bad);
    if (rc) return rc;
    GD_CHECK_ARG(!(h_bad & 1), "indices: row outside [0, m)");
    GD_CHECK_ARG(!(h_bad & 2), "indices: a row is listed more than once");
    hipLaunchKernelGGL(sg_count_kernel, dim3(sg_grid(n_p)), dim3(256), 0, s, n_p, idx, d_Ap, d_Aj,
                       d_Ax, color_of.as<int32_t>(), len.as<int32_t>(), diag.as<float>(),
                       bad.as<int>());
    GD_HIP_TRY(hipGetLastError());
    rc = read_flag(bad, s, &h_bad);
    if (rc) return rc;
    GD_CHECK_ARG(!(h_bad & 4), "coloring is not proper: an off-diagonal entry joins two rows of one color");
    GD_HIP_TRY(hipMemcpyAsync(h_len.data(), len.ptr, 4 * (size_t)n_p, hipMemcpyDeviceToHost, s));
    GD_HIP_TRY(hipStreamSynchronize(s));
  }
  // Per color: short rows by falling length, in chunks of kSortRows or all at
  // once (stable, so neighbours of one length stay neighbours), cut into slices;
  // long rows, the longest first (the color lasts as long as its longest row).
  std::vector<int32_t> h_order(n_p);
  std::vector<Slice> slices;
  std::vector<Tile> hubs;
  std::vector<int32_t> longs;
  p->slice_begin.assign(1, 0);
  p->hub_begin.assign(1, 0);
  int64_t deltas = 0, hub_nnz = 0;
  for (int c = 0; c < C; c++) {
    const int r0 = co[c] - co[0], r1 = co[c + 1] - co[0];
    longs.clear();
    int rows_of[kSeqRow + 1] = {}, n_short = 0;
    for (int i = r0; i < r1; i++) {
      p->nnz_p += h_len[i];
      p->max_row_len = std::max(p->max_row_len, (int)h_len[i]);
      if (h_len[i] <= kSeqRow) {
        rows_of[h_len[i]]++;
        n_short++;
      } else {
        longs.push_back(i);
      }
    }
    const int most = *std::max_element(rows_of, rows_of + kSeqRow + 1);
    const int chunk = 15 * (int64_t)most >= 14 * (int64_t)n_short ? std::max(n_short, 1) : kSortRows;
    int at = r0;
    for (int i0 = r0, i1; i0 < r1; i0 = i1) {
      int start[kSeqRow + 1] = {};  // rows of length l, then where they go
      int n = 0;
      for (i1 = i0; i1 < r1 && n < chunk; i1++)
        if (h_len[i1] <= kSeqRow) {
          start[h_len[i1]]++;
          n++;
        }
      for (int l = kSeqRow; l >= 0; l--) {
        const int rows = start[l];
        start[l] = at;
        at += rows;
      }
      for (int i = i0; i < i1; i++)
        if (h_len[i] <= kSeqRow) h_order[start[h_len[i]]++] = i;
    }
    for (int q = r0; q < at; q += kWave) {
      const int n = std::min(kWave, at - q);
      const int len = h_len[h_order[q]];
      const bool one_len = len > 0 && h_len[h_order[q + n - 1]] == len && deltas < kSgDeltaMax;
      slices.push_back(Slice{q, n, 0, len, 0, one_len ? (int)deltas : -1, 0});
      if (one_len) deltas += (len + 3) & ~3;
    }
    std::stable_sort(longs.begin(), longs.end(),
                     [&](int32_t x, int32_t y) { return h_len[x] > h_len[y]; });
    for (const int32_t i : longs) {
      hubs.push_back(Tile{at, -1, (int)hub_nnz, (int)hub_nnz + h_len[i]});
      h_order[at++] = i;
      hub_nnz += h_len[i];
    }
    p->slice_begin.push_back((int)slices.size());
    p->hub_begin.push_back((int)hubs.size());
  }
  p->hub_nnz = hub_nnz;
  const int n_sl = (int)slices.size();
  rc = p->slices.alloc(sizeof(Slice) * std::max<size_t>(slices.size(), 1));
  if (!rc) rc = p->delta.alloc(4 * (size_t)std::max<int64_t>(deltas, 1));
  if (!rc) rc = p->hubs.alloc(sizeof(Tile) * std::max<size_t>(hubs.size(), 1));
  if (!rc) rc = p->col.alloc(4 * (size_t)std::max<int64_t>(hub_nnz, 1));
  if (!rc) rc = p->val.alloc(4 * (size_t)std::max<int64_t>(hub_nnz, 1));
  if (rc) return rc;
  if (n_p > 0) {
    GD_HIP_TRY(hipMemcpyAsync(order.ptr, h_order.data(), 4 * (size_t)n_p, hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(sg_rec_kernel, dim3(sg_grid(n_p)), dim3(256), 0, s, n_p,
                       order.as<int32_t>(), idx, len.as<int32_t>(), diag.as<float>(),
                       p->rows.as<RowRec>());
  }
  if (n_sl > 0) {
    const size_t bytes = sizeof(Slice) * slices.size();
    const dim3 grid(sg_grid((int64_t)n_sl * kWave));
    GD_HIP_TRY(hipMemcpyAsync(p->slices.ptr, slices.data(), bytes, hipMemcpyHostToDevice, s));
    GD_HIP_TRY(hipMemsetAsync(p->delta.ptr, 0, 4 * (size_t)std::max<int64_t>(deltas, 1), s));
    hipLaunchKernelGGL(sg_uniform_kernel, grid, dim3(256), 0, s, n_sl, p->slices.as<Slice>(),
                       p->rows.as<RowRec>(), d_Ap, d_Aj, d_Ax, p->delta.as<int>());
    GD_HIP_TRY(hipGetLastError());
    GD_HIP_TRY(hipMemcpyAsync(slices.data(), p->slices.ptr, bytes, hipMemcpyDeviceToHost, s));
    GD_HIP_TRY(hipStreamSynchronize(s));
    int64_t at = 0;
    for (Slice& sl : slices) {
      sl.n = sl.delta >= 0 ? (sl.len + 3) / 4 : (sl.len + 1) / 2;
      sl.off = at;
      at += (int64_t)sl.n * sl.n_rows;
    }
    rc = p->ent.alloc(sizeof(int4) * (size_t)std::max<int64_t>(at, 1));
    if (rc) return rc;
    GD_HIP_TRY(hipMemcpyAsync(p->slices.ptr, slices.data(), bytes, hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(sg_slice_fill_kernel, grid, dim3(256), 0, s, n_sl, p->slices.as<Slice>(),
                       p->rows.as<RowRec>(), d_Ap, d_Aj, d_Ax, p->ent.as<int4>());
  }
  if (!hubs.empty()) {
    GD_HIP_TRY(hipMemcpyAsync(p->hubs.ptr, hubs.data(), sizeof(Tile) * hubs.size(),
                              hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(sg_hub_fill_kernel, dim3(sg_grid((int64_t)hubs.size())), dim3(256), 0, s,
                       (int)hubs.size(), p->hubs.as<Tile>(), p->rows.as<RowRec>(), d_Ap, d_Aj,
                       d_Ax, p->col.as<int32_t>(), p->val.as<float>());
  }
  GD_HIP_TRY(hipGetLastError());
  GD_HIP_TRY(hipStreamSynchronize(s));  // host vectors and scratch go out of scope
  return GD_OK;
}

// One color: one launch of symgs_color_kernel on s.
int sweep_color(gd_symgs_plan* p, int c, float* x, const float* b, hipStream_t s) {
  const int s0 = p->slice_begin[c], ns = p->slice_begin[c + 1] - s0;
  const int h0 = p->hub_begin[c], nh = p->hub_begin[c + 1] - h0;
  const SymgsArgs a{x,
                    b,
                    p->rows.as<RowRec>(),
                    p->slices.as<Slice>() + s0,
                    ns,
                    p->ent.as<int4>(),
                    p->delta.as<int>(),
                    p->hubs.as<Tile>() + h0,
                    nh,
                    p->col.as<int32_t>(),
                    p->val.as<float>(),
                    (int)std::max<int64_t>(p->hub_nnz - 1, 0)};
  constexpr int per = kBlock / kWave;
  if (nh > 0)
    hipLaunchKernelGGL(symgs_long_kernel, dim3((ns + per - 1) / per + nh), dim3(kBlock), 0, s, a);
  else if (ns > 0)
    hipLaunchKernelGGL(symgs_color_kernel, dim3(ns), dim3(kWave), 0, s, a);
  GD_HIP_TRY(hipGetLastError());
  return GD_OK;
}

}  // namespace

extern "C" {

int gd_symgs_plan_create(int m, int64_t nnz, const int32_t* d_Ap, const int32_t* d_Aj,
                         const float* d_Ax, const int32_t* d_indices,
                         const int32_t* color_offsets, int n_colors, void* stream,
                         gd_symgs_plan** out) {
  GD_CHECK_ARG(out != nullptr, "NULL plan output");
  *out = nullptr;
  GD_CHECK_ARG(m >= 0 && nnz >= 0 && nnz < (1ll << 31), "m / nnz out of range");
  GD_CHECK_ARG(n_colors >= 0 && color_offsets != nullptr, "NULL color offsets");
  GD_CHECK_ARG(d_Ap != nullptr && (nnz == 0 || (d_Aj && d_Ax)), "NULL matrix array");
  for (int c = 0; c < n_colors; c++)
    GD_CHECK_ARG(color_offsets[c] <= color_offsets[c + 1], "color offsets must be non-decreasing");
  GD_CHECK_ARG(color_offsets[0] >= 0 && color_offsets[n_colors] <= m,
               "color offsets must lie in [0, m]");
  GD_CHECK_ARG(d_indices != nullptr || color_offsets[n_colors] == color_offsets[0],
               "NULL indices");
  if (gd_device_count() <= 0) {
    set_error("no HIP device visible");
    return GD_ERR_NO_DEVICE;
  }
  const auto t0 = std::chrono::steady_clock::now();
  gd_symgs_plan* p = new (std::nothrow) gd_symgs_plan;
  if (!p) return GD_ERR_ALLOC;
  const int rc = plan_build(p, m, nnz, d_Ap, d_Aj, d_Ax, d_indices, color_offsets, n_colors,
                            (hipStream_t)stream);
  if (rc) {
    delete p;
    return rc;
  }
  p->plan_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0)
                   .count();
  *out = p;
  return GD_OK;
}

int gd_symgs_plan_run(gd_symgs_plan* p, float* d_x, const float* d_b, int sweeps, void* stream) {
  GD_CHECK_ARG(p != nullptr, "NULL plan");
  GD_CHECK_ARG(sweeps >= 0, "negative sweep count");
  GD_CHECK_ARG(p->n_p == 0 || (d_x && d_b), "NULL x / b");
  hipStream_t s = (hipStream_t)stream;
  for (int k = 0; k < sweeps; k++) {
    for (int c = 0; c < p->n_colors; c++) {
      const int rc = sweep_color(p, c, d_x, d_b, s);
      if (rc) return rc;
    }
    for (int c = p->n_colors - 1; c >= 0; c--) {
      const int rc = sweep_color(p, c, d_x, d_b, s);
      if (rc) return rc;
    }
  }
  return GD_OK;
}

int gd_symgs_plan_info(const gd_symgs_plan* p, gd_symgs_plan_info_t* info) {
  GD_CHECK_ARG(p != nullptr && info != nullptr, "NULL argument");
  memset(info, 0, sizeof(*info));
  info->rows = p->n_p;
  info->offdiag_nnz = p->nnz_p;
  info->n_colors = p->n_colors;
  info->n_tiles = p->slice_begin.back();
  info->n_exact_rows = p->hub_begin.back();
  info->max_row_len = p->max_row_len;
  info->plan_ms = p->plan_ms;
  return GD_OK;
}

int gd_symgs_plan_destroy(gd_symgs_plan* p) {
  delete p;
  return GD_OK;
}

int gd_symgs_solve(int m, int nnz, const int32_t* Ap, const int32_t* Aj, const int32_t* indices,
                   const float* Ax, float* x, const float* b, const int32_t* color_offsets,
                   int n_colors, float* kernel_ms) {
  GD_CHECK_ARG(m >= 0 && nnz >= 0, "negative size");
  GD_CHECK_ARG(Ap != nullptr && (m == 0 || (x && b && indices)), "NULL host array");
  GD_CHECK_ARG(nnz == 0 || (Aj && Ax), "NULL column indices / values");
  if (gd_device_count() <= 0) {
    set_error("no HIP device visible");
    return GD_ERR_NO_DEVICE;
  }
  DeviceBuffer dAp, dAj, dAx, didx, dx, db;
  int rc = dAp.alloc(4 * ((size_t)m + 1));
  if (!rc) rc = dAj.alloc(4 * (size_t)nnz);
  if (!rc) rc = dAx.alloc(4 * (size_t)nnz);
  if (!rc) rc = didx.alloc(4 * (size_t)m);
  if (!rc) rc = dx.alloc(4 * (size_t)m);
  if (!rc) rc = db.alloc(4 * (size_t)m);
  if (rc) return rc;
  GD_HIP_TRY(hipMemcpy(dAp.ptr, Ap, 4 * ((size_t)m + 1), hipMemcpyHostToDevice));
  if (m > 0) {
    GD_HIP_TRY(hipMemcpy(didx.ptr, indices, 4 * (size_t)m, hipMemcpyHostToDevice));
    GD_HIP_TRY(hipMemcpy(dx.ptr, x, 4 * (size_t)m, hipMemcpyHostToDevice));
    GD_HIP_TRY(hipMemcpy(db.ptr, b, 4 * (size_t)m, hipMemcpyHostToDevice));
  }
  if (nnz > 0) {
    GD_HIP_TRY(hipMemcpy(dAj.ptr, Aj, 4 * (size_t)nnz, hipMemcpyHostToDevice));
    GD_HIP_TRY(hipMemcpy(dAx.ptr, Ax, 4 * (size_t)nnz, hipMemcpyHostToDevice));
  }
  gd_symgs_plan* plan = nullptr;
  rc = gd_symgs_plan_create(m, nnz, dAp.as<int32_t>(), dAj.as<int32_t>(), dAx.as<float>(),
                            didx.as<int32_t>(), color_offsets, n_colors, nullptr, &plan);
  if (rc) return rc;
  EventPair evp;
  GD_HIP_TRY(evp.create());
  hipEvent_t t0 = evp.a, t1 = evp.b;
  GD_HIP_TRY(hipEventRecord(t0, nullptr));
  rc = gd_symgs_plan_run(plan, dx.as<float>(), db.as<float>(), 1, nullptr);
  GD_HIP_TRY(hipEventRecord(t1, nullptr));
  GD_HIP_TRY(hipEventSynchronize(t1));
  float ms = 0.0f;
  GD_HIP_TRY(hipEventElapsedTime(&ms, t0, t1));
  if (kernel_ms) *kernel_ms = ms;
  gd_symgs_plan_destroy(plan);
  if (rc) return rc;
  if (m > 0) GD_HIP_TRY(hipMemcpy(x, dx.ptr, 4 * (size_t)m, hipMemcpyDeviceToHost));
  return GD_OK;
}

}  // extern "C"
