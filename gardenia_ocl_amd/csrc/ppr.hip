// ppr.hip -- batched personalised PageRank (k seeds at once), gfx950.
//
// The same pull iteration as pr.hip, k columns wide: column j teleports its
// (1-d) mass to seed vertex seeds[j] instead of (1-d)/m to every vertex.
// Scores are stored vertex-major with the k seeds of a vertex contiguous
// (X[v*k + j]).  The columns are taken in groups of 32, one 128-byte line of a
// vertex's k-vector: 8 lanes gather an edge's line and each adds its 4 columns.
//
// Each column of every row is summed sequentially in CSR order, the scalar
// personalised loop's order and FP32 rounding, so every column is the
// single-seed run's bit for bit.  Rows longer than kHubEdges (hubs) run
// beside the tiles: one workgroup per (hub row, column group), three waves
// gathering chunks of the row into LDS while the fourth adds them in edge
// order, one column per lane.  Rows without in-edges keep their first score
// and run in two iterations only.  The per-iteration update is base + d*sum
// with two roundings (built with -ffp-contract=off).
//
// A persistent grid of workgroups walks the tile list; each workgroup keeps
// per-column L1 partials for the whole sweep, and one small kernel reduces
// them (deterministically) to per-column L1 values, their maximum and the
// convergence flag.
//
// Columns stop one by one: after the first iteration whose L1 change of
// column j is below tol, column j is frozen (its scores are final, exactly as
// a single-seed run would stop).  Frozen columns keep their values; between
// host checks the running columns are moved to the front of every vertex's
// k-vector (an in-place column permutation of X and the gathered contrib), so
// the lanes of frozen columns stop gathering.  The permutation is undone when
// the run ends.

#include <hip/hip_runtime.h>

#include <rocprim/device/device_scan.hpp>
#include <rocprim/iterator/counting_iterator.hpp>
#include <rocprim/iterator/transform_iterator.hpp>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "gardenia_hip.h"
#include "gd_common.h"
#include "relabel.h"

namespace gd {

namespace {

constexpr int kPBlock = 256;
constexpr int kPWaves = kPBlock / 64;
constexpr int kGroup = 32;        // columns per group: one 128-byte line of a vertex's k-vector
constexpr int kSub = 8;           // lanes that walk one row: 4 columns each
constexpr int kSubs = kPBlock / kSub;
constexpr int kHubEdges = 1024;   // rows longer than this are hubs (ppr_hub_chain_kernel)
constexpr int kTileEdges = 256;   // edges per tile, at most (one tile: one 16-lane subgroup)
constexpr int kMinTileEdges = 32;
constexpr int kMaxSlots = 2048;   // workgroups that sweep one column group
constexpr int kEmptySlots = 256;  // workgroups per column group in ppr_empty_kernel
constexpr int kRedSplits = 16;    // workgroups per column group in ppr_reduce_kernel

struct PprState {
  int iter;
  int done;
  int max_iter;
  unsigned ticket;  // ppr_reduce_kernel workgroups arrived in this iteration
  double tol;
};

typedef float f4 __attribute__((ext_vector_type(4)));

// score / outdeg, correctly rounded, from inv = 1 / outdeg in FP64.  The FP64
// product is within 2^-52 of the quotient of two 24-bit numbers, which is never
// closer than 2^-49 to a midpoint of two normal floats (a - m*d is a nonzero
// integer over m*d < 2^49), so it rounds to the same float as the IEEE division,
// at a third of its instructions.  Subnormal results may lie on a midpoint:
// they are divided.
__device__ __forceinline__ float div_outdeg(float a, double inv, const int32_t* outdeg) {
  const float q = (float)((double)a * inv);
  if (fabsf(q) < 0x1p-125f && a != 0.0f) return a / (float)*outdeg;
  return q;
}

// This lane's 4 columns of a vertex.
struct Lane {
  int seed[4];
  bool fz[4];  // frozen columns keep their score
  double err[4];

  __device__ __forceinline__ Lane(const int32_t* __restrict__ seeds,
                                  const int32_t* __restrict__ frozen, int col0) {
#pragma unroll
    for (int j = 0; j < 4; j++) {
      seed[j] = seeds[col0 + j];
      fz[j] = frozen[col0 + j] != 0;
      err[j] = 0.0;
    }
  }

  // X[o..] <- the new scores of row r, Cn[o..] <- their contributions (iv NaN:
  // nothing gathers this vertex), err += |change| (not read where frozen).
  __device__ __forceinline__ void update(int r, f4 sum, f4 old, double iv,
                                         const int32_t* __restrict__ outdeg, float teleport,
                                         float damp, float* __restrict__ X,
                                         float* __restrict__ Cn, int64_t o) {
    f4 nx;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const float b = seed[j] == r ? teleport : 0.0f;
      const float upd = b + damp * sum[j];
      nx[j] = fz[j] ? old[j] : upd;
      err[j] += (double)fabsf(nx[j] - old[j]);
    }
    __builtin_nontemporal_store(nx, reinterpret_cast<f4*>(X + o));
    if (iv == iv) {
      f4 nc;
#pragma unroll
      for (int j = 0; j < 4; j++) nc[j] = div_outdeg(nx[j], iv, outdeg + r);
      __builtin_nontemporal_store(nc, reinterpret_cast<f4*>(Cn + o));
    }
  }

  // The workgroup's partial per column: subgroups in order, through LDS.
  __device__ __forceinline__ void store_err(double* __restrict__ part) const {
    __shared__ double s_err[kSubs][kGroup];
    const int lane = threadIdx.x & (kSub - 1), sub = threadIdx.x / kSub;
#pragma unroll
    for (int j = 0; j < 4; j++) s_err[sub][4 * lane + j] = err[j];
    __syncthreads();
    if (threadIdx.x < kGroup) {
      double s = 0.0;
#pragma unroll
      for (int w = 0; w < kSubs; w++) s += s_err[w][threadIdx.x];
      part[threadIdx.x] = s;
    }
  }
};

// Rows without in-edges.  Their score is the teleport from the first iteration
// on, so they run in the first two (X and both contribution buffers), and once
// after the columns were permuted (the buffer that was not).
__global__ __launch_bounds__(kPBlock) void ppr_empty_kernel(
    const int32_t* __restrict__ rows, int n_rows, const int32_t* __restrict__ outdeg,
    const double* __restrict__ inv, const int32_t* __restrict__ seeds,
    const int32_t* __restrict__ frozen, int64_t k, float* __restrict__ X, float* __restrict__ C0,
    float* __restrict__ C1, double* __restrict__ err_part, const PprState* __restrict__ st,
    float teleport, float damp) {
  if (st->done) return;
  float* __restrict__ Cn = (st->iter & 1) ? C0 : C1;
  const int lane = threadIdx.x & (kSub - 1), sub = threadIdx.x / kSub;
  const int col0 = blockIdx.y * kGroup + 4 * lane;
  Lane me(seeds, frozen, col0);
  for (int i = blockIdx.x * kSubs + sub; i < n_rows; i += gridDim.x * kSubs) {
    const int r = rows[i];
    const int64_t o = (int64_t)r * k + col0;
    const f4 old = *reinterpret_cast<const f4*>(X + o);
    me.update(r, (f4){0.0f, 0.0f, 0.0f, 0.0f}, old, inv[r], outdeg, teleport, damp, X, Cn, o);
  }
  me.store_err(err_part + (int64_t)blockIdx.x * k + blockIdx.y * kGroup);
}

// Rows of 1 to kHubEdges edges.  An 8-lane subgroup walks the rows of a tile
// for one group of 32 columns (lane l: columns 4l .. 4l+3 of the group), 8 edges
// of one row in flight, each column added in edge order by its lane.  The ids of
// the next 8 edges are loaded a step ahead, by one lane each.  Edges past the
// row's end read vertex m, whose contributions are -0.0: they add nothing.
//
// Bound: bytes that miss the L2.  A column group is swept over all rows before
// the next one starts (gp groups at a time, each on 8/gp XCDs), so an XCD's 4 MB
// L2 holds the 32 columns of 4 times as many of the often gathered vertices as
// a sweep with 128 columns per edge did, and the Infinity Cache most of a
// group's.  Per iteration of 0.7 M vertices, 10.5 M edges, 128 columns (rows of
// up to 1024 edges): 462 us alone, 2.4 GB read past the L2; beside the hubs 500
// us against 890 before.  With 16 lanes of 2 columns and masked loads it was 704
// us: 241 M vector instructions against 73 M.  Gathers of rarely used vertices
// marked non-temporal miss the L2 less (2.0 GB) but are slower (594 us): they
// pass by the Infinity Cache, too.
__global__ __launch_bounds__(kPBlock) void ppr_pull_kernel(
    const Tile* __restrict__ tiles, int n_tiles, int m, const int2* __restrict__ rows,
    const int32_t* __restrict__ col, const int32_t* __restrict__ outdeg,
    const double* __restrict__ inv, const int32_t* __restrict__ seeds,
    const int32_t* __restrict__ frozen, int ka, int64_t k, int gp_log2, float* __restrict__ X,
    float* __restrict__ C0, float* __restrict__ C1, double* __restrict__ err_part,
    const PprState* __restrict__ st, float teleport, float damp) {
  if (st->done) return;
  const int xcd = blockIdx.x & 7;  // workgroups go to the XCDs in turn
  const int grp = (blockIdx.y << gp_log2) + (xcd & ((1 << gp_log2) - 1));
  if (grp * kGroup >= ka) return;
  const int slot = (blockIdx.x >> 3) * (8 >> gp_log2) + (xcd >> gp_log2);
  const int slots = gridDim.x >> gp_log2;
  const float* __restrict__ C = (st->iter & 1) ? C1 : C0;
  float* __restrict__ Cn = (st->iter & 1) ? C0 : C1;
  const int lane = threadIdx.x & (kSub - 1), sub = threadIdx.x / kSub;
  const int first = (threadIdx.x & 63 & ~(kSub - 1)) * 4;  // ds_bpermute address of lane 0
  const int col0 = grp * kGroup + 4 * lane;
  const float* __restrict__ Cc = C + col0;
  Lane me(seeds, frozen, col0);
  for (int t = slot * kSubs + sub; t < n_tiles; t += slots * kSubs) {
    const Tile tl = tiles[t];
    int at = tl.x, i = tl.z;
    int2 row = rows[at];  // vertex, end of its edges
    int32_t id = i + lane < tl.w ? col[i + lane] : m;
    f4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    while (at < tl.y) {  // every step ends a row or takes 8 edges of it
      const int n = row.y - i;
      const bool last = n <= kSub;
      const int mine = lane < n ? id : m;
      f4 g[kSub];
#pragma unroll
      for (int q = 0; q < kSub; q++) {
        const uint32_t u = (uint32_t)__builtin_amdgcn_ds_bpermute(first + 4 * q, mine);
        g[q] = *reinterpret_cast<const f4*>(Cc + (uint64_t)u * (uint32_t)k);
      }
      i += min(n, kSub);
      id = i + lane < tl.w ? col[i + lane] : m;
      f4 old = acc;
      double iv = 0.0;
      int2 next = row;
      const int64_t o = (int64_t)row.x * k + col0;
      if (last) {
        old = __builtin_nontemporal_load(reinterpret_cast<const f4*>(X + o));
        iv = inv[row.x];
        if (at + 1 < tl.y) next = rows[at + 1];
      }
#pragma unroll
      for (int q = 0; q < kSub; q++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[j] += g[q][j];
      if (last) {
        me.update(row.x, acc, old, iv, outdeg, teleport, damp, X, Cn, o);
        acc = (f4){0.0f, 0.0f, 0.0f, 0.0f};
        row = next;
        at++;
      }
    }
  }
  me.store_err(err_part + (int64_t)slot * k + grp * kGroup);
}

// Hub rows: workgroup b adds hub row hub_row[b / groups] for the COLS columns
// (gd_ppr_plan_config.hub_cols) of group b % groups, longest row first, in edge
// order.  Waves 1..3 gather 16 bytes a lane, 16 instructions in flight each, so
// a chunk is 48 KB (384 edges of 32 columns); lane c < COLS of wave 0 adds
// column c of the chunk from LDS while the next one is in flight.  One LDS
// buffer: the gathered chunk waits in registers until the adds are done.
// Rows are cut at 1024 edges: at 512 or 2048 an iteration takes 7 or 11
// percent longer.  98 rows of more than 4096 edges alone took 890 us with 96
// edges of 64 columns in flight; 1224 of more than 1024 take 284 us.
// hub_err row b / groups receives the row's per-column |change|.
constexpr int kHubLoads = 16;  // gathering instructions per wave per chunk

template <int COLS>  // columns per workgroup: 16, 32 or 64
__global__ __launch_bounds__(kPBlock) void ppr_hub_chain_kernel(
    const int32_t* __restrict__ hub_row, int groups, const int32_t* __restrict__ off,
    const int32_t* __restrict__ col, const int32_t* __restrict__ outdeg,
    const int32_t* __restrict__ seeds, const int32_t* __restrict__ frozen, int ka, int64_t k,
    float* __restrict__ X, float* __restrict__ C0, float* __restrict__ C1,
    double* __restrict__ hub_err, const PprState* __restrict__ st, float teleport, float damp) {
  constexpr int kLanes = COLS / 4;           // lanes per edge
  constexpr int kEpi = 64 / kLanes;          // edges per gathering instruction
  constexpr int kEdgesW = kHubLoads * kEpi;  // edges per gathering wave per chunk
  constexpr int kChunkE = 3 * kEdgesW;       // edges per chunk
  constexpr int kIdRegs = kEdgesW / 64;
  if (st->done) return;
  __shared__ float buf[kChunkE * COLS];
  const float* __restrict__ C = (st->iter & 1) ? C1 : C0;
  float* __restrict__ Cn = (st->iter & 1) ? C0 : C1;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = blockIdx.x / groups;
  const int g0 = (blockIdx.x % groups) * COLS;  // first column of the group (< k)
  const int row = hub_row[h];
  const int e0 = off[row];
  const int ne = off[row + 1] - e0;
  const int nchunks = (ne + kChunkE - 1) / kChunkE;
  const int gw = wid - 1;  // gathering wave 0..2
  const float* __restrict__ Cc = C + g0 + 4 * (lane % kLanes);
  int32_t ids[kIdRegs];
  f4 v[kHubLoads];
  // source ids of this wave's edges of chunk c: lane l holds edge l + 64 q; 0
  // (a valid vertex) past the row
  auto load_ids = [&](int c) {
#pragma unroll
    for (int q = 0; q < kIdRegs; q++) {
      const int e = c * kChunkE + gw * kEdgesW + q * 64 + lane;
      ids[q] = e < ne ? col[e0 + e] : 0;
    }
  };
  auto gather = [&]() {
#pragma unroll
    for (int i = 0; i < kHubLoads; i++) {
      const int e = i * kEpi + lane / kLanes;  // this lane's edge in the wave's part
      const uint32_t u = (uint32_t)__shfl(ids[(i * kEpi) / 64], e % 64, 64);
      v[i] = *reinterpret_cast<const f4*>(Cc + (uint64_t)u * (uint32_t)k);
    }
  };
  float s = 0.0f;
  if (wid != 0) {
    load_ids(0);
    gather();
    load_ids(1);
  }
  for (int c = 0; c < nchunks; c++) {
    if (wid != 0) {
      f4* dst = reinterpret_cast<f4*>(buf) + gw * kHubLoads * 64 + lane;
#pragma unroll
      for (int i = 0; i < kHubLoads; i++) dst[i * 64] = v[i];
    }
    __syncthreads();
    if (wid != 0) {
      if (c + 1 < nchunks) gather();
      load_ids(c + 2);
    } else if (lane < COLS) {
      const float* __restrict__ b = buf + lane;
      const int nc = min(kChunkE, ne - c * kChunkE);
      int e = 0;
      if (nc >= 16) {
        float a[16];
#pragma unroll
        for (int q = 0; q < 16; q++) a[q] = b[q * COLS];
        for (; e + 32 <= nc; e += 16) {  // the next 16 terms are read ahead of the adds
          float nx[16];
#pragma unroll
          for (int q = 0; q < 16; q++) nx[q] = b[(e + 16 + q) * COLS];
#pragma unroll
          for (int q = 0; q < 16; q++) s += a[q];
#pragma unroll
          for (int q = 0; q < 16; q++) a[q] = nx[q];
        }
#pragma unroll
        for (int q = 0; q < 16; q++) s += a[q];
        e += 16;
      }
      for (; e < nc; e++) s += b[e * COLS];
    }
    __syncthreads();
  }
  if (wid == 0 && lane < COLS) {
    const int my_col = g0 + lane;
    double err = 0.0;
    if (my_col < ka) {
      const int64_t o = (int64_t)row * k + my_col;
      const float old = X[o];
      const float b = seeds[my_col] == row ? teleport : 0.0f;
      const float upd = b + damp * s;
      const float nx = frozen[my_col] ? old : upd;
      X[o] = nx;
      Cn[o] = nx / (float)outdeg[row];
      err = (double)fabsf(nx - old);
    }
    hub_err[(int64_t)h * k + my_col] = err;
  }
}

// Per-column L1 of one iteration: workgroup (g, s) adds column group g's rows
// r = s mod kRedSplits of the partials (err_part's `slots`, then hub_err's
// `hubs`) in a fixed order; the last workgroup to arrive adds the splits of the
// columns still running (c < kact, not frozen), takes their maximum, stops the
// columns whose change is below tol (column_stop) and advances the state.
__global__ __launch_bounds__(kPBlock) void ppr_reduce_kernel(
    const double* __restrict__ err_part, int slots, const double* __restrict__ hub_err, int hubs,
    int64_t k, int kact, double* __restrict__ fin, double* __restrict__ col_err,
    int32_t* __restrict__ frozen, int32_t* __restrict__ col_iters, int column_stop,
    PprState* __restrict__ st, double* __restrict__ errors) {
  if (st->done) return;
  constexpr int kParts = kPBlock / kGroup;
  __shared__ double s_part[kParts][kGroup];
  __shared__ double s_max[kPBlock];
  __shared__ unsigned s_last;
  const int it = st->iter;
  const double tol = st->tol;
  const int lc = threadIdx.x % kGroup, part = threadIdx.x / kGroup;
  const int64_t c0 = (int64_t)blockIdx.x * kGroup + lc;
  double s = 0.0;
#pragma unroll 4
  for (int r = blockIdx.y * kParts + part; r < slots; r += kRedSplits * kParts)
    s += err_part[(int64_t)r * k + c0];
#pragma unroll 4
  for (int r = blockIdx.y * kParts + part; r < hubs; r += kRedSplits * kParts)
    s += hub_err[(int64_t)r * k + c0];
  s_part[part][lc] = s;
  __syncthreads();
  if (part == 0) {
    s = 0.0;
#pragma unroll
    for (int q = 0; q < kParts; q++) s += s_part[q][lc];
    fin[(int64_t)blockIdx.y * k + c0] = s;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    __threadfence();  // release fin before taking a ticket
    s_last = atomicAdd(&st->ticket, 1u) + 1 == gridDim.x * gridDim.y;
  }
  __syncthreads();
  if (!s_last) return;
  __threadfence();  // acquire: every workgroup's fin is visible
  double mx = 0.0;
  for (int c = threadIdx.x; c < kact; c += kPBlock) {
    if (frozen[c]) continue;
    double t = 0.0;
#pragma unroll
    for (int q = 0; q < kRedSplits; q++) t += fin[(int64_t)q * k + c];
    col_err[c] = t;
    col_iters[c] = it + 1;
    mx = fmax(mx, t);
    if (column_stop && t < tol) frozen[c] = 1;
  }
  s_max[threadIdx.x] = mx;
  __syncthreads();
  for (int w = kPBlock / 2; w > 0; w >>= 1) {
    if (threadIdx.x < w) s_max[threadIdx.x] = fmax(s_max[threadIdx.x], s_max[threadIdx.x + w]);
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    errors[it] = s_max[0];
    st->ticket = 0;
    st->iter = it + 1;
    // every running column below tol <=> the max over them is
    if (s_max[0] < tol || it + 1 >= st->max_iter) st->done = 1;
  }
}

__global__ void ppr_reset_cols_kernel(int k, int32_t* __restrict__ frozen,
                                      int32_t* __restrict__ col_iters) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j < k) {
    frozen[j] = 0;
    col_iters[j] = 0;
  }
}

// In-place column permutation of the rows of A (and of B when not NULL):
// row[c] <- row[newcol[c]] for c < kact, newcol a permutation of [0, kact).
// One wavefront per row through kact floats of LDS; every workgroup runs the
// same number of loop trips, so the barriers are uniform.
__global__ __launch_bounds__(kPBlock) void ppr_permute_cols_kernel(int m, int64_t k, int kact,
                                                                   const int32_t* __restrict__ newcol,
                                                                   float* __restrict__ A,
                                                                   float* __restrict__ B) {
  extern __shared__ float s_rows[];  // kPWaves * kact
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  float* my = s_rows + (size_t)wid * kact;
  const int passes = B ? 2 : 1;
  for (int base = blockIdx.x * kPWaves; base < m; base += gridDim.x * kPWaves) {
    const int v = base + wid;
    for (int pass = 0; pass < passes; pass++) {
      float* row = (pass ? B : A) + (int64_t)min(v, m - 1) * k;
      if (v < m)
        for (int c = lane; c < kact; c += 64) my[c] = row[c];
      __syncthreads();
      if (v < m)
        for (int c = lane; c < kact; c += 64) row[c] = my[newcol[c]];
      __syncthreads();
    }
  }
}

__global__ void ppr_mark_sources_kernel(int64_t nnz, const int32_t* __restrict__ col,
                                        uint8_t* __restrict__ mark) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nnz;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int u = col[i];
    if (!mark[u]) mark[u] = 1;
  }
}

// inv: 1 / outdeg in FP64, NaN for a vertex that no edge leaves; and vertex m's
// contributions of -0.0
__global__ void ppr_inv_kernel(int m, int k, const int32_t* __restrict__ outdeg,
                               const uint8_t* __restrict__ mark,
                               double* __restrict__ inv, float* __restrict__ C0,
                               float* __restrict__ C1) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v < m) inv[v] = mark[v] ? 1.0 / (double)(float)outdeg[v] : __builtin_nan("");
  if (v < k) C0[(int64_t)m * k + v] = C1[(int64_t)m * k + v] = -0.0f;
}

struct HasEdges {
  const int32_t* off;
  __device__ int operator()(int r) const { return off[r + 1] > off[r]; }
};

// Rows with edges to rows / ends, the others to empty, in order: at[r] rows with
// edges come before r.
__global__ void ppr_split_rows_kernel(int m, const int32_t* __restrict__ off,
                                      const int32_t* __restrict__ at, int2* __restrict__ rows,
                                      int32_t* __restrict__ ends, int32_t* __restrict__ empty) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= m) return;
  const int e = off[r + 1];
  if (e > off[r]) {
    rows[at[r]] = make_int2(r, e);
    ends[at[r]] = e;
  } else {
    empty[r - at[r]] = r;
  }
}

__global__ void ppr_hub_vertex_kernel(int n, const int2* __restrict__ rows,
                                      int32_t* __restrict__ hub_row) {
  const int h = blockIdx.x * blockDim.x + threadIdx.x;
  if (h < n) hub_row[h] = rows[hub_row[h]].x;
}

__global__ void ppr_init_kernel(int64_t n, int64_t k, const float* __restrict__ X,
                                const int32_t* __restrict__ outdeg, float* __restrict__ C0,
                                PprState* __restrict__ st, int max_iter, double tol) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    C0[i] = X[i] / (float)outdeg[i / k];
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    st->iter = 0;
    st->done = max_iter <= 0;
    st->max_iter = max_iter;
    st->ticket = 0;
    st->tol = tol;
  }
}

// rows of X between the user's vertex order and the plan's; on the way back
// (cperm not NULL) internal column j goes to user column cperm[j]
__global__ void ppr_permute_rows_kernel(int m, int64_t k, const int32_t* __restrict__ perm,
                                        const int32_t* __restrict__ cperm,
                                        const float* __restrict__ src, float* __restrict__ dst,
                                        int to_internal) {
  const int lane = threadIdx.x & 63;
  for (int i = blockIdx.x * (blockDim.x / 64) + threadIdx.x / 64; i < m;
       i += gridDim.x * (blockDim.x / 64)) {
    const int v = perm[i];
    const float* s = src + (int64_t)(to_internal ? v : i) * k;
    float* d = dst + (int64_t)(to_internal ? i : v) * k;
    for (int64_t j = lane; j < k; j += 64) d[cperm ? cperm[j] : j] = s[j];
  }
}

__global__ void ppr_map_seeds_kernel(int k, const int32_t* __restrict__ seeds,
                                     const int32_t* __restrict__ inv, int32_t* __restrict__ out) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j < k) out[j] = inv ? inv[seeds[j]] : seeds[j];
}

__global__ void check_seeds_kernel(int k, const int32_t* __restrict__ seeds, int m,
                                   int* __restrict__ bad) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j < k && (seeds[j] < 0 || seeds[j] >= m)) atomicOr(bad, 1);
}

}  // namespace

}  // namespace gd

using namespace gd;

struct gd_ppr_plan {
  int m = 0, k = 0;
  int kc = kGroup;         // columns swept at once
  int hub_cols = kGroup;   // columns per hub-row workgroup
  int64_t nnz = 0;
  hipStream_t stream = nullptr;
  bool relabel = false;
  const int32_t* off = nullptr;
  const int32_t* col = nullptr;
  const int32_t* outdeg = nullptr;
  Relabel rl;
  Schedule sched;
  int n_tiles = 0, n_hubs = 0, n_empty = 0, grid = 0;
  // hub rows run on the plan's stream beside the tiles on `side` (fork / join)
  hipStream_t side = nullptr;
  hipEvent_t fork_ev = nullptr, join_ev = nullptr;
  ~gd_ppr_plan() {
    if (fork_ev) (void)hipEventDestroy(fork_ev);
    if (join_ev) (void)hipEventDestroy(join_ev);
    if (side) (void)hipStreamDestroy(side);
  }
  DeviceBuffer tiles, rows, empty, hub_row, inv, err_part, hub_err, fin, col_err,
      C0, C1, Xint, seeds, state, errors, frozen, col_iters, newcol, cperm;
  int errors_cap = 0;
  bool column_stop = true;
  bool compact = true;
  std::vector<int32_t> last_col_iters;  // user column order
  float plan_ms = 0.0f;
};

namespace {

int ppr_build(gd_ppr_plan* p, const int32_t* d_off, const int32_t* d_col,
              const int32_t* d_outdeg) {
  const int m = p->m;
  int rc = check_columns(d_col, p->nnz, m, p->stream);
  if (rc) return rc;
  rc = check_offsets(d_off, m, p->nnz, p->stream);  // before any device walk
  if (rc) return rc;
  p->off = d_off;
  p->col = d_col;
  p->outdeg = d_outdeg;
  if (p->relabel) {
    rc = build_relabel(m, p->nnz, d_off, d_col, d_outdeg, p->stream, &p->rl);
    if (rc) return rc;
    p->off = p->rl.off.as<int32_t>();
    p->col = p->rl.col.as<int32_t>();
    p->outdeg = p->rl.outdeg.as<int32_t>();
  }
  // the rows with edges (vertex, end of its edges), and the others
  DeviceBuffer at, ends, tmp, mark;
  rocprim::transform_iterator<rocprim::counting_iterator<int>, HasEdges, int> flags(
      rocprim::counting_iterator<int>(0), HasEdges{p->off});
  size_t bytes = 0;
  GD_HIP_TRY(rocprim::exclusive_scan(nullptr, bytes, flags, (int32_t*)nullptr, 0, (size_t)m,
                                     rocprim::plus<int>(), p->stream));
  rc = at.alloc(4 * (size_t)m);
  if (!rc) rc = ends.alloc(4 * (size_t)m);
  if (!rc) rc = tmp.alloc(bytes);
  if (!rc) rc = mark.alloc((size_t)m);
  if (!rc) rc = p->rows.alloc(sizeof(int2) * (size_t)m);
  if (!rc) rc = p->empty.alloc(4 * (size_t)m);
  if (rc) return rc;
  GD_HIP_TRY(rocprim::exclusive_scan(tmp.ptr, bytes, flags, at.as<int32_t>(), 0, (size_t)m,
                                     rocprim::plus<int>(), p->stream));
  hipLaunchKernelGGL(ppr_split_rows_kernel, dim3((m + 255) / 256), dim3(256), 0, p->stream, m,
                     p->off, at.as<int32_t>(), p->rows.as<int2>(), ends.as<int32_t>(),
                     p->empty.as<int32_t>());
  GD_HIP_TRY(hipGetLastError());
  int32_t last[3];  // rows with edges before the last row, and its offsets
  GD_HIP_TRY(hipMemcpyAsync(last, at.as<int32_t>() + m - 1, 4, hipMemcpyDeviceToHost, p->stream));
  GD_HIP_TRY(hipMemcpyAsync(last + 1, p->off + m - 1, 8, hipMemcpyDeviceToHost, p->stream));
  GD_HIP_TRY(hipStreamSynchronize(p->stream));
  const int n_rows = last[0] + (last[2] > last[1] ? 1 : 0);
  p->n_empty = m - n_rows;
  std::vector<int32_t> row_off((size_t)n_rows + 1);  // edge offsets of the rows with edges
  row_off[0] = 0;
  if (n_rows)
    GD_HIP_TRY(hipMemcpyAsync(row_off.data() + 1, ends.ptr, 4 * (size_t)n_rows,
                              hipMemcpyDeviceToHost, p->stream));
  GD_HIP_TRY(hipStreamSynchronize(p->stream));
  // tiles: rows packed to tile_edges edges and a quarter as many rows, for each of
  // the kMaxSlots * kSubs subgroups of a sweep one or more; rows > kHubEdges are
  // hubs (ppr_hub_chain_kernel), longest first
  const int tile_edges = (int)std::max<int64_t>(
      kMinTileEdges, std::min<int64_t>(kTileEdges, p->nnz / (kMaxSlots * kSubs)));
  Schedule& s = p->sched;
  {
    Schedule packed;
    rc = build_schedule(n_rows, p->nnz, row_off.data(), tile_edges, tile_edges / 4, &packed);
    if (rc) return rc;
    s.max_row_len = packed.max_row_len;
    auto len = [&](int32_t i) { return row_off[i + 1] - row_off[i]; };
    std::stable_sort(packed.hub_row.begin(), packed.hub_row.end(),
                     [&](int32_t a, int32_t b) { return len(a) > len(b); });
    // heaviest work first: single rows of (tile_edges, kHubEdges] edges, then
    // the packed row tiles
    for (const int32_t i : packed.hub_row) {
      if (len(i) > kHubEdges)
        s.hub_row.push_back(i);  // its vertex below
      else
        s.tiles.push_back(Tile{i, i + 1, row_off[i], row_off[i + 1]});
    }
    for (const Tile& t : packed.tiles)
      if (t.y >= 0) s.tiles.push_back(t);
  }
  p->n_tiles = (int)s.tiles.size();
  p->n_hubs = (int)s.hub_row.size();
  // a multiple of 8 workgroups per group, so that every XCD keeps its share
  p->grid = std::max(8, std::min(kMaxSlots, (p->n_tiles + kSubs * 8 - 1) / (kSubs * 8) * 8));
  const size_t mk = (size_t)m * p->k;
  rc = p->tiles.alloc(sizeof(Tile) * p->n_tiles);
  if (!rc) rc = p->hub_row.alloc(4 * (size_t)std::max(1, p->n_hubs));
  if (!rc) rc = p->err_part.alloc(8 * (size_t)(p->grid + kEmptySlots) * p->k);
  if (!rc) rc = p->hub_err.alloc(8 * (size_t)std::max(1, p->n_hubs) * p->k);
  if (!rc) rc = p->fin.alloc(8 * (size_t)kRedSplits * p->k);
  if (!rc) rc = p->col_err.alloc(8 * (size_t)p->k);
  if (!rc) rc = p->inv.alloc(8 * (size_t)m);
  if (!rc) rc = p->C0.alloc(4 * (mk + p->k));  // vertex m: edges past a row's end
  if (!rc) rc = p->C1.alloc(4 * (mk + p->k));
  if (!rc && p->relabel) rc = p->Xint.alloc(4 * mk);
  if (!rc) rc = p->seeds.alloc(4 * (size_t)p->k);
  if (!rc) rc = p->frozen.alloc(4 * (size_t)p->k);
  if (!rc) rc = p->col_iters.alloc(4 * (size_t)p->k);
  if (!rc) rc = p->newcol.alloc(4 * (size_t)p->k);
  if (!rc) rc = p->cperm.alloc(4 * (size_t)p->k);
  if (!rc) rc = p->state.alloc(sizeof(PprState));
  if (rc) return rc;
  GD_HIP_TRY(hipMemsetAsync(mark.ptr, 0, (size_t)m, p->stream));
  if (p->nnz)
    hipLaunchKernelGGL(ppr_mark_sources_kernel,
                       dim3((unsigned)std::min<int64_t>((p->nnz + 255) / 256, 16384)), dim3(256), 0,
                       p->stream, p->nnz, p->col, mark.as<uint8_t>());
  hipLaunchKernelGGL(ppr_inv_kernel, dim3((std::max(m, p->k) + 255) / 256), dim3(256), 0, p->stream,
                     m, p->k, p->outdeg, mark.as<uint8_t>(), p->inv.as<double>(), p->C0.as<float>(),
                     p->C1.as<float>());
  GD_HIP_TRY(hipGetLastError());
  if (p->n_tiles)
    GD_HIP_TRY(hipMemcpyAsync(p->tiles.ptr, s.tiles.data(), sizeof(Tile) * p->n_tiles,
                              hipMemcpyHostToDevice, p->stream));
  if (p->n_hubs) {
    GD_HIP_TRY(hipMemcpyAsync(p->hub_row.ptr, s.hub_row.data(), 4 * p->n_hubs,
                              hipMemcpyHostToDevice, p->stream));
    hipLaunchKernelGGL(ppr_hub_vertex_kernel, dim3((p->n_hubs + 255) / 256), dim3(256), 0,
                       p->stream, p->n_hubs, p->rows.as<int2>(), p->hub_row.as<int32_t>());
    GD_HIP_TRY(hipGetLastError());
    GD_HIP_TRY(hipStreamCreateWithFlags(&p->side, hipStreamNonBlocking));
    GD_HIP_TRY(hipEventCreateWithFlags(&p->fork_ev, hipEventDisableTiming));
    GD_HIP_TRY(hipEventCreateWithFlags(&p->join_ev, hipEventDisableTiming));
  }
  GD_HIP_TRY(hipStreamSynchronize(p->stream));
  return GD_OK;
}

template <int COLS>
void ppr_launch_hubs(gd_ppr_plan* p, float* X, PprState* st, float teleport, float damp, int ka,
                     int kact) {
  const int groups = (kact + COLS - 1) / COLS;
  hipLaunchKernelGGL(ppr_hub_chain_kernel<COLS>, dim3((unsigned)(p->n_hubs * groups)),
                     dim3(kPBlock), 0, p->stream, p->hub_row.as<int32_t>(), groups, p->off, p->col,
                     p->outdeg, p->seeds.as<int32_t>(), p->frozen.as<int32_t>(), ka,
                     (int64_t)p->k, X, p->C0.as<float>(), p->C1.as<float>(),
                     p->hub_err.as<double>(), st, teleport, damp);
}

// One iteration over the running columns [0, ka); `empty`: with the rows that
// have no in-edges.
void ppr_launch(gd_ppr_plan* p, float* X, PprState* st, float teleport, float damp, int ka,
                bool empty) {
  const int groups = (ka + kGroup - 1) / kGroup;
  const int kact = groups * kGroup;
  // hub rows first, on the plan's stream, so their workgroups are placed before
  // the tiles fill the CUs; the tiles fork onto the side stream and join back
  hipStream_t ts = p->stream;
  if (p->n_hubs) {
    (void)hipEventRecord(p->fork_ev, p->stream);
    (void)hipStreamWaitEvent(p->side, p->fork_ev, 0);
    ts = p->side;
    if (p->hub_cols == 16)
      ppr_launch_hubs<16>(p, X, st, teleport, damp, ka, kact);
    else if (p->hub_cols == 32)
      ppr_launch_hubs<32>(p, X, st, teleport, damp, ka, kact);
    else
      ppr_launch_hubs<64>(p, X, st, teleport, damp, ka, kact);
  }
  int gp_log2 = 0;  // column groups swept at once: kc / kGroup = 1, 2, 4 or 8
  while ((kGroup << gp_log2) < p->kc) gp_log2++;
  const int gp = 1 << gp_log2;
  hipLaunchKernelGGL(ppr_pull_kernel, dim3(p->grid * gp, (groups + gp - 1) / gp), dim3(kPBlock),
                     0, ts, p->tiles.as<Tile>(), p->n_tiles, p->m, p->rows.as<int2>(), p->col, p->outdeg,
                     p->inv.as<double>(), p->seeds.as<int32_t>(), p->frozen.as<int32_t>(), ka, (int64_t)p->k, gp_log2,
                     X, p->C0.as<float>(), p->C1.as<float>(), p->err_part.as<double>(), st,
                     teleport, damp);
  empty = empty && p->n_empty;
  if (empty)
    hipLaunchKernelGGL(ppr_empty_kernel, dim3(kEmptySlots, groups), dim3(kPBlock), 0, ts,
                       p->empty.as<int32_t>(), p->n_empty, p->outdeg, p->inv.as<double>(),
                       p->seeds.as<int32_t>(), p->frozen.as<int32_t>(), (int64_t)p->k, X,
                       p->C0.as<float>(), p->C1.as<float>(),
                       p->err_part.as<double>() + (size_t)p->grid * p->k, st, teleport, damp);
  if (p->n_hubs) {
    (void)hipEventRecord(p->join_ev, p->side);
    (void)hipStreamWaitEvent(p->stream, p->join_ev, 0);
  }
  hipLaunchKernelGGL(ppr_reduce_kernel, dim3(groups, kRedSplits), dim3(kPBlock), 0, p->stream,
                     p->err_part.as<double>(), p->grid + (empty ? kEmptySlots : 0), p->hub_err.as<double>(), p->n_hubs,
                     (int64_t)p->k, kact, p->fin.as<double>(), p->col_err.as<double>(),
                     p->frozen.as<int32_t>(), p->col_iters.as<int32_t>(), p->column_stop ? 1 : 0,
                     st, p->errors.as<double>());
}

// Applies `order` (new column c <- old column order[c], c < ka) to the rows of
// X and of the contrib buffer the next iteration gathers, and to the k-length
// per-column arrays; cperm (internal -> user column) follows.
int ppr_compact(gd_ppr_plan* p, float* X, float* Cnext, int ka, const std::vector<int32_t>& order,
                std::vector<int32_t>& cperm) {
  GD_HIP_TRY(hipMemcpyAsync(p->newcol.ptr, order.data(), 4 * (size_t)ka, hipMemcpyHostToDevice,
                            p->stream));
  const int m = p->m;
  const int grid = std::max(1, std::min(16384, (m + kPWaves - 1) / kPWaves));
  hipLaunchKernelGGL(ppr_permute_cols_kernel, dim3(grid), dim3(kPBlock),
                     (size_t)kPWaves * ka * sizeof(float), p->stream, m, (int64_t)p->k, ka,
                     p->newcol.as<int32_t>(), X, Cnext);
  GD_HIP_TRY(hipGetLastError());
  std::vector<int32_t> seeds(ka), fz(ka), its(ka);
  std::vector<double> ce(ka);
  GD_HIP_TRY(hipMemcpyAsync(seeds.data(), p->seeds.ptr, 4 * (size_t)ka, hipMemcpyDeviceToHost,
                            p->stream));
  GD_HIP_TRY(hipMemcpyAsync(fz.data(), p->frozen.ptr, 4 * (size_t)ka, hipMemcpyDeviceToHost,
                            p->stream));
  GD_HIP_TRY(hipMemcpyAsync(its.data(), p->col_iters.ptr, 4 * (size_t)ka, hipMemcpyDeviceToHost,
                            p->stream));
  GD_HIP_TRY(hipMemcpyAsync(ce.data(), p->col_err.ptr, 8 * (size_t)ka, hipMemcpyDeviceToHost,
                            p->stream));
  GD_HIP_TRY(hipStreamSynchronize(p->stream));
  std::vector<int32_t> seeds2(ka), fz2(ka), its2(ka), cp2(ka);
  std::vector<double> ce2(ka);
  for (int c = 0; c < ka; c++) {
    const int o = order[c];
    seeds2[c] = seeds[o];
    fz2[c] = fz[o];
    its2[c] = its[o];
    ce2[c] = ce[o];
    cp2[c] = cperm[o];
  }
  for (int c = 0; c < ka; c++) cperm[c] = cp2[c];
  GD_HIP_TRY(hipMemcpyAsync(p->seeds.ptr, seeds2.data(), 4 * (size_t)ka, hipMemcpyHostToDevice,
                            p->stream));
  GD_HIP_TRY(hipMemcpyAsync(p->frozen.ptr, fz2.data(), 4 * (size_t)ka, hipMemcpyHostToDevice,
                            p->stream));
  GD_HIP_TRY(hipMemcpyAsync(p->col_iters.ptr, its2.data(), 4 * (size_t)ka, hipMemcpyHostToDevice,
                            p->stream));
  GD_HIP_TRY(hipMemcpyAsync(p->col_err.ptr, ce2.data(), 8 * (size_t)ka, hipMemcpyHostToDevice,
                            p->stream));
  GD_HIP_TRY(hipStreamSynchronize(p->stream));  // host vectors go out of scope
  return GD_OK;
}

}  // namespace

extern "C" {

void gd_ppr_default_plan_config(gd_ppr_plan_config* c) {
  c->relabel = -1;
  c->k_chunk = 0;
  c->column_stop = -1;
  c->compact = -1;
  c->hub_cols = 0;
}

int gd_ppr_plan_create(int m, int64_t nnz, const int32_t* d_off, const int32_t* d_col,
                       const int32_t* d_outdeg, int k, void* stream, const gd_ppr_plan_config* cfg,
                       gd_ppr_plan** out) {
  GD_CHECK_ARG(out != nullptr, "plan output pointer is NULL");
  *out = nullptr;
  GD_CHECK_ARG(m >= 0 && nnz >= 0 && nnz < (1ll << 31), "m/nnz out of range");
  GD_CHECK_ARG(m == 0 || (d_off && d_outdeg), "NULL device array");
  GD_CHECK_ARG(nnz == 0 || d_col, "NULL column indices");
  GD_CHECK_ARG(k > 0 && k % 64 == 0, "k must be a positive multiple of 64");
  gd_ppr_plan_config c;
  if (cfg)
    c = *cfg;
  else
    gd_ppr_default_plan_config(&c);
  GD_CHECK_ARG(c.k_chunk == 0 || c.k_chunk == 64 || c.k_chunk == 128 || c.k_chunk == 256,
               "k_chunk must be 0, 64, 128 or 256");
  GD_CHECK_ARG(c.k_chunk == 0 || k % c.k_chunk == 0, "k must be a multiple of k_chunk");
  GD_CHECK_ARG(c.hub_cols == 0 || c.hub_cols == 16 || c.hub_cols == 32 || c.hub_cols == 64,
               "hub_cols must be 0, 16, 32 or 64");
  if (gd_device_count() <= 0) {
    set_error("no HIP device visible");
    return GD_ERR_NO_DEVICE;
  }
  gd_ppr_plan* p = new gd_ppr_plan();
  p->m = m;
  p->nnz = nnz;
  p->k = k;
  p->kc = c.k_chunk ? c.k_chunk : kGroup;
  p->stream = (hipStream_t)stream;
  p->relabel = (c.relabel == 1) || (c.relabel == -1 && nnz >= (1 << 20));
  p->column_stop = c.column_stop != 0;
  // LDS of the in-place column permutation: kPWaves rows of k floats <= 64 KB
  p->compact = p->column_stop && c.compact != 0 && k <= 4096;
  p->hub_cols = c.hub_cols ? c.hub_cols : kGroup;
  int rc = GD_OK;
  if (m > 0) {
    hipEvent_t t0 = nullptr, t1 = nullptr;
    if (hipEventCreate(&t0) == hipSuccess && hipEventCreate(&t1) == hipSuccess)
      (void)hipEventRecord(t0, p->stream);
    rc = ppr_build(p, d_off, d_col, d_outdeg);
    if (t0 && t1) {
      (void)hipEventRecord(t1, p->stream);
      (void)hipEventSynchronize(t1);
      (void)hipEventElapsedTime(&p->plan_ms, t0, t1);
    }
    if (t0) (void)hipEventDestroy(t0);
    if (t1) (void)hipEventDestroy(t1);
  }
  if (rc) {
    delete p;
    return rc;
  }
  *out = p;
  return GD_OK;
}

int gd_ppr_plan_info(const gd_ppr_plan* p, gd_ppr_plan_info_t* info) {
  GD_CHECK_ARG(p != nullptr && info != nullptr, "NULL plan / info");
  info->n_tiles = p->n_tiles;
  info->n_hubs = p->n_hubs;
  info->k = p->k;
  info->k_chunk = p->kc;
  info->relabel = p->relabel ? 1 : 0;
  info->grid = p->grid;
  info->plan_ms = p->plan_ms;
  info->hub_cols = p->hub_cols;
  return GD_OK;
}

int gd_ppr_plan_column_iterations(const gd_ppr_plan* p, int32_t* iterations) {
  GD_CHECK_ARG(p != nullptr && iterations != nullptr, "NULL plan / output");
  for (int j = 0; j < p->k; j++)
    iterations[j] = j < (int)p->last_col_iters.size() ? p->last_col_iters[j] : 0;
  return GD_OK;
}

int gd_ppr_plan_destroy(gd_ppr_plan* p) {
  delete p;
  return GD_OK;
}

int gd_ppr_plan_run(gd_ppr_plan* p, const int32_t* d_seeds, float* d_X,
                    const gd_pr_options* opts, gd_pr_stats* stats, double* errors,
                    double* col_errors) {
  GD_CHECK_ARG(p != nullptr, "NULL plan");
  gd_pr_options o;
  if (opts)
    o = *opts;
  else
    gd_pr_default_options(&o);
  GD_CHECK_ARG(o.max_iter >= 0, "max_iter must be >= 0");
  gd_pr_stats s;
  memset(&s, 0, sizeof(s));
  const int m = p->m;
  if (m == 0) {
    if (stats) *stats = s;
    return GD_OK;
  }
  GD_CHECK_ARG(d_seeds != nullptr && d_X != nullptr, "NULL seeds / X");
  {
    DeviceBuffer bad;
    int rc = bad.alloc(4);
    if (rc) return rc;
    GD_HIP_TRY(hipMemsetAsync(bad.ptr, 0, 4, p->stream));
    hipLaunchKernelGGL(check_seeds_kernel, dim3((p->k + 255) / 256), dim3(256), 0, p->stream,
                       p->k, d_seeds, m, bad.as<int>());
    int h = 0;
    GD_HIP_TRY(hipMemcpyAsync(&h, bad.ptr, 4, hipMemcpyDeviceToHost, p->stream));
    GD_HIP_TRY(hipStreamSynchronize(p->stream));
    GD_CHECK_ARG(h == 0, "seed vertex out of range");
  }
  if (p->errors_cap < std::max(1, o.max_iter)) {
    int rc = p->errors.alloc(sizeof(double) * std::max(1, o.max_iter));
    if (rc) return rc;
    p->errors_cap = std::max(1, o.max_iter);
  }
  const float damp = o.damping, teleport = 1.0f - damp;
  const int chunk = o.chunk > 0 ? o.chunk : (o.tol > 0 ? 4 : std::max(1, o.max_iter));
  const int k = p->k;
  EventPair evp;
  GD_HIP_TRY(evp.create());
  hipEvent_t t0 = evp.a, t1 = evp.b;
  PprState* st = p->state.as<PprState>();
  float* X = p->relabel ? p->Xint.as<float>() : d_X;
  const int64_t n = (int64_t)m * k;
  GD_HIP_TRY(hipEventRecord(t0, p->stream));
  hipLaunchKernelGGL(ppr_map_seeds_kernel, dim3((k + 255) / 256), dim3(256), 0, p->stream, k,
                     d_seeds, p->relabel ? p->rl.inv.as<int32_t>() : nullptr,
                     p->seeds.as<int32_t>());
  if (p->relabel)
    hipLaunchKernelGGL(ppr_permute_rows_kernel, dim3(std::min(16384, (m + 3) / 4)), dim3(256), 0,
                       p->stream, m, (int64_t)k, p->rl.perm.as<int32_t>(), nullptr, d_X, X, 1);
  hipLaunchKernelGGL(ppr_init_kernel, dim3((int)std::min<int64_t>((n + 255) / 256, 65536)),
                     dim3(256), 0, p->stream, n, (int64_t)k, X, p->outdeg, p->C0.as<float>(),
                     st, o.max_iter, o.tol);
  hipLaunchKernelGGL(ppr_reset_cols_kernel, dim3((k + 255) / 256), dim3(256), 0, p->stream, k,
                     p->frozen.as<int32_t>(), p->col_iters.as<int32_t>());
  GD_HIP_TRY(hipGetLastError());
  std::vector<int32_t> cperm(k);  // internal column -> user column
  for (int j = 0; j < k; j++) cperm[j] = j;
  int ka = k;  // columns [0, ka) may still be running; the rest are frozen
  int launched = 0;
  int permuted_at = 0;  // the last iteration before which columns were permuted
  PprState h{};
  std::vector<int32_t> fz;
  while (launched < o.max_iter) {
    const int nl = std::min(chunk, o.max_iter - launched);
    for (int q = launched; q < launched + nl; q++)
      ppr_launch(p, X, st, teleport, damp, ka, q < 2 || q == permuted_at);
    GD_HIP_TRY(hipGetLastError());
    launched += nl;
    GD_HIP_TRY(hipMemcpyAsync(&h, st, sizeof(PprState), hipMemcpyDeviceToHost, p->stream));
    GD_HIP_TRY(hipStreamSynchronize(p->stream));
    if (h.done) break;
    if (!p->compact) continue;
    fz.resize(ka);
    GD_HIP_TRY(hipMemcpy(fz.data(), p->frozen.ptr, 4 * (size_t)ka, hipMemcpyDeviceToHost));
    int nf = 0;
    for (int c = 0; c < ka; c++) nf += fz[c] != 0;
    // a permutation costs about one pass over X and the contrib; it pays once a
    // few iterations skip the frozen columns' gathers
    if (nf < std::max(32, ka / 8) || nf >= ka) continue;
    std::vector<int32_t> order;
    order.reserve(ka);
    for (int c = 0; c < ka; c++)
      if (!fz[c]) order.push_back(c);
    for (int c = 0; c < ka; c++)
      if (fz[c]) order.push_back(c);
    float* Cnext = (h.iter & 1) ? p->C1.as<float>() : p->C0.as<float>();
    const int rc = ppr_compact(p, X, Cnext, ka, order, cperm);
    if (rc) return rc;
    permuted_at = launched;
    ka -= nf;
  }
  // back to the user's vertex and column order
  const bool permuted = ka < k;
  if (permuted)
    GD_HIP_TRY(hipMemcpyAsync(p->cperm.ptr, cperm.data(), 4 * (size_t)k, hipMemcpyHostToDevice,
                              p->stream));
  if (p->relabel) {
    hipLaunchKernelGGL(ppr_permute_rows_kernel, dim3(std::min(16384, (m + 3) / 4)), dim3(256), 0,
                       p->stream, m, (int64_t)k, p->rl.perm.as<int32_t>(),
                       permuted ? p->cperm.as<int32_t>() : nullptr, X, d_X, 0);
  } else if (permuted) {
    std::vector<int32_t> inv(k);  // user column u <- internal column inv[u]
    for (int j = 0; j < k; j++) inv[cperm[j]] = j;
    GD_HIP_TRY(hipMemcpyAsync(p->newcol.ptr, inv.data(), 4 * (size_t)k, hipMemcpyHostToDevice,
                              p->stream));
    const int grid = std::max(1, std::min(16384, (m + kPWaves - 1) / kPWaves));
    hipLaunchKernelGGL(ppr_permute_cols_kernel, dim3(grid), dim3(kPBlock),
                       (size_t)kPWaves * k * sizeof(float), p->stream, m, (int64_t)k, k,
                       p->newcol.as<int32_t>(), X, (float*)nullptr);
    GD_HIP_TRY(hipStreamSynchronize(p->stream));  // inv goes out of scope
  }
  GD_HIP_TRY(hipGetLastError());
  GD_HIP_TRY(hipEventRecord(t1, p->stream));
  GD_HIP_TRY(hipEventSynchronize(t1));
  GD_HIP_TRY(hipEventElapsedTime(&s.solve_ms, t0, t1));
  s.iterations = h.iter;
  std::vector<int32_t> its(k);
  std::vector<double> ce(k);
  GD_HIP_TRY(hipMemcpy(its.data(), p->col_iters.ptr, 4 * (size_t)k, hipMemcpyDeviceToHost));
  GD_HIP_TRY(hipMemcpy(ce.data(), p->col_err.ptr, 8 * (size_t)k, hipMemcpyDeviceToHost));
  p->last_col_iters.assign(k, 0);
  for (int j = 0; j < k; j++) p->last_col_iters[cperm[j]] = its[j];
  if (h.iter > 0) {
    std::vector<double> errs(h.iter);
    GD_HIP_TRY(hipMemcpy(errs.data(), p->errors.ptr, 8 * (size_t)h.iter, hipMemcpyDeviceToHost));
    s.final_error = errs[h.iter - 1];
    s.converged = s.final_error < o.tol;
    if (errors)
      for (int i = 0; i < h.iter; i++) errors[i] = errs[i];
    if (col_errors)
      for (int j = 0; j < k; j++) col_errors[cperm[j]] = ce[j];
  }
  if (stats) *stats = s;
  return GD_OK;
}

}  // extern "C"
