// spmv.hip -- CSR SpMV y <- y + A x for gfx950 (src/spmv/omp_base.cc:17-28).
//
// Same tile engine as PageRank: products x[Aj[k]] * Ax[k] are formed
// (rounded, this file is built with -ffp-contract=off) and staged
// in LDS; rows are then summed by one thread starting from
// y[row] in CSR order, which is exactly the reference's arithmetic; so are
// the longer rows of a tile (the owner thread's chain just runs longer).
// Rows longer than a tile get a workgroup each that feeds one lane's
// sequential chain in CSR order (hub_chain_sum), so every row is the
// reference's sum bit for bit.
//
// Where x exceeds an XCD's L2 and the rows gather from enough of it, the
// gathers go through windows of x (window_gather.h): a pass expands x into
// one slot per nonzero, and the tiles read their slots in runs.  The matrix
// values stay the caller's, read in CSR order.  Bound by HBM: 6 bytes per
// nonzero in the first pass, 14 in the second.  2^22 x 2^22, 32 random
// columns per row: 0.536 ms, 0.737 with one pass of the tiles per 1/8 of the
// columns over a reordered copy of the matrix, 1.9 with plain gathers.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <memory>
#include <mutex>
#include <vector>

#include "gardenia_hip.h"
#include "gd_common.h"
#include "pull_engine.h"
#include "tile_sort.h"
#include "window_gather.h"

namespace gd {

constexpr int kSpIPT = 8;
constexpr int kSpTileNnz = kBlock * kSpIPT;

struct SpGather {
  const float* __restrict__ x;
  const float* __restrict__ Ax;
  __device__ __forceinline__ float value(int e, int j) const { return x[j] * Ax[e]; }
};

// x[j] from its slot, Ax in CSR order.
struct SpSlotGather {
  const float* __restrict__ slots;
  const float* __restrict__ Ax;
  static constexpr bool kScaled = true;
  __device__ __forceinline__ float value(int e, int slot) const { return slots[slot] * Ax[e]; }
  __device__ __forceinline__ float raw(int slot) const { return slots[slot]; }
  __device__ __forceinline__ float factor(int e) const { return Ax[e]; }
};

struct SpEpilogue {
  float* __restrict__ y;
  using Pre = float;  // y[row] before the update
  __device__ __forceinline__ Pre pre(int r) const { return y[r]; }
  __device__ __forceinline__ float init(const Pre& y0) const { return y0; }
  __device__ __forceinline__ double finish(int r, float s, const Pre&) const {
    y[r] = s;
    return 0.0;
  }
};

// Workgroups [0, n_long) each add one row longer than
// a tile (2048 nonzeros) in CSR order on one lane (hub_chain_sum: products of
// both signs), the rest one LDS row tile each (every row summed by its owner
// thread in CSR order).  Every row is the reference's sum bit for bit.  LONG =
// false (no long rows) leaves the long-row code, and its registers, out.
// WIN: Aj holds slots, sorted by source within each tile, with their offsets
// there in pos; long rows always gather x itself.
template <bool LONG, bool WIN>
__global__ __launch_bounds__(kBlock) void spmv_pull_kernel(
    const Tile* __restrict__ tiles, int n_tiles, const Tile* __restrict__ long_tiles, int n_long,
    const int32_t* __restrict__ Ap, const int32_t* __restrict__ Aj,
    const uint16_t* __restrict__ pos, int e_max, const float* __restrict__ Ax,
    const float* __restrict__ x, float* __restrict__ y) {
  // a row tile's LDS, or a long row's two chunk buffers + the broadcast sum
  static_assert(sizeof(RowTileLds<kSpIPT>) >= (2 * kHubChunk + 1) * sizeof(float), "LDS union");
  __shared__ __align__(16) unsigned char smem[sizeof(RowTileLds<kSpIPT>)];
  RowTileLds<kSpIPT>& lds = *reinterpret_cast<RowTileLds<kSpIPT>*>(smem);
  using G = std::conditional_t<WIN, SpSlotGather, SpGather>;
  const G g{x, Ax};
  const int b = blockIdx.x;
  if (LONG && b < n_long) {
    float* const buf = reinterpret_cast<float*>(smem);
    const Tile t = long_tiles[b];
    const float s = hub_chain_sum<16, false>(Aj, nullptr, e_max, t.z, t.w - t.z, SpGather{x, Ax},
                                             y[t.x], buf, buf + kHubChunk, buf + 2 * kHubChunk);
    if (threadIdx.x == 0) y[t.x] = s;
  } else {
    const Tile t = tiles[WIN ? xcd_run_block(b - n_long, n_tiles) : b - n_long];
    const SpEpilogue e{y};
    (void)row_tile<kSpIPT, false, WIN, G, SpEpilogue, true>(
        Ap, Aj, pos, e_max, t.x, t.y, t.z, t.w - t.z, g, e, lds);
  }
}

// Pass 1 of a windowed SpMV (window_gather.h).
__global__ __launch_bounds__(kExpandBlock) void spmv_expand_kernel(
    const float* __restrict__ x, int cols, const int4* __restrict__ pieces,
    const uint16_t* __restrict__ sid, float* __restrict__ slots) {
  __shared__ float win[kWinSize];
  window_expand(x, cols, pieces[blockIdx.x], sid, slots, win);
}

// flag |= a row's columns are not strictly increasing
__global__ void sorted_rows_kernel(int rows, const int32_t* __restrict__ Ap,
                                   const int32_t* __restrict__ Aj, int* __restrict__ unsorted) {
  const int lane = threadIdx.x & 15;  // 16 lanes a row
  int bad = 0;
  for (int r = (blockIdx.x * blockDim.x + threadIdx.x) / 16; r < rows;
       r += gridDim.x * blockDim.x / 16) {
    const int b = Ap[r], e = Ap[r + 1];
    for (int k = b + 1 + lane; k < e; k += 16) bad |= Aj[k] <= Aj[k - 1];
  }
  if (bad) atomicOr(unsorted, 1);
}

}  // namespace gd

using namespace gd;

struct gd_spmv_plan {
  int rows = 0, cols = 0;
  int64_t nnz = 0;
  const int32_t* Ap = nullptr;
  const int32_t* Aj = nullptr;
  const float* Ax = nullptr;
  hipStream_t stream = nullptr;
  Schedule sched;
  int n_tiles = 0, n_hubs = 0;  // row tiles; rows longer than a tile
  DeviceBuffer tiles, long_tiles;
  DeviceBuffer dummy_col;  // 1 element, used as Aj when nnz == 0
  int e_max = 0;
  bool sliced = false;  // the reported mode
  // windowed gather: the nonzeros' slots, sorted within tiles, and their
  // offsets there
  WindowGather win;
  DeviceBuffer slot, pos;
  // long rows on `stream`, the tiles beside them on `side` (long_rows_beside)
  hipStream_t side = nullptr;
  hipEvent_t fork_ev = nullptr, join_ev = nullptr;
  // A run's launches pass x through `win` and order themselves by the events:
  // host threads queue whole runs.
  std::mutex run_lock;
  ~gd_spmv_plan() {
    if (fork_ev) (void)hipEventDestroy(fork_ev);
    if (join_ev) (void)hipEventDestroy(join_ev);
    if (side) (void)hipStreamDestroy(side);
  }
};

namespace {

// GD_ERR_INVALID unless every row's columns are strictly increasing.
int check_sorted(const gd_spmv_plan* p) {
  DeviceBuffer bad;
  int rc = bad.alloc(4);
  if (rc) return rc;
  GD_HIP_TRY(hipMemsetAsync(bad.ptr, 0, 4, p->stream));
  const int g = (int)std::max<int64_t>(1, std::min<int64_t>(((int64_t)p->rows + 15) / 16, 16384));
  hipLaunchKernelGGL(sorted_rows_kernel, dim3(g), dim3(256), 0, p->stream, p->rows, p->Ap, p->Aj,
                     bad.as<int>());
  GD_HIP_TRY(hipGetLastError());
  int h_bad = 0;
  GD_HIP_TRY(hipMemcpyAsync(&h_bad, bad.ptr, 4, hipMemcpyDeviceToHost, p->stream));
  GD_HIP_TRY(hipStreamSynchronize(p->stream));
  if (h_bad) {
    set_error("column-sliced SpMV needs sorted columns within each row");
    return GD_ERR_INVALID;
  }
  return GD_OK;
}

// Whether the long rows run as a launch of their own beside the tiles.  Their
// chain (3 ns per nonzero of the longest) holds 176 registers; tiles in the
// same launch run at 2 wavefronts per SIMD and take about 8 ps per nonzero.
// While the chain lasts longer than that, one launch costs the chain alone,
// two cost the fork and the join (15 us) as well.  Power-law matrices, us in
// one launch / beside (with windows where x is large): 0.6 M rows, 9 M
// nonzeros 100 / 142, 2 M, 8 M 88 / 99, 2 M, 19 M 166 / 182; 2.5 M, 38 M 337 /
// 252, 4 M, 61 M 538 / 379.
bool long_rows_beside(const gd_spmv_plan* p) {
  return !p->sched.hub_row.empty() &&
         (double)p->nnz * 8e-3 >= p->sched.max_row_len * 3.0 + 15000.0;
}

// Windows pay where x exceeds one XCD's 4 MB L2, its windows are filled for
// enough nonzeros (a piece of the expand pass copies its window into LDS
// first), and a tile gathers from many lines of x: the gathers of a band or of
// columns in runs hit the L1 and L2.  Only nonzeros in row tiles count: long
// rows gather x itself, and must not wait for the expand pass.
// us plain / windowed, nonzeros per column at random: 1 M columns x 1 14.5 /
// 17.2, 1.2 M x 1 14.7 / 15.6, x 2 21.7 / 19.4; 2 M x 1 31.5 / 23.2, 4 M x 0.5
// 36 / 21, x 1.75 107 / 40.
// Lines per nonzero: 4 M x 32 within 250 of the row 0.01, 230 / 511, within
// 16,000 0.43, 573 / 510; 4 M x 16 in runs of 4 0.25, 308 / 280, of 2 0.50, 503
// / 280.  Up to twice the L2 most of x stays there: 1.1 M x 16 in runs of 2
// 0.49, 68 / 77, x 8 within 16,000 0.43, 42.5 / 45.5, within 64,000 0.78, 47.8 /
// 45.3.
int wants_windows(const gd_spmv_plan* p, bool* want) {
  const int64_t cols = p->cols;
  const bool large = cols > 2 << 20;
  *want = cols > 1 << 20 && (p->sched.hub_row.empty() || long_rows_beside(p)) &&
          window_gather_fits(p->cols, p->nnz, (int64_t)p->sched.tiles.size());
  if (!*want) return GD_OK;
  int64_t in_tiles = 0;
  std::vector<int2> runs;
  for (const Tile& t : p->sched.tiles) {
    if (t.y < 0 || t.w == t.z) continue;
    runs.push_back(make_int2(t.z, t.w - t.z));
    in_tiles += t.w - t.z;
  }
  *want = in_tiles >= (large ? cols / 2 : 2 * cols);
  if (!*want) return GD_OK;
  double lines = 0.0;
  const int rc = gathered_lines(runs, p->Aj, p->stream, &lines);
  *want = lines >= (large ? 0.45 : 0.6);
  return rc;
}

int build_windows(gd_spmv_plan* p) {
  int rc = p->slot.alloc(4 * (size_t)p->nnz);
  if (!rc) rc = p->pos.alloc(2 * (size_t)p->nnz);
  if (rc) return rc;
  std::vector<int2> segs;
  rc = build_tile_sort(p->sched, kSpTileNnz, p->Aj, p->slot.as<int32_t>(), p->pos.as<uint16_t>(),
                       p->stream, true, 0, &segs);
  // long rows stay out: they gather x themselves, beside the expand pass
  segs.erase(std::remove_if(segs.begin(), segs.end(), [](const int2& s) { return s.y < 0; }),
             segs.end());
  int64_t in_tiles = 0;
  for (const int2& s : segs) in_tiles += s.y;
  if (!rc)
    rc = build_window_gather(p->cols, in_tiles, segs, p->slot.as<int32_t>(), p->stream, &p->win);
  return rc;
}

}  // namespace

extern "C" {

int gd_spmv_plan_create(int rows, int cols, int64_t nnz, const int32_t* d_Ap, const int32_t* d_Aj,
                        const float* d_Ax, void* stream, gd_spmv_plan** out) {
  return gd_spmv_plan_create_ex(rows, cols, nnz, d_Ap, d_Aj, d_Ax, stream, GD_SPMV_TILES, out);
}

int gd_spmv_plan_create_ex(int rows, int cols, int64_t nnz, const int32_t* d_Ap,
                           const int32_t* d_Aj, const float* d_Ax, void* stream, int mode,
                           gd_spmv_plan** out) {
  GD_CHECK_ARG(mode == GD_SPMV_AUTO || mode == GD_SPMV_TILES || mode == GD_SPMV_SLICED,
               "unknown SpMV mode");
  GD_CHECK_ARG(out != nullptr, "plan output pointer is NULL");
  *out = nullptr;
  GD_CHECK_ARG(rows >= 0 && cols >= 0 && nnz >= 0 && nnz < (1ll << 31), "size out of range");
  GD_CHECK_ARG(rows == 0 || d_Ap, "NULL row offsets");
  GD_CHECK_ARG(nnz == 0 || (d_Aj && d_Ax), "NULL column indices / values");
  if (gd_device_count() <= 0) {
    set_error("no HIP device visible");
    return GD_ERR_NO_DEVICE;
  }
  gd_spmv_plan* p = new gd_spmv_plan();
  p->rows = rows;
  p->cols = cols;
  p->nnz = nnz;
  p->Ap = d_Ap;
  p->Aj = d_Aj;
  p->Ax = d_Ax;
  p->stream = (hipStream_t)stream;
  int rc = GD_OK;
  if (rows > 0) {
    std::vector<int32_t> h_off(rows + 1);
    hipError_t e = hipMemcpyAsync(h_off.data(), d_Ap, sizeof(int32_t) * (rows + 1),
                                  hipMemcpyDeviceToHost, p->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(p->stream);
    if (e != hipSuccess) {
      set_error(std::string("copying row offsets: ") + hipGetErrorString(e));
      rc = GD_ERR_DEVICE;
    }
    if (!rc)
      rc = build_schedule(rows, nnz, h_off.data(), kSpTileNnz, kTileRows, &p->sched, kSpTileNnz);
    if (!rc) rc = check_columns(d_Aj, nnz, cols, p->stream);
    if (!rc && nnz > 0 && mode != GD_SPMV_TILES) {
      // auto: sliced when x spans more than one XCD's L2 and rows are short
      const bool want = mode == GD_SPMV_SLICED ||
                        ((int64_t)cols * 4 > (4 << 20) && p->sched.max_row_len <= kSeqRow);
      if (want) {
        rc = check_sorted(p);
        if (!rc) p->sliced = true;
        if (rc == GD_ERR_INVALID && mode == GD_SPMV_AUTO) rc = GD_OK;  // unsorted rows: tiles
      }
    }
    if (!rc && nnz > 0) {
      bool want = false;
      rc = wants_windows(p, &want);
      if (!rc && want) rc = build_windows(p);
      if (rc == GD_ERR_ALLOC) {  // no room for windows: x itself
        p->win.release();
        p->slot.release();
        p->pos.release();
        rc = GD_OK;
      }
    }
    if (!rc && nnz == 0) {
      rc = p->dummy_col.alloc(4);
      if (!rc && hipMemsetAsync(p->dummy_col.ptr, 0, 4, p->stream) != hipSuccess) rc = GD_ERR_DEVICE;
      p->Aj = p->dummy_col.as<int32_t>();
    }
    p->e_max = (int)std::max<int64_t>(nnz - 1, 0);
    if (!rc) {
      std::vector<Tile> row_tiles, longs;
      for (const Tile& t : p->sched.tiles) (t.y < 0 ? longs : row_tiles).push_back(t);
      std::stable_sort(longs.begin(), longs.end(),  // the longest rows start first
                       [](const Tile& a, const Tile& b) { return a.w - a.z > b.w - b.z; });
      p->n_tiles = (int)row_tiles.size();
      p->n_hubs = (int)longs.size();
      if (p->n_hubs && p->n_tiles && long_rows_beside(p) &&
          (hipStreamCreateWithFlags(&p->side, hipStreamNonBlocking) != hipSuccess ||
           hipEventCreateWithFlags(&p->fork_ev, hipEventDisableTiming) != hipSuccess ||
           hipEventCreateWithFlags(&p->join_ev, hipEventDisableTiming) != hipSuccess)) {
        set_error("creating the long rows' stream");
        rc = GD_ERR_DEVICE;
      }
      if (!rc) rc = p->tiles.alloc(sizeof(Tile) * std::max(1, p->n_tiles));
      if (!rc) rc = p->long_tiles.alloc(sizeof(Tile) * std::max(1, p->n_hubs));
      hipError_t e2 = hipSuccess;
      if (!rc && p->n_tiles)
        e2 = hipMemcpyAsync(p->tiles.ptr, row_tiles.data(), sizeof(Tile) * p->n_tiles,
                            hipMemcpyHostToDevice, p->stream);
      if (!rc && e2 == hipSuccess && p->n_hubs)
        e2 = hipMemcpyAsync(p->long_tiles.ptr, longs.data(), sizeof(Tile) * p->n_hubs,
                            hipMemcpyHostToDevice, p->stream);
      if (!rc && e2 == hipSuccess) e2 = hipStreamSynchronize(p->stream);
      if (!rc && e2 != hipSuccess) {
        set_error(std::string("uploading schedule: ") + hipGetErrorString(e2));
        rc = GD_ERR_DEVICE;
      }
    }
  }
  if (rc) {
    delete p;
    return rc;
  }
  *out = p;
  return GD_OK;
}

int gd_spmv_plan_run(gd_spmv_plan* p, const float* d_x, float* d_y) {
  GD_CHECK_ARG(p != nullptr, "NULL plan");
  if (p->rows == 0) return GD_OK;
  GD_CHECK_ARG(d_y != nullptr && (p->nnz == 0 || d_x != nullptr), "NULL x / y");
  std::unique_lock<std::mutex> lock(p->run_lock, std::defer_lock);
  if (p->side || p->win.on()) lock.lock();
  auto run = [&](auto kernel, int n_tiles, int n_long, const int32_t* aj, const float* src,
                 hipStream_t s) {
    hipLaunchKernelGGL(kernel, dim3(n_tiles + n_long), dim3(kBlock), 0, s, p->tiles.as<Tile>(),
                       n_tiles, p->long_tiles.as<Tile>(), n_long, p->Ap, aj, p->pos.as<uint16_t>(),
                       p->e_max, p->Ax, src, d_y);
  };
  hipStream_t ts = p->stream;
  int n_long = p->n_hubs;
  if (p->side) {  // long rows first, so that they are placed before the tiles fill the CUs
    GD_HIP_TRY(hipEventRecord(p->fork_ev, p->stream));
    GD_HIP_TRY(hipStreamWaitEvent(p->side, p->fork_ev, 0));
    ts = p->side;
    run(spmv_pull_kernel<true, false>, 0, n_long, p->Aj, d_x, p->stream);
    n_long = 0;
  }
  if (p->win.on()) {
    hipLaunchKernelGGL(spmv_expand_kernel, dim3(p->win.n_pieces), dim3(kExpandBlock), 0, ts, d_x,
                       p->cols, p->win.pieces.as<int4>(), p->win.sid.as<uint16_t>(),
                       p->win.stage.as<float>());
    run(spmv_pull_kernel<false, true>, p->n_tiles, 0, p->slot.as<int32_t>(),
        p->win.stage.as<float>(), ts);
  } else if (n_long) {
    run(spmv_pull_kernel<true, false>, p->n_tiles, n_long, p->Aj, d_x, ts);
  } else if (p->n_tiles) {
    run(spmv_pull_kernel<false, false>, p->n_tiles, 0, p->Aj, d_x, ts);
  }
  if (p->side) {
    GD_HIP_TRY(hipEventRecord(p->join_ev, p->side));
    GD_HIP_TRY(hipStreamWaitEvent(p->stream, p->join_ev, 0));
  }
  GD_HIP_TRY(hipGetLastError());
  return GD_OK;
}

int gd_spmv_plan_refresh_values(gd_spmv_plan* p) {
  GD_CHECK_ARG(p != nullptr, "NULL plan");
  return GD_OK;  // every mode reads the caller's values directly
}

int gd_spmv_plan_mode(const gd_spmv_plan* p) {
  return p == nullptr ? -1 : (p->sliced ? GD_SPMV_SLICED : GD_SPMV_TILES);
}

int gd_spmv_plan_windowed(const gd_spmv_plan* p) { return p && p->win.on() ? 1 : 0; }

int gd_spmv_plan_info(const gd_spmv_plan* p, int64_t* n_tiles, int64_t* n_hubs,
                      int32_t* max_row_len) {
  GD_CHECK_ARG(p != nullptr, "NULL plan");
  if (n_tiles) *n_tiles = p->n_tiles;
  if (n_hubs) *n_hubs = p->n_hubs;
  if (max_row_len) *max_row_len = p->sched.max_row_len;
  return GD_OK;
}

int gd_spmv_plan_destroy(gd_spmv_plan* p) {
  delete p;
  return GD_OK;
}

int gd_spmv_solve(int m, int nnz, const int32_t* Ap, const int32_t* Aj, const float* Ax,
                  const float* x, float* y, float* kernel_ms) {
  GD_CHECK_ARG(m >= 0 && nnz >= 0, "negative size");
  GD_CHECK_ARG(m == 0 || (Ap && x && y), "NULL host array");
  GD_CHECK_ARG(nnz == 0 || (Aj && Ax), "NULL column indices / values");
  if (gd_device_count() <= 0) {
    set_error("no HIP device visible");
    return GD_ERR_NO_DEVICE;
  }
  DeviceBuffer dAp, dAj, dAx, dx, dy;
  int rc = dAp.alloc(4 * ((size_t)m + 1));
  if (!rc) rc = dAj.alloc(4 * (size_t)nnz);
  if (!rc) rc = dAx.alloc(4 * (size_t)nnz);
  if (!rc) rc = dx.alloc(4 * (size_t)m);
  if (!rc) rc = dy.alloc(4 * (size_t)m);
  if (rc) return rc;
  if (m > 0) {
    GD_HIP_TRY(hipMemcpy(dAp.ptr, Ap, 4 * ((size_t)m + 1), hipMemcpyHostToDevice));
    GD_HIP_TRY(hipMemcpy(dx.ptr, x, 4 * (size_t)m, hipMemcpyHostToDevice));
    GD_HIP_TRY(hipMemcpy(dy.ptr, y, 4 * (size_t)m, hipMemcpyHostToDevice));
  }
  if (nnz > 0) {
    GD_HIP_TRY(hipMemcpy(dAj.ptr, Aj, 4 * (size_t)nnz, hipMemcpyHostToDevice));
    GD_HIP_TRY(hipMemcpy(dAx.ptr, Ax, 4 * (size_t)nnz, hipMemcpyHostToDevice));
  }
  gd_spmv_plan* plan = nullptr;
  rc = gd_spmv_plan_create_ex(m, m, nnz, dAp.as<int32_t>(), dAj.as<int32_t>(), dAx.as<float>(),
                              nullptr, GD_SPMV_AUTO, &plan);
  if (rc) return rc;
  std::unique_ptr<gd_spmv_plan> owner(plan);  // destroyed on every return below
  EventPair evp;
  GD_HIP_TRY(evp.create());
  hipEvent_t t0 = evp.a, t1 = evp.b;
  GD_HIP_TRY(hipEventRecord(t0, nullptr));
  rc = gd_spmv_plan_run(plan, dx.as<float>(), dy.as<float>());
  GD_HIP_TRY(hipEventRecord(t1, nullptr));
  GD_HIP_TRY(hipEventSynchronize(t1));
  float ms = 0.0f;
  GD_HIP_TRY(hipEventElapsedTime(&ms, t0, t1));
  if (kernel_ms) *kernel_ms = ms;
  if (rc) return rc;
  if (m > 0) GD_HIP_TRY(hipMemcpy(y, dy.ptr, 4 * (size_t)m, hipMemcpyDeviceToHost));
  return GD_OK;
}

}  // extern "C"
