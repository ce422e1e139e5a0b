// window_gather.hip -- slot layout of a windowed gather (see window_gather.h).
#include "window_gather.h"

#include <rocprim/device/device_scan.hpp>

#include <algorithm>

namespace gd {

namespace {

constexpr int kSegBlock = 256;

// The runs of one segment, edges of one window: s_start[w] = the run's first
// edge in the segment, f(w, run length) for each run.  Every thread returns
// after a barrier, so s_start may be read.
template <class F>
__device__ __forceinline__ void segment_runs(const int32_t* __restrict__ col, int e0, int n,
                                             int* s_start, F f) {
  for (int i = threadIdx.x; i < n; i += kSegBlock) {
    const int w = col[e0 + i] >> kWinBits;
    if (i == 0 || (col[e0 + i - 1] >> kWinBits) != w) s_start[w] = i;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < n; i += kSegBlock) {
    const int w = col[e0 + i] >> kWinBits;
    if (i == n - 1 || (col[e0 + i + 1] >> kWinBits) != w) f(w, i + 1 - s_start[w]);
  }
}

// cnt[w * segs + s] = edges of segment s in window w (zeroed before; only
// windows in use are written).
__global__ __launch_bounds__(kSegBlock) void window_count_kernel(const int2* __restrict__ seg,
                                                                 int64_t segs,
                                                                 const int32_t* __restrict__ col,
                                                                 int32_t* __restrict__ cnt) {
  __shared__ int s_start[kWinMax];
  const int2 g = seg[blockIdx.x];
  segment_runs(col, g.x, g.y, s_start,
               [&](int w, int len) { cnt[(int64_t)w * segs + blockIdx.x] = len; });
}

// slot of edge i of segment s = at[w * segs + s] + shift[w] + its place in its
// run; col[e] = slot, sid[slot] = source - window base.
__global__ __launch_bounds__(kSegBlock) void window_slots_kernel(const int2* __restrict__ seg,
                                                                 int64_t segs,
                                                                 const int32_t* __restrict__ at,
                                                                 const int32_t* __restrict__ shift,
                                                                 int32_t* __restrict__ col,
                                                                 uint16_t* __restrict__ sid) {
  __shared__ int s_start[kWinMax];
  const int2 g = seg[blockIdx.x];
  segment_runs(col, g.x, g.y, s_start, [&](int w, int) {
    s_start[w] = at[(int64_t)w * segs + blockIdx.x] + shift[w] - s_start[w];
  });
  __syncthreads();
  for (int i = threadIdx.x; i < g.y; i += kSegBlock) {
    const int u = col[g.x + i];
    const int slot = s_start[u >> kWinBits] + i;
    col[g.x + i] = slot;
    sid[slot] = (uint16_t)(u & (kWinSize - 1));
  }
}

__global__ void window_starts_kernel(int windows, int64_t segs, const int32_t* __restrict__ at,
                                     int32_t* __restrict__ start) {
  const int w = blockIdx.x * blockDim.x + threadIdx.x;
  if (w < windows) start[w] = at[(int64_t)w * segs];
}

// lines[b] = distinct lines of 32 sources among the edges of the b-th range
// (x: first edge, y: edges).  A bit of LDS per line; vectors of more than
// 2^25 sources have several lines to a bit.
constexpr int kLineBits = 1 << 20;

__global__ __launch_bounds__(kExpandBlock) void count_lines_kernel(
    const int2* __restrict__ range, const int32_t* __restrict__ col, int32_t* __restrict__ lines) {
  __shared__ uint32_t s_set[kLineBits / 32];
  __shared__ int s_n;
  for (int i = threadIdx.x; i < kLineBits / 32; i += kExpandBlock) s_set[i] = 0u;
  if (threadIdx.x == 0) s_n = 0;
  __syncthreads();
  const int2 g = range[blockIdx.x];
  int mine = 0;
  for (int i = threadIdx.x; i < g.y; i += kExpandBlock) {
    const uint32_t line = ((uint32_t)col[g.x + i] >> 5) % kLineBits, bit = 1u << (line & 31);
    mine += (atomicOr(&s_set[line >> 5], bit) & bit) == 0u;
  }
  atomicAdd(&s_n, mine);
  __syncthreads();
  if (threadIdx.x == 0) lines[blockIdx.x] = s_n;
}

}  // namespace

int gathered_lines(const std::vector<int2>& runs, const int32_t* d_col, hipStream_t stream,
                   double* lines_per_edge) {
  *lines_per_edge = 0.0;
  std::vector<int2> range;
  int64_t edges = 0;
  const size_t step = std::max<size_t>(1, runs.size() / kLineRuns);
  for (size_t i = 0; i < runs.size(); i += step) {
    range.push_back(runs[i]);
    edges += runs[i].y;
  }
  if (edges == 0) return GD_OK;
  DeviceBuffer d_range, d_lines;
  int rc = d_range.alloc(sizeof(int2) * range.size());
  if (!rc) rc = d_lines.alloc(4 * range.size());
  if (rc) return rc;
  std::vector<int32_t> lines(range.size());
  GD_HIP_TRY(hipMemcpyAsync(d_range.ptr, range.data(), sizeof(int2) * range.size(),
                            hipMemcpyHostToDevice, stream));
  hipLaunchKernelGGL(count_lines_kernel, dim3((unsigned)range.size()), dim3(kExpandBlock), 0,
                     stream, d_range.as<int2>(), d_col, d_lines.as<int32_t>());
  GD_HIP_TRY(hipGetLastError());
  GD_HIP_TRY(hipMemcpyAsync(lines.data(), d_lines.ptr, 4 * range.size(), hipMemcpyDeviceToHost,
                            stream));
  GD_HIP_TRY(hipStreamSynchronize(stream));
  int64_t n = 0;
  for (const int32_t l : lines) n += l;
  *lines_per_edge = (double)n / (double)edges;
  return GD_OK;
}

int gathered_lines(int64_t nnz, int run, const int32_t* d_col, hipStream_t stream,
                   double* lines_per_edge) {
  std::vector<int2> runs;
  for (int64_t e = 0; e < nnz; e += run)
    runs.push_back(make_int2((int)e, (int)std::min<int64_t>(run, nnz - e)));
  return gathered_lines(runs, d_col, stream, lines_per_edge);
}

bool window_gather_fits(int n_src, int64_t nnz, int64_t segs) {
  const int64_t windows = ((int64_t)n_src + kWinSize - 1) >> kWinBits;
  return nnz > 0 && windows <= kWinMax && windows * segs <= (1ll << 28) &&
         nnz + windows * kWinAlign < (1ll << 31) - 4 * kExpandBlock * kWinAlign;
}

int build_window_gather(int n_src, int64_t nnz, const std::vector<int2>& segs, int32_t* d_col,
                        hipStream_t stream, WindowGather* g) {
  const int windows = (int)(((int64_t)n_src + kWinSize - 1) >> kWinBits);
  const int64_t ns = (int64_t)segs.size();
  if (ns == 0) return GD_OK;  // no edge to lay out: off
  const size_t table = (size_t)windows * ns;
  DeviceBuffer d_segs, cnt, at, start, tmp;
  int rc = d_segs.alloc(sizeof(int2) * (size_t)ns);
  if (!rc) rc = cnt.alloc(4 * table);
  if (!rc) rc = at.alloc(4 * table);
  if (!rc) rc = start.alloc(4 * (size_t)windows);
  if (rc) return rc;
  GD_HIP_TRY(hipMemcpyAsync(d_segs.ptr, segs.data(), sizeof(int2) * (size_t)ns,
                            hipMemcpyHostToDevice, stream));
  GD_HIP_TRY(hipMemsetAsync(cnt.ptr, 0, 4 * table, stream));
  hipLaunchKernelGGL(window_count_kernel, dim3((unsigned)ns), dim3(kSegBlock), 0, stream,
                     d_segs.as<int2>(), ns, d_col, cnt.as<int32_t>());
  GD_HIP_TRY(hipGetLastError());
  size_t bytes = 0;
  GD_HIP_TRY(rocprim::exclusive_scan(nullptr, bytes, cnt.as<int32_t>(), at.as<int32_t>(), 0, table,
                                     rocprim::plus<int32_t>(), stream));
  rc = tmp.alloc(bytes);
  if (rc) return rc;
  GD_HIP_TRY(rocprim::exclusive_scan(tmp.ptr, bytes, cnt.as<int32_t>(), at.as<int32_t>(), 0, table,
                                     rocprim::plus<int32_t>(), stream));
  hipLaunchKernelGGL(window_starts_kernel, dim3((windows + 255) / 256), dim3(256), 0, stream,
                     windows, ns, at.as<int32_t>(), start.as<int32_t>());
  GD_HIP_TRY(hipGetLastError());
  std::vector<int32_t> h(windows + 1), shift(windows);
  GD_HIP_TRY(hipMemcpyAsync(h.data(), start.ptr, 4 * (size_t)windows, hipMemcpyDeviceToHost,
                            stream));
  GD_HIP_TRY(hipStreamSynchronize(stream));
  h[windows] = (int32_t)nnz;
  // Pieces: about 8 per CU, so the last round of workgroups is short, of at
  // least half a window's slots, so filling the LDS stays a small part.
  const int64_t want = std::max<int64_t>(kWinSize / 2, (nnz + 2047) / 2048);
  std::vector<int4> pieces;
  int64_t slot = 0;
  for (int w = 0; w < windows; w++) {
    const int64_t n = (int64_t)h[w + 1] - h[w];
    shift[w] = (int32_t)(slot - h[w]);
    const int64_t padded = (n + kWinAlign - 1) / kWinAlign * kWinAlign;
    const int64_t k = (padded + want - 1) / want;
    for (int64_t q = 0; q < k; q++)
      pieces.push_back(make_int4(w << kWinBits,
                                 (int)(slot + padded / kWinAlign * q / k * kWinAlign),
                                 (int)(slot + padded / kWinAlign * (q + 1) / k * kWinAlign), 0));
    slot += padded;
  }
  g->n_src = n_src;
  g->slots = slot;
  rc = g->sid.alloc(2 * (size_t)slot);
  if (!rc) rc = g->stage.alloc(4 * (size_t)slot);
  if (!rc) rc = g->pieces.alloc(sizeof(int4) * std::max<size_t>(1, pieces.size()));
  if (rc) return rc;
  GD_HIP_TRY(hipMemsetAsync(g->sid.ptr, 0, 2 * (size_t)slot, stream));  // the windows' padding
  GD_HIP_TRY(hipMemcpyAsync(start.ptr, shift.data(), 4 * (size_t)windows, hipMemcpyHostToDevice,
                            stream));
  GD_HIP_TRY(hipMemcpyAsync(g->pieces.ptr, pieces.data(), sizeof(int4) * pieces.size(),
                            hipMemcpyHostToDevice, stream));
  hipLaunchKernelGGL(window_slots_kernel, dim3((unsigned)ns), dim3(kSegBlock), 0, stream,
                     d_segs.as<int2>(), ns, at.as<int32_t>(), start.as<int32_t>(), d_col,
                     g->sid.as<uint16_t>());
  GD_HIP_TRY(hipGetLastError());
  GD_HIP_TRY(hipStreamSynchronize(stream));  // scratch and host vectors go out of scope
  g->n_pieces = (int)pieces.size();
  return GD_OK;
}

}  // namespace gd
