// window_gather.h -- gathers of a vector that exceeds an XCD's L2, as two
// streaming passes (propagation blocking in the pull direction).
//
// A sorted tile of 4096 edges gathers its sources with about 0.7 L2 requests
// per edge, and when the gathered vector exceeds the 4 MB L2 of an XCD about
// a third of them go to the Infinity Cache: the gather is bound by those
// requests (RMAT-24: 140 G/s), far below the rate of a stream.  Instead, the
// sources are cut into windows of kWinSize vertices (128 KB of LDS) and every
// edge gets a slot, in (window, tile, source) order:
//   1. expand (window_expand_kernel): a workgroup holds one window in LDS and
//      writes slot after slot its source's value; a slot's source is 16 bits;
//   2. the tile then gathers its slots instead of its sources.  Its edges,
//      sorted by source, lie in one run of consecutive slots per window, so
//      64 lanes read a few whole lines.
// The values, and the order in which a row adds them, stay the same.  Both
// passes are bound by HBM: 6 bytes per edge in the first (5.2 TB/s), 10 in the
// second (5.1).  RMAT-24, per iteration: 1.34 ms with plain gathers; expand 0.32,
// hub staging 0.11, row tiles and hubs 0.56.  The order of the tiles matters: a tile's
// run shares its first and last line with the neighbouring tiles', so with
// neighbours on different XCDs the tiles fetched 3.3 GB instead of 2.5.
#ifndef GD_WINDOW_GATHER_H_
#define GD_WINDOW_GATHER_H_

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <vector>

#include "gd_common.h"

namespace gd {

constexpr int kWinBits = 15;
constexpr int kWinSize = 1 << kWinBits;  // sources per window
constexpr int kWinMax = 4096;            // windows at most (LDS of the layout kernels)
constexpr int kWinAlign = 8;             // window starts and pieces: multiples of 8 slots
constexpr int kExpandBlock = 1024;

struct WindowGather {
  int n_src = 0;
  int n_pieces = 0;
  int64_t slots = 0;
  DeviceBuffer sid;     // uint16[slots]: source - window base
  DeviceBuffer stage;   // float[slots]: the expanded values
  DeviceBuffer pieces;  // int4[n_pieces]: window's first source, first slot, end slot
  bool on() const { return n_pieces > 0; }
  void release() {
    sid.release();
    stage.release();
    pieces.release();
    n_pieces = 0;
  }
};

// Whether a layout of `segs` segments over n_src sources stays in bounds
// (windows in LDS, a (window, segment) count table of at most 2^28 entries,
// 32-bit slots).
bool window_gather_fits(int n_src, int64_t nnz, int64_t segs);

// Distinct 128-byte lines of the gathered float vector per edge, each of the
// runs of edges (x: first, y: edges) by itself, over up to kLineRuns of them
// spread evenly: about 1 for sources at random, 1/32 for neighbouring ones.
// What the gathers of a workgroup, or of those that run side by side, share in
// the caches.  Synchronises `stream`.
constexpr int kLineRuns = 512;
int gathered_lines(const std::vector<int2>& runs, const int32_t* d_col, hipStream_t stream,
                   double* lines_per_edge);
// The same over runs of `run` edges of all nnz.
int gathered_lines(int64_t nnz, int run, const int32_t* d_col, hipStream_t stream,
                   double* lines_per_edge);

// Slots for the edges of the segments (x: first edge, y: edges; each
// segment's sources ascending in `col`).  col[e] is replaced by the edge's
// slot.  Without segments the gather stays off; GD_ERR_ALLOC leaves `col` as it
// is (a plan then gathers plainly).  Synchronises `stream`.
int build_window_gather(int n_src, int64_t nnz, const std::vector<int2>& segs, int32_t* d_col,
                        hipStream_t stream, WindowGather* g);

// Block b of n in an order that gives every XCD runs of kXcdRun consecutive
// blocks (blocks are dispatched to the 8 XCDs round-robin): neighbouring tiles'
// runs of slots share lines, which one XCD's L2 then reads once.
constexpr int kXcdRun = 32;
__device__ __forceinline__ int xcd_run_block(int b, int n) {
  constexpr int span = 8 * kXcdRun;
  if (b >= n / span * span) return b;
  const int r = b % span;
  return b - r + (r % 8) * kXcdRun + r / 8;
}

// The body of an expand kernel: piece p of the source vector `src`.
__device__ __forceinline__ void window_expand(const float* __restrict__ src, int n_src, int4 p,
                                              const uint16_t* __restrict__ sid,
                                              float* __restrict__ stage, float* win) {
  const int tid = threadIdx.x;
  const int n = min(kWinSize, n_src - p.x);
  constexpr int kU = 8;         // window loads in flight per thread
  constexpr int kQ = 4;         // slot groups in flight per thread
  constexpr int kG = 4;         // slots per group: a wavefront stores 1 KB runs
  constexpr int step = kExpandBlock * kG;
  int s = p.y + tid * kG;
  uint2 q[kQ];
#pragma unroll
  for (int t = 0; t < kQ; t++)
    q[t] = *reinterpret_cast<const uint2*>(sid + min(s + t * step, p.z - kG));
  for (int i = tid; i < n; i += kU * kExpandBlock) {
    float v[kU];
#pragma unroll
    for (int t = 0; t < kU; t++) v[t] = src[p.x + min(i + t * kExpandBlock, n - 1)];
#pragma unroll
    for (int t = 0; t < kU; t++)
      if (i + t * kExpandBlock < n) win[i + t * kExpandBlock] = v[t];
  }
  __syncthreads();
  for (; s < p.z; s += kQ * step) {
    uint2 nx[kQ];
#pragma unroll
    for (int t = 0; t < kQ; t++)
      nx[t] = *reinterpret_cast<const uint2*>(sid + min(s + (kQ + t) * step, p.z - kG));
#pragma unroll
    for (int t = 0; t < kQ; t++)
      if (s + t * step < p.z)
        *reinterpret_cast<float4*>(stage + s + t * step) =
            make_float4(win[q[t].x & 0xffffu], win[q[t].x >> 16], win[q[t].y & 0xffffu],
                        win[q[t].y >> 16]);
#pragma unroll
    for (int t = 0; t < kQ; t++) q[t] = nx[t];
  }
}

}  // namespace gd

#endif  // GD_WINDOW_GATHER_H_
