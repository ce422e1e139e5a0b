// csr_device.hip -- CSR construction from an edge list on the device, with the
// semantics of the reference's fill_data() (include/graph_io.h:21-130) and
// the same flags as gd_csr_from_edges (the host builder):
//
//   1. placement (graph_io.h:245-257): every edge pushes one record to the
//      row of its source (its destination with transpose), preceded by a
//      mirrored record when symmetrising; once a mirrored record has been
//      pushed the transpose flag stays cleared for the rest of the list (the
//      reference's loop resets it), so placement is a prefix sum over the
//      per-edge record counts plus the index of the first mirrored edge;
//   2. a stable radix sort of the records by row (by (row, column) when
//      `sorted`), so each row keeps its push order.  std::sort in the
//      reference is not stable: with `sorted` and duplicate edges of different
//      weights, the weight kept by step 4 may differ; the structure, and
//      unweighted graphs, are identical;
//   3. self-loops dropped (graph_io.h:32-45);
//   4. ADJACENT duplicates dropped, comparing with the previous kept record of
//      the row (graph_io.h:48-61);
//   5. row offsets from the row boundaries of the sorted records, degree =
//      row length (graph_io.h:72-78, :289-293).
//
// Two calls around the one point where the host must know the edge count:
// gd_csr_sort_edges (1, 2 and a count of the records that 3 and 4 keep) and
// gd_csr_finish (3, 4 and 5 in one pass into the caller's arrays), both in a
// workspace of the caller's.  A program that builds graphs repeatedly keeps
// that memory: allocating and freeing several GB per call costs far more than
// the build once the GPU has handed out its fresh memory (60 M edges: 11.5 ms
// per call while it had some, 173 ms after that).  The edge list never leaves
// HBM.
//
// What bounds it: the radix sort's passes over the records.  A record is one
// 64-bit key of exactly 2 * ceil(log2 m) bits (row and column side by side,
// so 44 bits sort in 6 byte passes instead of the 7 that a column in its own
// 32 bits takes), and the weight travels only where there is one.  Placement
// reads the edges once (checks included), and steps 3-5 read the sorted
// records twice (count, write) instead of two rounds of flags, scan and
// scatter.

#include <hip/hip_runtime.h>
#include <rocprim/device/device_scan.hpp>
#include <rocprim/device/device_radix_sort.hpp>

#include <algorithm>
#include <cstring>

#include "gardenia_hip.h"
#include "gd_common.h"

namespace gd {
namespace {

constexpr int kB = 256;
constexpr int kWaveRecs = 1024;  // records per wavefront of the count and write passes
constexpr int kEdgeBlock = 2048;  // edges per workgroup of the symmetrised placement

int grid_for(int64_t n) {
  return (int)std::max<int64_t>(1, std::min<int64_t>((n + kB - 1) / kB, 65536));
}

#define GRID_LOOP(i, n) \
  for (int64_t i = (int64_t)blockIdx.x * kB + threadIdx.x; i < (n); i += (int64_t)gridDim.x * kB)

// Device-side results of the build (one per workspace).
struct Scalars {
  unsigned long long first_mirror;  // first edge with a mirrored record
  int bad;                          // an endpoint outside [0, m)
  int pad;
};

__global__ void scalars_init_kernel(Scalars* s, unsigned long long n, int64_t* cnt_end) {
  s->first_mirror = n;
  s->bad = 0;
  s->pad = 0;
  if (cnt_end) *cnt_end = 0;
}

// A record's key: the part that is sorted in the high bits.  `sorted`: row,
// then column; else (column, row) sorted on the row's bits only.  bits =
// ceil(log2 m) of each.
struct KeyFormat {
  int bits;
  int sorted;
  __device__ __forceinline__ uint64_t make(int32_t r, int32_t c) const {
    const uint32_t hi = sorted ? r : c, lo = sorted ? c : r;
    return ((uint64_t)hi << bits) | lo;
  }
  __device__ __forceinline__ int32_t row(uint64_t k) const {
    return (int32_t)(sorted ? (k >> bits) : (k & ((1ull << bits) - 1)));
  }
  __device__ __forceinline__ int32_t col(uint64_t k) const {
    return (int32_t)(sorted ? (k & ((1ull << bits) - 1)) : (k >> bits));
  }
};

// Symmetrised lists: records pushed by each block of kEdgeBlock edges, the
// first edge with a mirrored record, the endpoint check.
__global__ __launch_bounds__(kB) void edge_count_kernel(int64_t n, const int32_t* __restrict__ src,
                                                        const int32_t* __restrict__ dst, int m,
                                                        int mirror, int64_t* __restrict__ cnt,
                                                        Scalars* __restrict__ sc) {
  __shared__ int s_cnt[kB / 64];
  __shared__ unsigned long long s_first[kB / 64];
  const int64_t e0 = (int64_t)blockIdx.x * kEdgeBlock;
  int c = 0, bad = 0;
  unsigned long long first = ~0ull;
  for (int64_t i = e0 + threadIdx.x; i < min(e0 + kEdgeBlock, n); i += kB) {
    const int32_t s = src[i], d = dst[i];
    bad |= (s < 0) | (s >= m) | (d < 0) | (d >= m);
    const int two = mirror || s != d;
    c += 1 + two;
    if (two) first = min(first, (unsigned long long)i);
  }
  for (int o = 32; o > 0; o >>= 1) {
    c += __shfl_xor(c, o, 64);
    first = min(first, (unsigned long long)__shfl_xor((long long)first, o, 64));
  }
  if (__any(bad) && (threadIdx.x & 63) == 0) atomicOr(&sc->bad, 1);
  if ((threadIdx.x & 63) == 0) {
    s_cnt[threadIdx.x / 64] = c;
    s_first[threadIdx.x / 64] = first;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int t = 0;
    unsigned long long f = ~0ull;
    for (int w = 0; w < kB / 64; w++) {
      t += s_cnt[w];
      f = min(f, s_first[w]);
    }
    cnt[blockIdx.x] = t;
    if (f != ~0ull) atomicMin(&sc->first_mirror, f);
  }
}

// Records in push order of a symmetrised list: each wavefront takes its
// block's edges 64 at a time in order, so an edge's records start at the
// block's base plus the records of the block's earlier edges.
__global__ __launch_bounds__(kB) void place_sym_kernel(
    int64_t n, const int32_t* __restrict__ src, const int32_t* __restrict__ dst,
    const float* __restrict__ wt, const int64_t* __restrict__ base, int mirror, int transpose,
    const Scalars* __restrict__ sc, KeyFormat kf, uint64_t* __restrict__ key,
    float* __restrict__ rw) {
  __shared__ int s_two[kEdgeBlock / 64];
  constexpr int kPer = kEdgeBlock / kB;  // steps of 64 edges per wavefront
  const int lane = threadIdx.x & 63, wid = threadIdx.x / 64;
  const int64_t e0 = (int64_t)blockIdx.x * kEdgeBlock;
  int32_t s[kPer], d[kPer];
  int two[kPer], before[kPer];
#pragma unroll
  for (int q = 0; q < kPer; q++) {
    const int g = wid * kPer + q;  // this wavefront's q-th group of 64 edges
    const int64_t i = e0 + g * 64 + lane;
    s[q] = i < n ? src[i] : 0;
    d[q] = i < n ? dst[i] : 0;
    two[q] = i < n && (mirror || s[q] != d[q]);
    const uint64_t b = __ballot(two[q]);
    before[q] = __popcll(b & ((1ull << lane) - 1));
    if (lane == 0) s_two[g] = __popcll(b);
  }
  __syncthreads();
  const unsigned long long fm = sc->first_mirror;
  const int64_t b0 = base[blockIdx.x];
  int extra = 0;
  for (int g = 0; g < wid * kPer; g++) extra += s_two[g];
#pragma unroll
  for (int q = 0; q < kPer; q++) {
    const int g = wid * kPer + q;
    const int64_t i = e0 + g * 64 + lane;
    if (i < n) {
      int64_t p = b0 + g * 64 + lane + extra + before[q];
      const float w = wt ? wt[i] : 1.0f;
      if (two[q]) {  // the mirrored record is pushed first
        key[p] = kf.make(d[q], s[q]);
        if (wt) rw[p] = w;
        p++;
      }
      const bool tr = transpose && (unsigned long long)i < fm;
      key[p] = tr ? kf.make(d[q], s[q]) : kf.make(s[q], d[q]);
      if (wt) rw[p] = w;
    }
    extra += s_two[g];
  }
}

// One record per edge (no symmetrising), with the endpoint check.
__global__ __launch_bounds__(kB) void place_kernel(int64_t n, const int32_t* __restrict__ src,
                                                   const int32_t* __restrict__ dst, int m,
                                                   int transpose, KeyFormat kf,
                                                   uint64_t* __restrict__ key,
                                                   Scalars* __restrict__ sc) {
  int bad = 0;
  GRID_LOOP(i, n) {
    const int32_t s = src[i], d = dst[i];
    bad |= (s < 0) | (s >= m) | (d < 0) | (d >= m);
    key[i] = transpose ? kf.make(d, s) : kf.make(s, d);
  }
  if (__any(bad) && (threadIdx.x & 63) == 0) atomicOr(&sc->bad, 1);
}

// The record of one lane, the same for all.
__device__ __forceinline__ uint64_t lane_record(uint64_t k, int lane) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)k, lane);
  return ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(k >> 32), lane) << 32) | lo;
}

// The last record before `i0` of row r that is no self-loop, by the wavefront:
// 1024 records a step, since a row may hold any number of them.
__device__ __forceinline__ bool last_no_loop(const uint64_t* __restrict__ key, int64_t i0, int32_t r,
                                             const KeyFormat& kf, uint64_t* rec) {
  const int lane = threadIdx.x & 63;
  for (int64_t e = i0; e > 0; e -= kWaveRecs) {
    uint64_t k[kWaveRecs / 64];
#pragma unroll
    for (int q = 0; q < kWaveRecs / 64; q++) k[q] = key[max(e - 1 - q * 64 - lane, (int64_t)0)];
#pragma unroll
    for (int q = 0; q < kWaveRecs / 64; q++) {
      const bool ends = kf.row(k[q]) != r || kf.col(k[q]) != r || e - 1 - q * 64 - lane <= 0;
      const uint64_t b = __ballot(ends);
      if (b) {
        *rec = lane_record(k[q], __builtin_ctzll(b));
        return kf.row(*rec) == r && kf.col(*rec) != r;
      }
    }
  }
  return false;
}

// The sorted records [1024 w, + 1024) in order, 64 at a time, by one wavefront:
// f(index, in range, record, row of the record before it or -1, kept).  Kept: not
// a self-loop (rm_self), and not equal to the last record before it that is no
// dropped self-loop (rm_dup).  That record is one of the 64, or carried from
// those before; only the wavefront's first record that is no loop may have to
// look back over loops before the wavefront, and not in rows sorted by column,
// where a row's records on the two sides of its loops differ.  (When every
// record looked back by itself, 200,000 loops of one vertex ahead of 1 M edges
// took 64 ms.)
template <class F>
__device__ __forceinline__ void for_records(int64_t n, int64_t w, const uint64_t* __restrict__ key,
                                            const KeyFormat& kf, int rm_self, int rm_dup, F f) {
  const int lane = threadIdx.x & 63;
  const int64_t i0 = w * kWaveRecs;
  auto loop = [&](uint64_t k) { return rm_self && kf.row(k) == kf.col(k); };
  uint64_t last = key[max(i0 - 1, (int64_t)0)];  // the last that is no loop, if there is one
  bool have = i0 > 0 && !loop(last);
  if (i0 > 0 && !have && rm_dup && !kf.sorted) {
    uint64_t b = 0;
    for (int64_t i = i0 + lane; !b && i - lane < min(i0 + kWaveRecs, n); i += 64) {
      const uint64_t k = key[min(i, n - 1)];
      b = __ballot(i < n && !loop(k));
      if (b) have = last_no_loop(key, i0, kf.row(lane_record(k, __builtin_ctzll(b))), kf, &last);
    }
  }
#pragma unroll 4
  for (int q = 0; q < kWaveRecs / 64; q++) {
    const int64_t i = i0 + q * 64 + lane;
    const uint64_t k = key[min(i, n - 1)], prev = key[max(min(i, n) - 1, (int64_t)0)];
    const bool in = i < n, real = in && !loop(k);
    const uint64_t b = __ballot(real);
    const uint64_t lower = b & ((1ull << lane) - 1);
    uint64_t near = prev;
    if (b != __ballot(in))  // a loop among the 64
      near = (uint64_t)__shfl((long long)k, lower ? 63 - __builtin_clzll(lower) : 0, 64);
    const bool twin = lower ? near == k : have && last == k;
    f(i, in, k, i > 0 ? kf.row(prev) : -1, real && !(rm_dup && twin));
    if (b) {
      last = lane_record(k, 63 - __builtin_clzll(b));
      have = true;
    }
  }
}

// cnt[w] = records kept among sorted records [1024 w, + 1024), one wavefront each.
__global__ __launch_bounds__(kB) void kept_count_kernel(int64_t n, int64_t waves,
                                                        const uint64_t* __restrict__ key,
                                                        KeyFormat kf, int rm_self, int rm_dup,
                                                        int64_t* __restrict__ cnt) {
  const int64_t w = (int64_t)blockIdx.x * (kB / 64) + threadIdx.x / 64;
  if (w >= waves) return;
  int c = 0;
  for_records(n, w, key, kf, rm_self, rm_dup,
              [&](int64_t, bool, uint64_t, int32_t, bool keep) { c += __popcll(__ballot(keep)); });
  if ((threadIdx.x & 63) == 0) cnt[w] = c;
}

// Writes the kept records (columns, weights) at their place, base[w] kept
// records before wavefront w's, and the row offsets: off[q] = records kept
// before the first record of a row >= q, set by the first record of each row
// for the rows since the previous record's (every entry is written once).
__global__ __launch_bounds__(kB) void kept_write_kernel(
    int64_t n, int64_t waves, int m, const uint64_t* __restrict__ key,
    const float* __restrict__ rw, KeyFormat kf, int rm_self, int rm_dup,
    const int64_t* __restrict__ base, int32_t* __restrict__ off, int32_t* __restrict__ col,
    float* __restrict__ wout) {
  const int lane = threadIdx.x & 63;
  const int64_t w = (int64_t)blockIdx.x * (kB / 64) + threadIdx.x / 64;
  if (w >= waves) return;
  int64_t at = base[w];
  for_records(n, w, key, kf, rm_self, rm_dup,
              [&](int64_t i, bool in, uint64_t k, int32_t prev, bool keep) {
                const uint64_t b = __ballot(keep);
                const int64_t p = at + __popcll(b & ((1ull << lane) - 1));
                at += __popcll(b);
                if (keep) {
                  col[p] = kf.col(k);
                  if (wout) wout[p] = rw ? rw[i] : 1.0f;
                }
                if (in) {
                  const int32_t r = kf.row(k);
                  for (int32_t t = prev + 1; t <= r; t++) off[t] = (int32_t)p;
                  if (i == n - 1)
                    for (int32_t t = r + 1; t <= m; t++) off[t] = (int32_t)(p + keep);
                }
              });
}

__global__ void fill_kernel(int64_t n, int32_t v, int32_t* __restrict__ a) { GRID_LOOP(i, n) a[i] = v; }

__global__ void degree_kernel(int m, const int32_t* __restrict__ off, int32_t* __restrict__ deg) {
  GRID_LOOP(i, m) deg[i] = off[i + 1] - off[i];
}

int sync_read(const void* dptr, void* h, size_t bytes, hipStream_t s) {
  GD_HIP_TRY(hipMemcpyAsync(h, dptr, bytes, hipMemcpyDeviceToHost, s));
  GD_HIP_TRY(hipStreamSynchronize(s));
  return GD_OK;
}

int bits_for(int m) {
  int bits = 1;
  while (bits < 31 && ((int64_t)1 << bits) < m) bits++;
  return bits;
}

// Where everything lies in the workspace (byte offsets, 256-byte aligned).
struct Layout {
  int64_t cap = 0;   // records at most
  int64_t cnts = 0;  // counters: per edge block or per wavefront of records
  size_t scalars = 0, cnt = 0, base = 0, keys[2] = {0, 0}, wts[2] = {0, 0}, tmp = 0;
  size_t tmp_bytes = 0, total = 0;
};

int layout(int m, int64_t n, bool weights, bool sym, bool sorted, Layout* L) {
  size_t at = 0;
  auto take = [&](size_t bytes) {
    const size_t p = at;
    at += (bytes + 255) & ~(size_t)255;
    return p;
  };
  L->cap = sym ? 2 * n : n;
  const int64_t blocks = (n + kEdgeBlock - 1) / kEdgeBlock;
  const int64_t waves = (L->cap + kWaveRecs - 1) / kWaveRecs;
  L->cnts = std::max<int64_t>(sym ? blocks : 0, waves) + 1;
  L->scalars = take(sizeof(Scalars));
  L->cnt = take(8 * (size_t)L->cnts);
  L->base = take(8 * (size_t)L->cnts);
  const size_t capb = (size_t)std::max<int64_t>(L->cap, 1);
  for (int q = 0; q < 2; q++) L->keys[q] = take(8 * capb);
  for (int q = 0; q < 2; q++) L->wts[q] = weights ? take(4 * capb) : 0;
  size_t scan = 0, sort = 0;
  GD_HIP_TRY(rocprim::exclusive_scan(nullptr, scan, (int64_t*)nullptr, (int64_t*)nullptr,
                                     (int64_t)0, (size_t)L->cnts, rocprim::plus<int64_t>()));
  const int bits = bits_for(m), end = sorted ? 2 * bits : bits;
  rocprim::double_buffer<uint64_t> k(nullptr, nullptr);
  if (weights) {
    rocprim::double_buffer<float> v(nullptr, nullptr);
    GD_HIP_TRY(rocprim::radix_sort_pairs(nullptr, sort, k, v, capb, 0, end));
  } else {
    GD_HIP_TRY(rocprim::radix_sort_keys(nullptr, sort, k, capb, 0, end));
  }
  L->tmp_bytes = std::max(scan, sort);
  L->tmp = take(std::max<size_t>(L->tmp_bytes, 1));
  L->total = at;
  return GD_OK;
}

int scan_counts(char* ws, const Layout& L, int64_t n, hipStream_t s) {
  size_t bytes = L.tmp_bytes;
  GD_HIP_TRY(rocprim::exclusive_scan(ws + L.tmp, bytes, (int64_t*)(ws + L.cnt),
                                     (int64_t*)(ws + L.base), (int64_t)0, (size_t)n,
                                     rocprim::plus<int64_t>(), s));
  return GD_OK;
}

int sort_edges(int m, int64_t n, const int32_t* d_src, const int32_t* d_dst, const float* d_wt,
               char* ws, const Layout& L, hipStream_t s, gd_csr_job* job) {
  const bool sym = job->symmetrize, sorted = job->sorted;
  Scalars* sc = (Scalars*)(ws + L.scalars);
  int64_t* cnt = (int64_t*)(ws + L.cnt);
  uint64_t* key = (uint64_t*)(ws + L.keys[0]);
  float* wt = d_wt ? (float*)(ws + L.wts[0]) : nullptr;
  const KeyFormat kf{bits_for(m), sorted};
  int64_t cap = n;
  const int64_t blocks = (n + kEdgeBlock - 1) / kEdgeBlock;
  hipLaunchKernelGGL(scalars_init_kernel, dim3(1), dim3(1), 0, s, sc, (unsigned long long)n,
                     sym ? cnt + blocks : nullptr);
  if (sym) {
    hipLaunchKernelGGL(edge_count_kernel, dim3((unsigned)blocks), dim3(kB), 0, s, n, d_src, d_dst,
                       m, job->mirror_selfloops, cnt, sc);
    GD_HIP_TRY(hipGetLastError());
    int rc = scan_counts(ws, L, blocks + 1, s);
    Scalars h;
    if (!rc) GD_HIP_TRY(hipMemcpyAsync(&h, sc, sizeof(h), hipMemcpyDeviceToHost, s));
    if (!rc) rc = sync_read((int64_t*)(ws + L.base) + blocks, &cap, 8, s);
    if (rc) return rc;
    GD_CHECK_ARG(h.bad == 0, "edge endpoint out of range [0, m)");
    GD_CHECK_ARG(cap < (1ll << 31), "more than 2^31 - 1 edges after symmetrisation");
    hipLaunchKernelGGL(place_sym_kernel, dim3((unsigned)blocks), dim3(kB), 0, s, n, d_src, d_dst,
                       d_wt, (int64_t*)(ws + L.base), job->mirror_selfloops, job->transpose, sc,
                       kf, key, wt);
  } else {
    hipLaunchKernelGGL(place_kernel, dim3(grid_for(n)), dim3(kB), 0, s, n, d_src, d_dst, m,
                       job->transpose, kf, key, sc);
    if (wt) GD_HIP_TRY(hipMemcpyAsync(wt, d_wt, 4 * (size_t)n, hipMemcpyDeviceToDevice, s));
  }
  GD_HIP_TRY(hipGetLastError());
  const int end = sorted ? 2 * kf.bits : kf.bits;
  rocprim::double_buffer<uint64_t> k(key, (uint64_t*)(ws + L.keys[1]));
  rocprim::double_buffer<float> v(wt, wt ? (float*)(ws + L.wts[1]) : nullptr);
  auto sort = [&](void* tmp, size_t& bytes) {
    return wt ? rocprim::radix_sort_pairs(tmp, bytes, k, v, (size_t)cap, 0, end, s)
              : rocprim::radix_sort_keys(tmp, bytes, k, (size_t)cap, 0, end, s);
  };
  size_t bytes = 0;
  GD_HIP_TRY(sort(nullptr, bytes));
  DeviceBuffer more;  // fewer records than the layout's may take another algorithm's scratch
  if (bytes > L.tmp_bytes) {
    const int rc = more.alloc(bytes);
    if (rc) return rc;
  }
  GD_HIP_TRY(sort(more.ptr ? more.ptr : ws + L.tmp, bytes));
  job->weights = wt ? v.current() : nullptr;
  job->keys = k.current();
  job->records = cap;
  const int64_t waves = (cap + kWaveRecs - 1) / kWaveRecs;
  GD_HIP_TRY(hipMemsetAsync(cnt + waves, 0, 8, s));
  hipLaunchKernelGGL(kept_count_kernel, dim3((unsigned)((waves + 3) / 4)), dim3(kB), 0, s, cap,
                     waves, (const uint64_t*)job->keys, kf, job->remove_selfloops,
                     job->remove_redundents, cnt);
  GD_HIP_TRY(hipGetLastError());
  int rc = scan_counts(ws, L, waves + 1, s);
  Scalars h;
  if (!rc) GD_HIP_TRY(hipMemcpyAsync(&h, sc, sizeof(h), hipMemcpyDeviceToHost, s));
  if (!rc) rc = sync_read((int64_t*)(ws + L.base) + waves, &job->nnz, 8, s);
  if (rc) return rc;
  GD_CHECK_ARG(h.bad == 0, "edge endpoint out of range [0, m)");
  job->base = (int64_t*)(ws + L.base);
  return GD_OK;
}

}  // namespace
}  // namespace gd

using namespace gd;

extern "C" {

int gd_csr_workspace(int m, int64_t n, int have_weight, int symmetrize, int sorted,
                     size_t* bytes) {
  GD_CHECK_ARG(bytes != nullptr, "NULL output");
  GD_CHECK_ARG(m >= 0 && n >= 0 && n < (1ll << 31), "m / n out of range");
  if (gd_device_count() <= 0) {
    set_error("no HIP device visible");
    return GD_ERR_NO_DEVICE;
  }
  Layout L;
  const int rc = layout(m, n, have_weight != 0, symmetrize != 0, sorted != 0, &L);
  *bytes = L.total;
  return rc;
}

int gd_csr_sort_edges(int m, int64_t n, const int32_t* d_src, const int32_t* d_dst,
                      const float* d_wt, int symmetrize, int transpose, int sorted,
                      int remove_selfloops, int remove_redundents, int mirror_selfloops,
                      void* d_workspace, size_t workspace_bytes, void* stream, gd_csr_job* job) {
  GD_CHECK_ARG(job != nullptr, "NULL output");
  memset(job, 0, sizeof(*job));
  GD_CHECK_ARG(m >= 0 && n >= 0 && n < (1ll << 31), "m / n out of range");
  GD_CHECK_ARG(n == 0 || (d_src && d_dst), "NULL edge arrays");
  if (gd_device_count() <= 0) {
    set_error("no HIP device visible");
    return GD_ERR_NO_DEVICE;
  }
  gd_csr_job j;
  memset(&j, 0, sizeof(j));
  j.m = m;
  j.symmetrize = symmetrize != 0;
  j.transpose = transpose != 0;
  j.sorted = sorted != 0;
  j.remove_selfloops = remove_selfloops != 0;
  j.remove_redundents = remove_redundents != 0;
  j.mirror_selfloops = mirror_selfloops != 0;
  if (n > 0) {
    Layout L;
    int rc = layout(m, n, d_wt != nullptr, j.symmetrize, j.sorted, &L);
    if (rc) return rc;
    GD_CHECK_ARG(d_workspace != nullptr && workspace_bytes >= L.total &&
                     ((uintptr_t)d_workspace & 255) == 0,
                 "workspace too small or not 256-byte aligned");
    rc = sort_edges(m, n, d_src, d_dst, d_wt, (char*)d_workspace, L, (hipStream_t)stream, &j);
    if (rc) return rc;
  }
  *job = j;
  return GD_OK;
}

int gd_csr_finish(const gd_csr_job* job, int32_t* d_off, int32_t* d_col, float* d_weight,
                  int32_t* d_degree, void* stream) {
  GD_CHECK_ARG(job != nullptr && d_off != nullptr, "NULL argument");
  GD_CHECK_ARG(job->nnz == 0 || d_col != nullptr, "NULL column output");
  GD_CHECK_ARG(job->m == 0 || d_degree != nullptr, "NULL degree output");
  hipStream_t s = (hipStream_t)stream;
  const int m = job->m;
  if (job->records > 0) {
    const int64_t waves = (job->records + kWaveRecs - 1) / kWaveRecs;
    const KeyFormat kf{bits_for(m), job->sorted};
    hipLaunchKernelGGL(kept_write_kernel, dim3((unsigned)((waves + 3) / 4)), dim3(kB), 0, s,
                       job->records, waves, m, (const uint64_t*)job->keys,
                       (const float*)job->weights, kf, job->remove_selfloops,
                       job->remove_redundents, (const int64_t*)job->base, d_off, d_col, d_weight);
  } else {
    hipLaunchKernelGGL(fill_kernel, dim3(grid_for((int64_t)m + 1)), dim3(kB), 0, s,
                       (int64_t)m + 1, 0, d_off);
  }
  if (m > 0)
    hipLaunchKernelGGL(degree_kernel, dim3(grid_for(m)), dim3(kB), 0, s, m, d_off, d_degree);
  GD_HIP_TRY(hipGetLastError());
  return GD_OK;
}

int gd_csr_from_edges_device(int m, int64_t n, const int32_t* d_src, const int32_t* d_dst,
                             const float* d_wt, int symmetrize, int transpose, int sorted,
                             int remove_selfloops, int remove_redundents, int mirror_selfloops,
                             void* stream, gd_device_csr* out) {
  GD_CHECK_ARG(out != nullptr, "NULL output");
  memset(out, 0, sizeof(*out));
  GD_CHECK_ARG(m >= 0 && n >= 0 && n < (1ll << 31), "m / n out of range");
  GD_CHECK_ARG(n == 0 || (d_src && d_dst), "NULL edge arrays");
  DeviceBuffer ws, off, col, wout, deg;
  size_t bytes = 0;
  int rc = gd_csr_workspace(m, n, d_wt != nullptr, symmetrize, sorted, &bytes);
  if (!rc) rc = ws.alloc(bytes);
  if (rc) return rc;
  gd_csr_job job;
  rc = gd_csr_sort_edges(m, n, d_src, d_dst, d_wt, symmetrize, transpose, sorted, remove_selfloops,
                         remove_redundents, mirror_selfloops, ws.ptr, bytes, stream, &job);
  if (!rc) rc = off.alloc(4 * ((size_t)m + 1));
  if (!rc) rc = col.alloc(4 * (size_t)std::max<int64_t>(job.nnz, 1));
  if (!rc) rc = wout.alloc(4 * (size_t)std::max<int64_t>(job.nnz, 1));
  if (!rc) rc = deg.alloc(4 * (size_t)std::max(m, 1));
  if (!rc)
    rc = gd_csr_finish(&job, off.as<int32_t>(), col.as<int32_t>(), wout.as<float>(),
                       deg.as<int32_t>(), stream);
  if (rc) return rc;
  GD_HIP_TRY(hipStreamSynchronize((hipStream_t)stream));  // the workspace is freed on return
  out->m = m;
  out->nnz = job.nnz;
  out->row_offsets = off.as<int32_t>();
  out->column_indices = col.as<int32_t>();
  out->weight = wout.as<float>();
  out->degree = deg.as<int32_t>();
  off.ptr = col.ptr = wout.ptr = deg.ptr = nullptr;  // ownership moves to *out
  return GD_OK;
}

int gd_device_csr_copy(const gd_device_csr* c, int32_t* d_off, int32_t* d_col, float* d_w,
                       int32_t* d_deg, void* stream) {
  GD_CHECK_ARG(c != nullptr, "NULL csr");
  hipStream_t s = (hipStream_t)stream;
  const size_t m = (size_t)c->m, nnz = (size_t)c->nnz;
  if (d_off) GD_HIP_TRY(hipMemcpyAsync(d_off, c->row_offsets, 4 * (m + 1), hipMemcpyDeviceToDevice, s));
  if (d_col && nnz)
    GD_HIP_TRY(hipMemcpyAsync(d_col, c->column_indices, 4 * nnz, hipMemcpyDeviceToDevice, s));
  if (d_w && nnz) GD_HIP_TRY(hipMemcpyAsync(d_w, c->weight, 4 * nnz, hipMemcpyDeviceToDevice, s));
  if (d_deg && m) GD_HIP_TRY(hipMemcpyAsync(d_deg, c->degree, 4 * m, hipMemcpyDeviceToDevice, s));
  return GD_OK;
}

int gd_device_csr_free(gd_device_csr* c) {
  if (!c) return GD_OK;
  for (void* p : {(void*)c->row_offsets, (void*)c->column_indices, (void*)c->weight,
                  (void*)c->degree})
    if (p) (void)hipFree(p);
  memset(c, 0, sizeof(*c));
  return GD_OK;
}

}  // extern "C"
