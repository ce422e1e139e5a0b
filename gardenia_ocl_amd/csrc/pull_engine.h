// pull_engine.h -- device building blocks of the CSR pull engine (wave64).
//
// A workgroup of NB threads (kBlock = 256 by default) owns one Tile of up to
// NB*IPT edges and 4*NB rows.  Latency is paid once per tile:
// every load the tile needs (edge indices, row offsets, the epilogue's
// per-row operands) is issued unconditionally up front -- addresses of idle
// lanes are clamped into the tile instead of branching -- and only then does
// the tile wait, gather (IPT independent gathers in flight per thread), stage
// the gathered values in LDS and reduce rows:
//   * rows of <= kSeqRow edges: the owning thread, sequentially in CSR order
//     (the reference's summation order, so the result is bit-identical);
//   * longer rows: one wavefront, lane-strided partials + xor butterfly; the
//     sum goes back through LDS to the owning thread for the epilogue.
// Hub segments gather kBlock*IPT edges of one long row into a partial sum.
//
// Row r of the tile is owned by thread (r - r0) % NB, so per-row reads and
// writes are coalesced.
#ifndef GD_PULL_ENGINE_H_
#define GD_PULL_ENGINE_H_

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "gd_common.h"

namespace gd {

constexpr int kBlock = 256;
constexpr int kWave = 64;
constexpr int kWaves = kBlock / kWave;
constexpr int kRowsPerThread = 4;  // rows per thread of a row tile (any block size)
constexpr int kTileRows = kRowsPerThread * kBlock;
constexpr int kOffLoads = kRowsPerThread + 1;  // ceil((rows + 1) / threads)
constexpr int kSeqRow = 64;

// Loads / stores of arrays streamed once per launch.  With NT the accesses
// carry the non-temporal hint, so the 1 GB-per-iteration index stream does not
// evict the cache-resident part of the gathered vector.
template <bool NT, typename T>
__device__ __forceinline__ T ld_stream(const T* p) {
  if constexpr (NT)
    return __builtin_nontemporal_load(p);
  else
    return *p;
}

template <bool NT, typename T>
__device__ __forceinline__ void st_stream(T* p, T v) {
  if constexpr (NT)
    __builtin_nontemporal_store(v, p);
  else
    *p = v;
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
  return v;
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
  return v;
}

// Sum of one value per thread over a workgroup of NWAVES waves, fixed order;
// result valid in thread 0.  `s_tmp` holds NWAVES values.
template <int NWAVES, typename T>
__device__ __forceinline__ T block_sum(T v, T* s_tmp) {
  v = wave_sum(v);
  const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
  if (lane == 0) s_tmp[wid] = v;
  __syncthreads();
  T t = T(0);
  if (threadIdx.x == 0)
#pragma unroll
    for (int w = 0; w < NWAVES; w++) t += s_tmp[w];
  return t;
}

// s + the first nb blocks of 4*kQ floats of v, in order with FP32 rounding, by
// the calling lane, from 16-byte aligned LDS: the next block's reads in flight
// while the current one is added (the adds are one dependent chain).
// kQ = 8 (reads 32 terms ahead) hides the LDS latency behind the chain: at
// RMAT-24 the pull phase took 1.339 ms against 1.367 ms with kQ = 4, at
// RMAT-16 32.8 against 35.5 us per iteration; kQ = 12 was no faster and costs
// the row tiles 24 more VGPRs.
template <int kQ>  // float4 reads per block
__device__ __forceinline__ float lane_chain(float s, const float4* __restrict__ v4, int nb) {
  float4 A[kQ], B[kQ];
  auto load = [&](float4(&R)[kQ], int blk) {
#pragma unroll
    for (int k = 0; k < kQ; k++) R[k] = v4[blk * kQ + k];
  };
  auto add = [&](const float4(&R)[kQ]) {
#pragma unroll
    for (int k = 0; k < kQ; k++) {
      s += R[k].x;
      s += R[k].y;
      s += R[k].z;
      s += R[k].w;
    }
  };
  if (nb > 0) {
    load(A, 0);
    int b = 0;
    // scheduling barriers keep each block's reads issued before the previous
    // block's adds, so the adds wait only for reads issued one block earlier
    for (; b + 2 <= nb; b += 2) {
      load(B, b + 1);
      __builtin_amdgcn_sched_barrier(0);
      add(A);
      __builtin_amdgcn_sched_barrier(0);
      load(A, min(b + 2, nb - 1));  // unconditional (clamped): A and B keep their registers
      __builtin_amdgcn_sched_barrier(0);
      add(B);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (b < nb) add(A);
  }
  return s;
}

// s + v[0] + ... + v[n-1], v 16-byte aligned.
template <int kQ>
__device__ __forceinline__ float lane_seq_sum(float s, const float* __restrict__ v, int n) {
  const int nb = n / (4 * kQ);
  s = lane_chain<kQ>(s, reinterpret_cast<const float4*>(v), nb);
  for (int i = nb * 4 * kQ; i < n; i++) s += v[i];
  return s;
}

// Sequential sum s + v[b] + ... + v[e-1] from LDS (`v` 16-byte aligned, the
// granule of 4 that holds e - 1 readable) by the calling lane, in order with
// FP32 rounding.  All reads are whole granules, issued ahead of the adds that
// need them; terms outside the row are replaced by -0.0, which added to any s
// gives s.  (Reading the ends of a row term by term made each of up to 34 terms
// wait for its own LDS read: the sums took 4-7 us of a row tile's 11-16 us.)
//
// seq_sum, for plans of many iterations over one graph: little code, since a
// launch of a few tiles waits for its instructions most of the time.  Rows of
// more than kChainRow terms take the first granule, blocks of 8 (lane_chain) and
// the rest a granule at a time; shorter ones all of it that way, two granules
// read ahead.
// seq_sum_wide, for the others (SpMV, the adjoint): blocks of 4 granules
// double-buffered, up to 4 granules at the end, unrolled.
// us, seq_sum / seq_sum_wide: 20 PageRank iterations on 3,000 vertices x 24 264 /
// 298, 9,001 x 32 298 / 350, 1,000 x 4 206 / 215; 64 graphs 3750 / 3851; but SpMV
// 2^22 x 32 548 / 537, weighted RMAT-20 16,410 / 16,220.
constexpr int kChainRow = 48;

__device__ __forceinline__ float seq_sum(float s, const float* __restrict__ v, int b, int e) {
  if (b >= e) return s;
  const float4* __restrict__ v4 = reinterpret_cast<const float4*>(v);
  const int g1 = (e + 3) >> 2;
  int g = b >> 2;
  auto add = [&](const float4& x) {  // granule g
    const unsigned n = (unsigned)(e - b), o = (unsigned)(4 * g - b);
    s += o < n ? x.x : -0.0f;
    s += o + 1u < n ? x.y : -0.0f;
    s += o + 2u < n ? x.z : -0.0f;
    s += o + 3u < n ? x.w : -0.0f;
    g++;
  };
  if (e - b > kChainRow) {
    add(v4[g]);
    const int nb = ((e >> 2) - g) >> 3;
    s = lane_chain<8>(s, v4 + g, nb);
    g += 8 * nb;
    if (g >= g1) return s;
  }
  float4 x = v4[g], y = v4[min(g + 1, g1 - 1)];
#pragma unroll 1
  do {
    const float4 z = v4[min(g + 2, g1 - 1)];
    add(x);
    x = y;
    y = z;
  } while (g < g1);
  return s;
}

__device__ __forceinline__ float seq_sum_wide(float s, const float* __restrict__ v, int b, int e) {
  if (b >= e) return s;
  const float4* __restrict__ v4 = reinterpret_cast<const float4*>(v);
  const int g1 = (e + 3) >> 2, m0 = (b >> 2) + 1;
  const int nb = max((e >> 2) - m0, 0) >> 2;
  const int t0 = m0 + 4 * nb;
  const float4 h = v4[m0 - 1];
  float4 A[4], B[4];
  auto load = [&](float4(&R)[4], int g) {
#pragma unroll
    for (int k = 0; k < 4; k++) R[k] = v4[min(g + k, g1 - 1)];
  };
  load(A, m0);  // the first block, or the last granules
  auto masked = [&](const float4& x, int i) {  // the granule at term i
    const unsigned n = (unsigned)(e - b), o = (unsigned)(i - b);
    s += o < n ? x.x : -0.0f;
    s += o + 1u < n ? x.y : -0.0f;
    s += o + 2u < n ? x.z : -0.0f;
    s += o + 3u < n ? x.w : -0.0f;
  };
  masked(h, 4 * (m0 - 1));
  auto add = [&](const float4(&R)[4]) {
#pragma unroll
    for (int q = 0; q < 4; q++) {
      s += R[q].x;
      s += R[q].y;
      s += R[q].z;
      s += R[q].w;
    }
  };
  int k = 0;
  for (; k + 2 <= nb; k += 2) {
    load(B, m0 + 4 * (k + 1));
    __builtin_amdgcn_sched_barrier(0);
    add(A);
    __builtin_amdgcn_sched_barrier(0);
    load(A, m0 + 4 * (k + 2));
    __builtin_amdgcn_sched_barrier(0);
    add(B);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (k < nb) {
    load(B, t0);
    add(A);
#pragma unroll
    for (int q = 0; q < 4; q++) A[q] = B[q];
  }
#pragma unroll
  for (int q = 0; q < 4; q++)
    if (t0 + q < g1) masked(A[q], 4 * (t0 + q));
  return s;
}

// ---------------------------------------------------------------------------
// Sequential-order sums of long rows in parallel.
//
// wave_exact_seg / exact_row_sum return s0 + v[0] + v[1] + ... + v[n-1]
// rounded exactly as the sequential FP32 loop `s = s0; for (i) s += v[i];`
// rounds it (the reference's per-row loop, src/pr/omp_base.cc:34-37):
//   While the running sum s > 0 lies in one binade [B, 2B) and no term is
//   negative, a step s + v advances s by a whole number of ulps that depends
//   on v and, through ties (round to even), on the parity of s alone.  So a
//   lane adds its terms in FP32 twice, from B and from B + ulp; the two
//   advances are its map of the running value (Steps), the hardware having
//   rounded every step.  Maps compose into maps of the same form, and a
//   prefix over the lanes' maps gives the running value after every lane's
//   terms; where no lane's advance depends on the parity (most wavefronts of
//   a long row) it is a prefix of integers.
//   The running values never decrease, so the binade holds up to a lane
//   exactly when the value after that lane is below 2B.  The first lane past
//   it, or one with a negative term, adds its terms from the running value
//   itself, and the prefix restarts after it in the new binade.  inf and NaN
//   terms carry a lane past any binade.  A zero s skips to the first nonzero
//   term; a subnormal, negative or non-finite s takes a lane's terms as they
//   are.
// For sums of positive terms (PageRank) the restarts are the ~log2(n) binade
// crossings.  A pass over 16 terms a lane is 32 FP32 additions and the prefix
// (about 0.3 us per 1024 terms); one lane's dependent chain costs about 3 ns
// per term, and the form before this one, which rounded each term to ulps in
// integers and checked every running value, about 1,230 vector instructions
// a pass: the 48,023-edge hub of a 1 M-vertex RMAT graph took 67 us of a
// staged 84-us iteration.
// ---------------------------------------------------------------------------

constexpr int kScanPT = 16;                   // terms per thread per chunk
constexpr int kScanChunk = kBlock * kScanPT;  // 4096
constexpr uint32_t kBinade = 1u << 23;        // ulps from a binade's start to its end

// A run of steps as one map of the running value x, in ulps: x -> x + a0 for
// even x, x + a1 for odd x.
struct Steps {
  uint32_t a0, a1;
};

__device__ __forceinline__ Steps compose(Steps p, Steps q) {  // p, then q
  const uint32_t d = q.a0 ^ q.a1;  // selects without branches: q.a1 = q.a0 ^ d
  return Steps{p.a0 + (q.a0 ^ (d & (0u - (p.a0 & 1u)))), p.a1 + (q.a1 ^ (d & (0u - (p.a1 & 1u))))};
}
__device__ __forceinline__ uint32_t apply(Steps p, uint32_t x) {
  return x + (p.a0 ^ ((p.a0 ^ p.a1) & (0u - (x & 1u))));
}

// Inclusive prefixes over the 64 lanes of a wavefront: DPP row shifts inside
// each row of 16 lanes, then row broadcasts across rows (lanes whose source
// is outside the row read 0, the identity).
#define GD_DPP(V, CTRL, ROWS) \
  (uint32_t) __builtin_amdgcn_update_dpp(0, (int)(V), CTRL, ROWS, 0xf, false)
#define GD_SCAN_STEPS(STEP)                                                              \
  STEP(0x111, 0xf) STEP(0x112, 0xf) STEP(0x114, 0xf) STEP(0x118, 0xf) /* row_shr:1,2,4,8 */ \
  STEP(0x142, 0xa) STEP(0x143, 0xc) /* row_bcast:15 -> rows 1, 3; row_bcast:31 -> rows 2, 3 */

__device__ __forceinline__ uint32_t wave_incl_scan_add(uint32_t x) {
#define GD_STEP(CTRL, ROWS) x += GD_DPP(x, CTRL, ROWS);
  GD_SCAN_STEPS(GD_STEP)
#undef GD_STEP
  return x;
}

__device__ __forceinline__ Steps wave_incl_scan_steps(Steps x) {
#define GD_STEP(CTRL, ROWS) x = compose(Steps{GD_DPP(x.a0, CTRL, ROWS), GD_DPP(x.a1, CTRL, ROWS)}, x);
  GD_SCAN_STEPS(GD_STEP)
#undef GD_STEP
  return x;
}
#undef GD_SCAN_STEPS
#undef GD_DPP

// Wavefront-uniform values kept in scalar registers.
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ float uniform(float v) {
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}
__device__ __forceinline__ uint32_t read_lane(uint32_t v, int lane) {
  return (uint32_t)__builtin_amdgcn_readlane((int)v, lane);
}

// s > 0 is a normal number; its binade starts at binade(s), and it lies
// ulps(s) >= 2^23 ulps above zero.  Inside one binade the bits of a float
// count ulps.
__device__ __forceinline__ bool in_binade(float s) {
  const uint32_t b = __float_as_uint(s);
  return b >= kBinade && b < 0x7f800000u;
}
__device__ __forceinline__ uint32_t binade(float s) { return __float_as_uint(s) & 0x7f800000u; }

// Some term of the lane has its sign bit set.
template <int K>
__device__ __forceinline__ bool lane_negative(const float (&v)[K]) {
  uint32_t b = 0u;
#pragma unroll
  for (int k = 0; k < K; k++) b |= __float_as_uint(v[k]);
  return b >> 31;
}

// The inclusive prefix of the wavefront's maps in the binade that starts at
// the float bits `base`.  Inactive lanes are identities.  `stop`: the lane is
// negative or leaves a binade by itself; such a lane counts as a binade, so
// lanes before the first stop see sums below 2^30.
template <int K>
__device__ __forceinline__ Steps wave_steps(const float (&v)[K], bool active, bool negative,
                                            uint32_t base, bool& stop) {
  float x0 = __uint_as_float(base), x1 = __uint_as_float(base + 1u);
#pragma unroll
  for (int k = 0; k < K; k++) {
    x0 += v[k];
    x1 += v[k];
  }
  Steps L{__float_as_uint(x0) - base, __float_as_uint(x1) - (base + 1u)};
  stop = negative || L.a0 >= kBinade - 1u || L.a1 >= kBinade - 1u;
  if (stop) L = Steps{kBinade, kBinade};
  if (!active) L = Steps{0u, 0u};
  stop = stop && active;
  if (__ballot(L.a0 != L.a1)) return wave_incl_scan_steps(L);
  const uint32_t a = wave_incl_scan_add(L.a0);
  return Steps{a, a};
}

// s + the wavefront's terms in lane order (lane l: v[0..K-1] are terms l*K ..
// l*K+K-1; missing terms 0), rounded as the sequential loop.  The whole
// wavefront calls it with one s; every pass finishes a lane, so it ends.
template <int K>
__device__ __forceinline__ float wave_exact_seg(float s, const float (&v)[K]) {
  const int lane = threadIdx.x & (kWave - 1);
  const bool negative = lane_negative<K>(v);
  s = uniform(s);
  // Terms of both signs: a lane at a time from the start, nothing else in the
  // loop (weighted PageRank, RMAT of 100,000 vertices, 2 percent of the weights
  // negative, 20 iterations and the gradient: 1,473 us, 2,584 in the loop below).
  if (__popcll(__ballot(negative)) > 4) {
#pragma unroll 2
    for (int f = 0; f < kWave; f++) {
      float t = s;
#pragma unroll
      for (int k = 0; k < K; k++) t += v[k];
      s = __uint_as_float(read_lane(__float_as_uint(t), f));
    }
    return s;
  }
  int from = 0;  // lanes before it are added
  for (;;) {
    int f = from;
    if (in_binade(s)) {
      const uint32_t base = binade(s), at = __float_as_uint(s) - base;
      bool stop;
      const Steps inc = wave_steps<K>(v, lane >= from, negative, base, stop);
      const uint32_t r = apply(inc, at);
      const uint64_t m = __ballot(stop || r >= kBinade);
      if (!m) return __uint_as_float(base + read_lane(r, kWave - 1));
      f = __builtin_ctzll(m);
      if (f > 0) s = __uint_as_float(base + read_lane(r, f - 1));
    } else if (__float_as_uint(s) == 0u) {
      uint32_t any = 0u;
#pragma unroll
      for (int k = 0; k < K; k++) any |= __float_as_uint(v[k]) << 1;
      const uint64_t m = __ballot(lane >= from && any != 0u);
      if (!m) return s;
      f = __builtin_ctzll(m);
    }
    float t = s;  // lane f's terms from s (every lane computes its own)
#pragma unroll
    for (int k = 0; k < K; k++) t += v[k];
    s = __uint_as_float(read_lane(__float_as_uint(t), f));
    from = f + 1;
    if (from >= kWave) return s;
  }
}

// The whole row v[b, e) of LDS (`v` 16-byte aligned) by one wavefront: the
// first terms, where s crosses a binade every few terms, as a plain chain,
// then 256 terms a pass, then 1024.
constexpr int kRowHead = 64;

template <int K>
__device__ __forceinline__ void wave_terms(const float* __restrict__ v, int i, int e,
                                           float (&t)[K]) {
  const int at = i + (threadIdx.x & (kWave - 1)) * K;
#pragma unroll
  for (int k = 0; k < K; k += 4) {
    const float4 x = *reinterpret_cast<const float4*>(v + (at + k < e ? at + k : i));
    t[k] = at + k < e ? x.x : 0.0f;
    t[k + 1] = at + k + 1 < e ? x.y : 0.0f;
    t[k + 2] = at + k + 2 < e ? x.z : 0.0f;
    t[k + 3] = at + k + 3 < e ? x.w : 0.0f;
  }
}

__device__ __forceinline__ float wave_exact_row(float s, const float* __restrict__ v, int b, int e) {
  int i = min(e, (b + kRowHead) & ~3);
  s = seq_sum(s, v, b, i);
  while (i < e && (i < b + 512 || e - i <= 512)) {
    float t[4];
    wave_terms<4>(v, i, e, t);
    s = wave_exact_seg<4>(s, t);
    i += 4 * kWave;
  }
  while (i < e) {
    float t[kScanPT];
    wave_terms<kScanPT>(v, i, e, t);
    s = wave_exact_seg<kScanPT>(s, t);
    i += kScanPT * kWave;
  }
  return s;
}

struct ExactLds {
  Steps tot[2][kWaves];  // wave totals of the maps, by pass parity
  int stop[2][kWaves];   // the wave has a stop of its own
  float s[2];
};

// s + one chunk of the row, thread t's terms being its 16t .. 16t+15 (v,
// missing terms 0).  The waves' totals in s's binade are combined in order;
// a wave in which the binade ends (or that holds a negative term) adds its
// terms by itself, and the waves after it go on in the new binade.  Every
// pass finishes a wave.  `pass` counts the workgroup's passes (the parity of
// the buffers: one barrier apart, a buffer is written again two passes later).
__device__ __forceinline__ float exact_scan_chunk(const float (&v)[kScanPT], float s, int& pass,
                                                  ExactLds& x) {
  const int lane = threadIdx.x & (kWave - 1);
  const int wid = uniform((int)(threadIdx.x / kWave));
  const bool negative = lane_negative<kScanPT>(v);
  int fw = 0;  // waves before it are added
  s = uniform(s);
  while (fw < kWaves) {
    int w = fw;
    if (in_binade(s)) {
      const uint32_t base = binade(s);
      const int p = pass & 1;
      pass++;
      if (wid >= fw) {
        bool stop;
        const Steps inc = wave_steps<kScanPT>(v, true, negative, base, stop);
        const int any = __ballot(stop) != 0;
        if (lane == kWave - 1) {
          x.tot[p][wid] = inc;
          x.stop[p][wid] = any;
        }
      }
      __syncthreads();
      uint32_t at = __float_as_uint(s) - base;
      for (; w < kWaves; w++) {
        const uint32_t r = apply(x.tot[p][w], at);
        if (uniform((int)(x.stop[p][w] || r >= kBinade))) break;
        at = r;
      }
      s = uniform(__uint_as_float(base + at));
    }
    if (w < kWaves) {
      const int p = pass & 1;
      pass++;
      if (wid == w) {
        const float t = wave_exact_seg<kScanPT>(s, v);
        if (lane == 0) x.s[p] = t;
      }
      __syncthreads();
      s = uniform(x.s[p]);
      w++;
    }
    fw = w;
  }
  return s;
}

// s0 + the gathered values of edges [e0, e0+ne) in edge order, rounded as the
// sequential FP32 loop starting from s0 (all threads return it).  `buf`: a
// 16-byte aligned LDS buffer of kScanChunk floats.  Chunk c is gathered as
// thread t's terms t + 256 j (coalesced index loads), stored at their
// position in the chunk, and scanned as thread t's terms 16t..16t+15; chunk
// c+1's gathers and chunk c+2's index loads are in flight meanwhile.  (Every
// scan has a barrier after all threads have read their terms, so one buffer
// serves every chunk.)
// STAGED: the row's values were gathered beforehand into a 16-byte aligned
// buffer (g.s, padded to a multiple of 4): each thread loads its terms from
// there, the next chunk's in flight, and no LDS is needed for them.
template <bool NT, class G, bool STAGED = false>
__device__ float exact_row_sum(const int32_t* __restrict__ col, int e_max, int e0, int ne,
                               const G& g, float s0, float* __restrict__ buf, ExactLds& x) {
  const int tid = threadIdx.x;
  const int nchunks = (ne + kScanChunk - 1) / kScanChunk;
  float s = s0;
  int pass = 0;
  if (nchunks == 0) return s;
  if constexpr (STAGED) {
    float4 nx[kScanPT / 4];
    auto load = [&](int c) {
      const int at = c * kScanChunk + tid * kScanPT;
#pragma unroll
      for (int k = 0; k < kScanPT / 4; k++)
        nx[k] = *reinterpret_cast<const float4*>(g.s + (at + 4 * k < ne ? at + 4 * k : 0));
    };
    load(0);
    for (int c = 0; c < nchunks; c++) {
      const int at = c * kScanChunk + tid * kScanPT;
      float v[kScanPT];
#pragma unroll
      for (int k = 0; k < kScanPT / 4; k++) {
        v[4 * k] = at + 4 * k < ne ? nx[k].x : 0.0f;
        v[4 * k + 1] = at + 4 * k + 1 < ne ? nx[k].y : 0.0f;
        v[4 * k + 2] = at + 4 * k + 2 < ne ? nx[k].z : 0.0f;
        v[4 * k + 3] = at + 4 * k + 3 < ne ? nx[k].w : 0.0f;
      }
      if (c + 1 < nchunks) load(c + 1);
      s = exact_scan_chunk(v, s, pass, x);
    }
    return s;
  } else {
    int idx[kScanPT];
    float vv[kScanPT];
    auto elem = [&](int c, int j) {  // edge offset in the row, clamped into it
      return min(c * kScanChunk + tid + j * kBlock, ne - 1);
    };
    auto load_idx = [&](int c) {
#pragma unroll
      for (int j = 0; j < kScanPT; j++)
        idx[j] = ld_stream<NT>(col + min(e0 + elem(c, j), e_max));
    };
    auto gather = [&](int c) {
#pragma unroll
      for (int j = 0; j < kScanPT; j++) vv[j] = g.value(e0 + elem(c, j), idx[j]);
    };
    load_idx(0);
    gather(0);
    if (nchunks > 1) load_idx(1);
    for (int c = 0; c < nchunks; c++) {
#pragma unroll
      for (int j = 0; j < kScanPT; j++)
        buf[tid + j * kBlock] = c * kScanChunk + tid + j * kBlock < ne ? vv[j] : 0.0f;
      if (c + 1 < nchunks) {
        gather(c + 1);                         // in flight during the scan of chunk c
        if (c + 2 < nchunks) load_idx(c + 2);  // likewise
      }
      __syncthreads();
      float v[kScanPT];
      const float4* v4 = reinterpret_cast<const float4*>(buf + tid * kScanPT);
#pragma unroll
      for (int k = 0; k < kScanPT / 4; k++) {
        const float4 t = v4[k];
        v[4 * k] = t.x;
        v[4 * k + 1] = t.y;
        v[4 * k + 2] = t.z;
        v[4 * k + 3] = t.w;
      }
      s = exact_scan_chunk(v, s, pass, x);
    }
    return s;
  }
}

// Loads the tile's edge indices col[e0 + tid + j*kBlock] (clamped into the
// tile so all IPT loads issue back to back).  Requires ne >= 1.
template <int IPT, bool NT, int NB = kBlock>
__device__ __forceinline__ void load_indices(const int32_t* __restrict__ col, int e0, int ne,
                                             int (&idx)[IPT]) {
  const int last = ne - 1;
#pragma unroll
  for (int j = 0; j < IPT; j++)
    idx[j] = ld_stream<NT>(col + e0 + min((int)threadIdx.x + j * NB, last));
}

// Tiles whose edges are stored sorted by source (SORTED) carry, per edge, its
// offset in the tile: pos[] (16 bits).  The gather functor always sees the
// edge's CSR index.
template <int IPT, bool NT, int NB = kBlock>
__device__ __forceinline__ void load_positions(const uint16_t* __restrict__ pos, int e0, int ne,
                                               int (&p)[IPT]) {
  const int last = ne - 1;
#pragma unroll
  for (int j = 0; j < IPT; j++)
    p[j] = (int)ld_stream<NT>(pos + e0 + min((int)threadIdx.x + j * NB, last));
}

// Gathers of the form factor(e) * raw(u) (G::kScaled): in a sorted tile the
// factors, stored in CSR order, are loaded in that order and applied once the
// gathered values are back at their CSR positions in LDS (scale_tile).
template <class G, class = void>
struct scaled_gather : std::false_type {};
template <class G>
struct scaled_gather<G, std::void_t<decltype(G::kScaled)>> : std::bool_constant<G::kScaled> {};

template <int IPT, bool SORTED, class G, int NB = kBlock>
__device__ __forceinline__ void gather_values(const G& g, int e0, int ne, const int (&idx)[IPT],
                                              const int (&p)[IPT], float (&v)[IPT]) {
  const int last = ne - 1;
#pragma unroll
  for (int j = 0; j < IPT; j++) {
    if constexpr (SORTED && scaled_gather<G>::value)
      v[j] = g.raw(idx[j]);
    else
      v[j] = g.value(e0 + (SORTED ? p[j] : min((int)threadIdx.x + j * NB, last)), idx[j]);
  }
}

// factor(e) of this thread's edges e0 + tid + j*NB (clamped), in CSR order.
template <int IPT, class G, int NB = kBlock>
__device__ __forceinline__ void load_factors(const G& g, int e0, int ne, float (&f)[IPT]) {
#pragma unroll
  for (int j = 0; j < IPT; j++) f[j] = g.factor(e0 + min((int)threadIdx.x + j * NB, ne - 1));
}

// val[i] *= factor of edge i, between two barriers.
template <int IPT, int NB = kBlock>
__device__ __forceinline__ void scale_tile(float* val, int ne, const float (&f)[IPT]) {
  __syncthreads();
#pragma unroll
  for (int j = 0; j < IPT; j++)
    if ((int)threadIdx.x + j * NB < ne) val[threadIdx.x + j * NB] *= f[j];
}

// Sum of the gathered values of a hub segment [e0, e0+ne), ne >= 1: per-thread
// partial in j order, wave butterfly, then waves in order.  Valid in thread 0.
// A sorted segment's values go back to their CSR positions through `val`
// (kBlock*IPT floats of LDS) first, so the sum is the same bits.
template <int IPT, bool NT, bool SORTED, class G>
__device__ __forceinline__ float segment_sum(const int32_t* __restrict__ col,
                                             const uint16_t* __restrict__ pos, int e0, int ne,
                                             const G& g, float* val) {
  int idx[IPT], p[IPT];
  float v[IPT];
  load_indices<IPT, NT>(col, e0, ne, idx);
  if constexpr (SORTED) load_positions<IPT, NT>(pos, e0, ne, p);
  gather_values<IPT, SORTED>(g, e0, ne, idx, p, v);
  if constexpr (SORTED) {
    float f[IPT];
    if constexpr (scaled_gather<G>::value) load_factors<IPT>(g, e0, ne, f);
#pragma unroll
    for (int j = 0; j < IPT; j++)
      if ((int)threadIdx.x + j * kBlock < ne) val[p[j]] = v[j];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < IPT; j++) {
      v[j] = val[min((int)threadIdx.x + j * kBlock, ne - 1)];
      if constexpr (scaled_gather<G>::value) v[j] *= f[j];
    }
    __syncthreads();  // val is reused by the block sum
  }
  float s = 0.0f;
#pragma unroll
  for (int j = 0; j < IPT; j++) s += ((int)threadIdx.x + j * kBlock < ne) ? v[j] : 0.0f;
  return block_sum<kWaves>(s, val);
}

// Where the epilogue's terms are never negative (E::kWaveRows), a tile whose
// longest row exceeds kWaveTile has its rows of more than kWaveRow edges added
// by a wavefront each (wave_exact_row), the shorter ones by their owner
// threads, side by side.  The wavefronts start when the longest of those chains
// (3 ns a term) has ended and cost about 2 us themselves, so a tile whose
// longest row is near kWaveRow is better off with the chain.  20 iterations,
// us, kWaveTile 512 / 1200 / 1536 / 2000: 5,000 vertices x 24 332 / 330 / 291 / 300,
// 9,001 x 32 340 / 337 / 298 / 307, 12,000 x 8 338 / 331 / 292 / 299, 12,000 x 32 328
// / 325 / 323 / 329.
constexpr int kWaveRow = 512;
constexpr int kWaveTile = 1536;
constexpr int kNoWaveRows = 0x7fffffff;

template <class E, class = void>
struct wave_rows : std::false_type {};
template <class E>
struct wave_rows<E, std::void_t<decltype(E::kWaveRows)>> : std::bool_constant<E::kWaveRows> {};

// from[t] = kWaveRow where tile t has wavefront rows, else kNoWaveRows; one
// wavefront per tile.
[[maybe_unused]] static __global__ __launch_bounds__(kBlock) void wave_rows_kernel(
    const Tile* __restrict__ tiles, int n, const int32_t* __restrict__ off,
    int32_t* __restrict__ from) {
  const int t = blockIdx.x * kWaves + threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
  if (t >= n) return;
  const Tile tile = tiles[t];
  int longest = 0;
  for (int r = tile.x + lane; r < tile.y; r += kWave) longest = max(longest, off[r + 1] - off[r]);
  const bool any = __ballot(longest > kWaveTile) != 0;
  if (lane == 0) from[t] = any ? kWaveRow : kNoWaveRows;
}

// LDS of one row tile of a workgroup of NB threads.
template <int IPT, int NB = kBlock>
struct RowTileLds {
  alignas(16) float val[NB * IPT + 4];       // gathered per-edge values, a spare place
  int off[kRowsPerThread * NB + 1];          // row offsets, rebased to the tile on use
  float longsum[kRowsPerThread * NB];        // sums of the rows that wavefronts add
  // rows of more than kWaveRow edges, added by a wavefront each (wave_rows epilogues)
  int n_long;
  int16_t long_row[NB * IPT / kWaveRow];
};

// Registers holding the loads of one tile that do not depend on a gather:
// its edge indices, and for a row tile its row offsets and each owned row's
// epilogue operands.  Issued as early as possible (see pr_pull_persistent).
template <int IPT, class Pre, int NB = kBlock>
struct TileRegs {
  int idx[IPT];
  int pos[IPT];  // sorted tiles only
  int offv[kOffLoads];
  Pre pre[kRowsPerThread];
};

// Phase A: issue every gather-independent load of tile t, without branches
// (a branch here would make the compiler's wait counting conservative and
// serialize the prefetch with the gathers).  Addresses of idle lanes are
// clamped: an empty tile re-reads its first edge, a hub segment reads the
// offsets and operands of its own row.
// `e_max` is the last valid index of `col` (the arrays hold >= 1 element).
template <int IPT, bool NT, bool SORTED, class E, int NB = kBlock>
__device__ __forceinline__ void issue_tile_loads(const Tile& t, const int32_t* __restrict__ off,
                                                 const int32_t* __restrict__ col,
                                                 const uint16_t* __restrict__ pos, int e_max,
                                                 const E& e, TileRegs<IPT, typename E::Pre, NB>& R) {
  const int tid = threadIdx.x;
  const int last = max(t.w - t.z - 1, 0);
#pragma unroll
  for (int j = 0; j < IPT; j++)
    R.idx[j] = ld_stream<NT>(col + min(t.z + min(tid + j * NB, last), e_max));
  if constexpr (SORTED) {
#pragma unroll
    for (int j = 0; j < IPT; j++)
      R.pos[j] = (int)ld_stream<NT>(pos + min(t.z + min(tid + j * NB, last), e_max));
  }
  const int nr = (t.y >= 0) ? t.y - t.x : 1;
#pragma unroll
  for (int q = 0; q < kOffLoads; q++)
    R.offv[q] = ld_stream<NT>(off + t.x + min(tid + q * NB, nr));
#pragma unroll
  for (int q = 0; q < kRowsPerThread; q++) R.pre[q] = e.pre(t.x + min(tid + q * NB, nr - 1));
}

// Phases C-E of a row tile whose gathered values are already in lds.val and
// rebased offsets in lds.off (after a barrier): reduce rows, epilogue.
// SEQ_ALL: every row, whatever its length, is summed by its owner thread in
// CSR order (no wavefront tree): bit-identical sums for any row the tile holds.
template <int IPT, class E, bool SEQ_ALL = false, int NB = kBlock>
__device__ __forceinline__ double reduce_row_tile(int r0, int nr, const E& e,
                                                  const typename E::Pre (&pre)[kRowsPerThread],
                                                  RowTileLds<IPT, NB>& lds,
                                                  int wave_from = kNoWaveRows) {
  const int tid = threadIdx.x;
  float sum[kRowsPerThread];
  bool have_long = false;
  constexpr bool kWaves1 = SEQ_ALL && wave_rows<E>::value;
#pragma unroll
  for (int q = 0; q < kRowsPerThread; q++) {
    const int i = tid + q * NB;
    sum[q] = e.init(pre[q]);
    if (i < nr) {
      const int b = lds.off[i], en = lds.off[i + 1];
      if (kWaves1 && en - b > wave_from) {
        lds.long_row[atomicAdd(&lds.n_long, 1)] = (int16_t)i;
        lds.longsum[i] = sum[q];
      } else if (SEQ_ALL || en - b <= kSeqRow)
        sum[q] = wave_rows<E>::value ? seq_sum(sum[q], lds.val, b, en)
                                     : seq_sum_wide(sum[q], lds.val, b, en);
      else
        have_long = true;
    }
  }
  if constexpr (kWaves1) {
    if (wave_from < kNoWaveRows) {
      __syncthreads();
      const int n = lds.n_long;
      for (int k = uniform((int)(tid / kWave)); k < n; k += NB / kWave) {
        const int row = uniform((int)lds.long_row[k]);
        const float s = wave_exact_row(uniform(lds.longsum[row]), lds.val, uniform(lds.off[row]),
                                       uniform(lds.off[row + 1]));
        if ((tid & (kWave - 1)) == 0) lds.longsum[row] = s;
      }
      __syncthreads();
#pragma unroll
      for (int q = 0; q < kRowsPerThread; q++) {
        const int i = tid + q * NB;
        if (i < nr && lds.off[i + 1] - lds.off[i] > wave_from) sum[q] = lds.longsum[i];
      }
    }
  }
  if (!SEQ_ALL && __syncthreads_or(have_long)) {
    const int lane = tid & (kWave - 1), wid = tid / kWave;
    for (int c = wid * kWave; c < nr; c += NB) {
      const int i = c + lane;
      const bool lr = (i < nr) && (lds.off[i + 1] - lds.off[i] > kSeqRow);
      uint64_t mask = __ballot(lr);
      while (mask) {
        const int row = c + __builtin_ctzll(mask);
        mask &= mask - 1;
        const int b = lds.off[row], en = lds.off[row + 1];
        float s = 0.0f;
        int k = b + lane;
        for (; k + 3 * kWave < en; k += 4 * kWave) {
          const float a0 = lds.val[k], a1 = lds.val[k + kWave], a2 = lds.val[k + 2 * kWave],
                      a3 = lds.val[k + 3 * kWave];
          s += a0;
          s += a1;
          s += a2;
          s += a3;
        }
        for (; k < en; k += kWave) s += lds.val[k];
        s = wave_sum(s);
        if (lane == 0) lds.longsum[row] = s;
      }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kRowsPerThread; q++) {
      const int i = tid + q * NB;
      if (i < nr && lds.off[i + 1] - lds.off[i] > kSeqRow) sum[q] += lds.longsum[i];
    }
  }
  double acc = 0.0;
#pragma unroll
  for (int q = 0; q < kRowsPerThread; q++) {
    const int i = tid + q * NB;
    if (i < nr) acc += e.finish(r0 + i, sum[q], pre[q]);
  }
  return acc;
}

// Stage a row tile's gathered values and rebased offsets into LDS.
template <int IPT, bool SORTED, class Pre, int NB = kBlock>
__device__ __forceinline__ void stage_row_tile(const Tile& t, const TileRegs<IPT, Pre, NB>& R,
                                               const float (&v)[IPT], RowTileLds<IPT, NB>& lds) {
  const int tid = threadIdx.x;
  const int ne = t.w - t.z;
  if (tid == 0) lds.n_long = 0;
  // No branch per store: each was two jumps of instruction fetches (RMAT-16 10
  // percent of its time).  Offsets past the tile's rows are off[nr] (clamped
  // loads), values past its edges go to a spare place.
#pragma unroll
  for (int q = 0; q < kOffLoads; q++)
    lds.off[min(tid + q * NB, kRowsPerThread * NB)] = R.offv[q] - t.z;
#pragma unroll
  for (int j = 0; j < IPT; j++) {
    const int at = tid + j * NB;
    lds.val[at < ne ? (SORTED ? R.pos[j] : at) : NB * IPT] = v[j];
  }
}

// One row tile: rows [r0, r1) whose edges are [e0, e0+ne).  The epilogue E
// provides
//   typename E::Pre          per-row operands, loaded before the gather
//   Pre pre(int row)         (clamped row: always a valid index)
//   float init(const Pre&)   value the row sum starts from
//   double finish(int row, float sum, const Pre&)   writes the row, returns
//                            its contribution to the tile's double accumulator
template <int IPT, bool NT, bool SORTED, class G, class E, bool SEQ_ALL = false,
          int NB = kBlock>
__device__ __forceinline__ double row_tile(const int32_t* __restrict__ off,
                                           const int32_t* __restrict__ col,
                                           const uint16_t* __restrict__ pos, int e_max, int r0,
                                           int r1, int e0, int ne, const G& g, const E& e,
                                           RowTileLds<IPT, NB>& lds,
                                           int wave_from = kNoWaveRows) {
  const Tile t{r0, r1, e0, e0 + ne};
  TileRegs<IPT, typename E::Pre, NB> R;
  issue_tile_loads<IPT, NT, SORTED, E, NB>(t, off, col, pos, e_max, e, R);
  float v[IPT] = {};
  if (ne > 0) gather_values<IPT, SORTED, G, NB>(g, e0, ne, R.idx, R.pos, v);
  if constexpr (SORTED && scaled_gather<G>::value) {
    float f[IPT];
    if (ne > 0) load_factors<IPT, G, NB>(g, e0, ne, f);
    stage_row_tile<IPT, SORTED, typename E::Pre, NB>(t, R, v, lds);
    scale_tile<IPT, NB>(lds.val, ne, f);
  } else {
    stage_row_tile<IPT, SORTED, typename E::Pre, NB>(t, R, v, lds);
  }
  __syncthreads();
  return reduce_row_tile<IPT, E, SEQ_ALL, NB>(r0, r1 - r0, e, R.pre, lds, wave_from);
}

// ---------------------------------------------------------------------------
// Long rows summed in edge order by one lane.
//
// The reference adds a row's terms one after the other in FP32
// (src/pr/omp_base.cc:34-37, src/spmv/omp_base.cc:21-26); for a row longer
// than a tile the fastest way to the same bits is that dependent chain
// itself, on one lane, with the rest of the workgroup keeping it fed
// (hub_chain_sum).  Measured on the MI355X the chain costs 2.8-3.4 ns per
// term (a dependent v_add_f32 every ~4.8 cycles when the terms sit in
// registers; the LDS reads feeding it take the rest), independent of the
// terms' signs, ties or magnitudes.

// s0 + the gathered values of edges [e0, e0+ne) in edge order, rounded as the
// sequential FP32 loop, with the workgroup split by role: lane 0 of wave 0
// adds chunk c (kHubChunk entries, LDS) while waves 1..3 gather chunk c+1
// into the other buffer (their column loads of chunk c+2 already in flight),
// so no gather waits on the chain and the chain wave issues nothing else.
// SORTED: each chunk is stored sorted by source and pos[e] is the edge's
// offset within its chunk; values go back to edge order in LDS.  Buffers:
// two 16-byte aligned arrays of kHubChunk floats, one float for the sum.
// All threads return the sum.
template <int kQ, bool SORTED, class G>
__device__ float hub_chain_sum(const int32_t* __restrict__ col, const uint16_t* __restrict__ pos,
                               int e_max, int e0, int ne, const G& g, float s0,
                               float* __restrict__ buf0, float* __restrict__ buf1,
                               float* __restrict__ s_out) {
  constexpr int kProd = kBlock - kWave;  // gathering lanes
  constexpr int PPT = kHubChunk / kProd;
  static_assert(PPT * kProd == kHubChunk && kHubChunk % (4 * kQ) == 0, "hub chunk shape");
  const int tid = threadIdx.x;
  const bool chain_wave = tid < kWave;
  const int pt = tid - kWave;
  const int nchunks = (ne + kHubChunk - 1) / kHubChunk;
  int idx[PPT], p[PPT];
  auto slot = [&](int c, int j) {  // clamped into the chunk
    return min(pt + j * kProd, min(kHubChunk, ne - c * kHubChunk) - 1);
  };
  auto load_idx = [&](int c) {
#pragma unroll
    for (int j = 0; j < PPT; j++) idx[j] = col[min(e0 + c * kHubChunk + slot(c, j), e_max)];
    if constexpr (SORTED) {
#pragma unroll
      for (int j = 0; j < PPT; j++) p[j] = (int)pos[min(e0 + c * kHubChunk + slot(c, j), e_max)];
    }
  };
  auto produce = [&](int c, float* buf) {  // gathers chunk c (indices loaded), stores it
    const int nc = min(kHubChunk, ne - c * kHubChunk);
    float v[PPT];
    int o[PPT];
#pragma unroll
    for (int j = 0; j < PPT; j++) {
      o[j] = SORTED ? p[j] : slot(c, j);
      v[j] = g.value(e0 + c * kHubChunk + o[j], idx[j]);
    }
#pragma unroll
    for (int j = 0; j < PPT; j++)
      if (pt + j * kProd < nc) buf[o[j]] = v[j];
  };
  if (chain_wave) __builtin_amdgcn_s_setprio(3);
  if (!chain_wave && nchunks > 0) {
    load_idx(0);
    produce(0, buf0);
    if (nchunks > 1) load_idx(1);
  }
  __syncthreads();
  float s = s0;
  for (int c = 0; c < nchunks; c++) {
    float* cur = (c & 1) ? buf1 : buf0;
    float* nxt = (c & 1) ? buf0 : buf1;
    if (chain_wave) {
      if (tid == 0) s = lane_seq_sum<kQ>(s, cur, min(kHubChunk, ne - c * kHubChunk));
    } else if (c + 1 < nchunks) {
      produce(c + 1, nxt);
      if (c + 2 < nchunks) load_idx(c + 2);  // in flight across the barrier
    }
    __syncthreads();
  }
  if (chain_wave) __builtin_amdgcn_s_setprio(0);
  if (tid == 0) *s_out = s;
  __syncthreads();
  return *s_out;
}

}  // namespace gd

#endif  // GD_PULL_ENGINE_H_
