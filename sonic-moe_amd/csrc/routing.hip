// Routing kernels for gfx950: fused top-K + softmax, expert histogram / prefix sum, stable counting-sort routing
// metadata, router backward.  All integer outputs are deterministic (no order-dependent atomics reach an output).
#include <hip/hip_fp16.h>

#include <mutex>

#include "routing_common.h"

namespace smoe {

// ============================================================================================================
// top-K + softmax
// ============================================================================================================
// One row is owned by a group of G consecutive lanes (G a power of two <= 64); lane g of the group holds the
// VPL consecutive columns [g*VPL, (g+1)*VPL) as keys
//     key = (order-preserving image of the value's bits) << W | (2^W - 1 - column)
// with W = 32 for fp32 (two words) and W = 16 for the 16-bit types, so that the maximum key is the largest value and, among
// equal values, the lowest column.  K rounds of "group arg-max, then retire the winner" give the winners in descending order.
// A round is a chain of maxima, and the winners' exponentials are taken behind the rounds (bf16, one row, E = 128, K = 8:
// 3.8 us; 40960 rows, E = 256: 18; fp32 5.2 and 29).

template <typename T, int VPL>
__global__ __launch_bounds__(256) void topk_softmax_kernel(const T* __restrict__ logits, int64_t row_stride,
                                                           int64_t Trows, int E, int K, int G, uint32_t clear_mask,
                                                           float* __restrict__ scores, int32_t* __restrict__ indices,
                                                           int do_softmax) {
  const int lane_in_block = threadIdx.x;
  const int rows_per_block = 256 / G;
  const int g = lane_in_block % G;
  const int64_t row = (int64_t)blockIdx.x * rows_per_block + lane_in_block / G;
  const bool row_ok = row < Trows;
  const int64_t rrow = row_ok ? row : 0;

  typedef TopkKey<T> TK;
  typedef typename TK::Key Key;
  Key key[VPL];
  const T* src = logits + rrow * row_stride;
  // all loads of a lane at once, those past the end from the last column (taken under a condition each, they were VPL
  // round trips to memory: one row, E = 128, K = 8 10.7 -> 8.3 us)
  uint32_t bits[VPL];
#pragma unroll
  for (int i = 0; i < VPL; i++) {
    const int col = g * VPL + i;
    bits[i] = TK::load(src + (col < E ? col : E - 1), clear_mask);
  }
#pragma unroll
  for (int i = 0; i < VPL; i++) {
    const int col = g * VPL + i;
    // 0 = retired / out of range: below every real key (real keys have a non-zero column part)
    const uint32_t v = opaque(bits[i]);
    key[i] = col < E ? TK::make(v, col) : TK::none();
  }

  pick_winners<TK>(key, G, g, lane_in_block & 63, row_ok, K, do_softmax != 0, scores + rrow * K, indices + rrow * K, nullptr);
}

template <typename T>
static int launch_topk(const void* logits, int64_t T_, int E, int K, int64_t row_stride, float* scores,
                       int32_t* indices, int softmax, uint32_t clear_mask, hipStream_t st) {
  // Columns per lane.  With few a round is a short chain and many lanes run; with many it takes fewer instructions in all,
  // which counts once the chip is full.  us, 4 / 8 / 16 columns: bf16 E = 128, K = 8 8192 rows 5.0/5.3/6.2, 16384 7.0/6.7/8.2,
  // 40960 13.0/11.2/14.1; E = 100, K = 5 8192 4.9/5.1/4.7, 40960 11.4/9.7/8.4; E = 256, K = 16 4096 7.3/7.1/8.1, 40960
  // 38/27/27.  fp32, whose keys are two words, E = 128, K = 8 8192 7.7/7.8/9.1, 16384 11.1/10.5/11.3, 40960 22/19/18;
  // E = 256, K = 16 4096 13/12/14, 40960 74/53/45.
  const int64_t logits_count = T_ * E;
  const int cols = logits_count <= 1 << 20 ? 4 : sizeof(T) == 2 || logits_count <= 1 << 21 ? 8 : 16;
  int G = 1;
  while (G < 64 && G * cols < E) G <<= 1;
  int vpl = 1;
  while (vpl * G < E) vpl <<= 1;
  const int rows_per_block = 256 / G;
  const dim3 grid((unsigned)ceil_div(T_, rows_per_block)), block(256);
  const T* p = (const T*)logits;
#define SMOE_TOPK_CASE(V)                                                                                          \
  case V:                                                                                                          \
    hipLaunchKernelGGL((topk_softmax_kernel<T, V>), grid, block, 0, st, p, row_stride, T_, E, K, G, clear_mask,    \
                       scores, indices, softmax);                                                                  \
    break;
  switch (vpl) {
    SMOE_TOPK_CASE(1)
    SMOE_TOPK_CASE(2)
    SMOE_TOPK_CASE(4)
    SMOE_TOPK_CASE(8)
    SMOE_TOPK_CASE(16)
    SMOE_TOPK_CASE(32)
    SMOE_TOPK_CASE(64)
    default:
      set_error("topk: unsupported E=%d", E);
      return SMOE_ERR_UNSUPPORTED;
  }
#undef SMOE_TOPK_CASE
  SMOE_LAUNCH_CHECK();
  return SMOE_OK;
}

// ============================================================================================================
// router backward
// ============================================================================================================
template <typename T>
SMOE_DEV void store_from_f32(T* p, float v);
template <>
__device__ __forceinline__ void store_from_f32<uint16_t>(uint16_t* p, float v) {
  *p = (uint16_t)f32_to_bf16_bits(v);
}
template <>
__device__ __forceinline__ void store_from_f32<__half>(__half* p, float v) {
  *p = __float2half(v);
}
template <>
__device__ __forceinline__ void store_from_f32<float>(float* p, float v) {
  *p = v;
}

template <typename T>
__global__ __launch_bounds__(256) void softmax_topk_bwd_kernel(T* __restrict__ dlogits, int64_t row_stride,
                                                               const T* dlogits_add, const float* __restrict__ dscores,
                                                               const float* __restrict__ scores,
                                                               const int32_t* __restrict__ indices, int64_t Trows,
                                                               int K) {
  const int64_t row = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (row >= Trows) return;
  const float* g = dscores + row * K;
  const float* s = scores + row * K;
  const int32_t* ix = indices + row * K;
  float dot = 0.f;
  for (int k = 0; k < K; k++) dot += g[k] * s[k];
  T* out = dlogits + row * row_stride;
  // dlogits_add (may be dlogits itself): a gradient that reached the selected logits some other way is added in
  const T* add = dlogits_add ? dlogits_add + row * row_stride : nullptr;
  for (int k = 0; k < K; k++) {
    float v = s[k] * (g[k] - dot);
    if (add) v += __uint_as_float(load_as_f32_bits<T>(add + ix[k]));
    store_from_f32<T>(out + ix[k], v);
  }
}

// The whole gradient of the router logits: the scatter above onto whatever gradient reached the logits from outside (the
// load-balancing loss), or onto zeros, in one pass that writes every row.  As a zero fill, the scatter and an add it was
// three launches and five passes over (T, E); T = 6001, E = 128, K = 8: 11.2 -> 4.0 us, T = 40960: 17.5 -> 10.0.
// A thread owns VEC columns of a row and looks for the row's K winners among them.  WIDE: they are one aligned piece of 16
// bytes.  Otherwise they are read and written one by one and lie `pieces` apart, so that neighbouring lanes have
// neighbouring columns; still VEC to a thread, because the search costs the same for one column as for eight (E = 100,
// K = 5, T = 40960, bf16: three launches 12.8 us, one column to a thread 32, eight adjacent ones 15.2, eight apart 12.6).
// outside may be dlogits itself, with the same stride: a thread reads its columns before it writes them (and what it reads of
// another's, past the end of a row, it does not use).
template <typename T, int VEC, bool WIDE>
__global__ __launch_bounds__(256) void router_logit_grad_kernel(T* dlogits, int64_t row_stride,
                                                                const T* outside, int64_t outside_stride,
                                                                const float* __restrict__ dscores,
                                                                const float* __restrict__ scores,
                                                                const int32_t* __restrict__ indices, int64_t Trows, int E,
                                                                int K, int pieces, int rows_per_block) {
  struct alignas(sizeof(T) * VEC) Pack {
    T e[VEC];
  };
  const int64_t row = (int64_t)blockIdx.x * rows_per_block + threadIdx.x / pieces;
  if ((int)threadIdx.x / pieces >= rows_per_block || row >= Trows) return;
  const float* g = dscores + row * K;
  const float* s = scores + row * K;
  const int32_t* ix = indices + row * K;
  float dot = 0.f;
  for (int k = 0; k < K; k++) dot += g[k] * s[k];
  constexpr int FIRST = WIDE ? VEC : 1;
  const int gap = WIDE ? 1 : pieces;  // from one of a thread's columns to the next
  for (int c0 = (int)threadIdx.x % pieces * FIRST; c0 < E; c0 += pieces * VEC) {
    float v[VEC];
    Pack p;
    if (outside != nullptr) {
      const T* src = outside + row * outside_stride;
      if constexpr (WIDE) {
        p = *(const Pack*)(src + c0);
      } else {
#pragma unroll
        for (int j = 0; j < VEC; j++) p.e[j] = src[c0 + j * gap < E ? c0 + j * gap : E - 1];
      }
    }
#pragma unroll
    for (int j = 0; j < VEC; j++) v[j] = outside != nullptr ? __uint_as_float(load_as_f32_bits<T>(&p.e[j])) : 0.f;
    for (int k = 0; k < K; k++) {
      const int c = ix[k] - c0;
      const float add = s[k] * (g[k] - dot);
#pragma unroll
      for (int j = 0; j < VEC; j++) v[j] = c == j * gap ? v[j] + add : v[j];
    }
#pragma unroll
    for (int j = 0; j < VEC; j++) store_from_f32<T>(&p.e[j], v[j]);
    T* dst = dlogits + row * row_stride + c0;
    if constexpr (WIDE) {
      *(Pack*)dst = p;
    } else {
#pragma unroll
      for (int j = 0; j < VEC; j++)
        if (c0 + j * gap < E) dst[j * gap] = p.e[j];
    }
  }
}

template <typename T>
static void launch_router_logit_grad(void* dlogits, int64_t row_stride, const void* outside, int64_t outside_stride,
                                     const float* dscores, const float* scores, const int32_t* indices, int64_t T_, int E,
                                     int K, hipStream_t st) {
  constexpr int VEC = 16 / sizeof(T);
  const bool wide = E % VEC == 0 && row_stride % VEC == 0 && aligned16(dlogits) &&
                    (outside == nullptr || (outside_stride % VEC == 0 && aligned16(outside)));
  const int pieces = (int)ceil_div(E, VEC);
  const int columns = pieces < 256 ? pieces : 256;  // threads of a row
  const int rows_per_block = 256 / columns;
  const dim3 grid((unsigned)ceil_div(T_, rows_per_block)), block(256);
  if (wide)
    hipLaunchKernelGGL((router_logit_grad_kernel<T, VEC, true>), grid, block, 0, st, (T*)dlogits, row_stride,
                       (const T*)outside, outside_stride, dscores, scores, indices, T_, E, K, columns, rows_per_block);
  else
    hipLaunchKernelGGL((router_logit_grad_kernel<T, VEC, false>), grid, block, 0, st, (T*)dlogits, row_stride,
                       (const T*)outside, outside_stride, dscores, scores, indices, T_, E, K, columns, rows_per_block);
}

// Backward of the un-fused top-K (values without softmax): the gradient of a selected logit is the gradient of its
// value.  One thread per token; the caller has zero-filled dlogits.
template <typename T>
__global__ __launch_bounds__(256) void topk_bwd_kernel(T* __restrict__ dlogits, int64_t row_stride,
                                                       const float* __restrict__ dvalues,
                                                       const int32_t* __restrict__ indices, int64_t Trows, int K) {
  const int64_t row = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (row >= Trows) return;
  T* out = dlogits + row * row_stride;
  for (int k = 0; k < K; k++) store_from_f32<T>(out + indices[row * K + k], dvalues[row * K + k]);
}

// ============================================================================================================
// count + inclusive cumsum (standalone operator)
// ============================================================================================================
__global__ void fill_i32_kernel(int32_t* p, int64_t n, int32_t v) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

template <typename IdxT, bool USE_LDS>
__global__ __launch_bounds__(1024) void count_kernel(const IdxT* __restrict__ x, int64_t n, int E,
                                                     int32_t* __restrict__ count) {
  extern __shared__ int32_t hist[];
  if (USE_LDS) {
    for (int e = threadIdx.x; e < E; e += blockDim.x) hist[e] = 0;
    __syncthreads();
  }
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const int64_t v = (int64_t)x[i];
    if (v >= 0 && v < E) {
      if (USE_LDS)
        atomicAdd(&hist[v], 1);
      else
        atomicAdd(&count[v], 1);
    }
  }
  if (USE_LDS) {
    __syncthreads();
    for (int e = threadIdx.x; e < E; e += blockDim.x) {
      const int32_t c = hist[e];
      if (c) atomicAdd(&count[e], c);
    }
  }
}

// single block, 1024 threads: inclusive scan of count[0..E)
__global__ __launch_bounds__(1024) void inclusive_scan_kernel(const int32_t* __restrict__ count, int E,
                                                              int32_t* __restrict__ cumsum) {
  __shared__ int32_t wave_tot[16];
  const int per = (E + 1023) / 1024;
  const int lo = threadIdx.x * per;
  int32_t local = 0;
  for (int i = 0; i < per; i++)
    if (lo + i < E) local += count[lo + i];
  // inclusive scan of `local` across the block
  int32_t v = local;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int d = 1; d < 64; d <<= 1) {
    int32_t o = __shfl_up(v, d, 64);
    if (lane >= d) v += o;
  }
  if (lane == 63) wave_tot[wave] = v;
  __syncthreads();
  int32_t base = 0;
  for (int w = 0; w < wave; w++) base += wave_tot[w];
  int32_t run = base + v - local;  // exclusive prefix of this thread's chunk
  for (int i = 0; i < per; i++)
    if (lo + i < E) {
      run += count[lo + i];
      cumsum[lo + i] = run;
    }
}

// ============================================================================================================
// routing metadata: stable counting sort of TK expert ids
// ============================================================================================================
// A "segment" is SEG consecutive flat slots, owned by ONE workgroup, whose wavefronts own consecutive quarters of it, so
// that the order inside a segment is the wavefront / lane / iteration order.  Pass A: per-segment histogram ->
// hist_t[e][s].  Pass B: one wavefront per expert scans its row of hist_t -> base_t[e][s] (slots of expert e that precede
// segment s) and freq[e].  Pass C: every segment rebuilds off[] from freq, seeds a cursor per wavefront and expert and
// assigns positions with ballot-based ranking.
// All three wait for memory and for chains of dependent instructions, so the ranking is spread over four wavefronts (four
// steps of 64 slots each instead of sixteen in a row) and takes a slot's token by ONE 32-bit division (two 64-bit ones
// were half of its instructions).  The three passes, us, one wavefront per segment -> four: 16384 slots, E = 128 22.7 -> 10.9;
// 48008 23.1 -> 11.4; 327680 26.2 -> 16.5; 10000 slots, E = 4096 77 -> 28.
constexpr int SEG = 1024;
constexpr int META_WAVES = 4;
constexpr int SEG_STEPS = SEG / 64 / META_WAVES;  // steps of one wavefront

// The expert ids of a wavefront's quarter of a segment, -1 past the end: all loads before the first use (taken one step at
// a time, and under a condition each, every step of the histogram and of the ranking began with a round trip to memory).
SMOE_DEV void load_segment(const int32_t* __restrict__ expert_idx, int lo, int TK, int lane, int (&ids)[SEG_STEPS]) {
#pragma unroll
  for (int i = 0; i < SEG_STEPS; i++) {
    const uint32_t j = (uint32_t)lo + i * 64 + lane;
    ids[i] = TK > 0 ? expert_idx[j < (uint32_t)TK ? j : TK - 1] : -1;
  }
#pragma unroll
  for (int i = 0; i < SEG_STEPS; i++) ids[i] = (uint32_t)lo + i * 64 + lane < (uint32_t)TK ? (int)opaque(ids[i]) : -1;
}

__global__ __launch_bounds__(64 * META_WAVES) void meta_hist_kernel(const int32_t* __restrict__ expert_idx, int TK, int E,
                                                                    int NS, int32_t* __restrict__ hist_t) {
  extern __shared__ int32_t hist[];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int s = blockIdx.x;
  int ids[SEG_STEPS];
  load_segment(expert_idx, s * SEG + wave * (SEG / META_WAVES), TK, lane, ids);
  for (int e = tid; e < E; e += 64 * META_WAVES) hist[e] = 0;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < SEG_STEPS; i++)
    if (ids[i] >= 0 && ids[i] < E) atomicAdd(&hist[ids[i]], 1);
  __syncthreads();
  for (int e = tid; e < E; e += 64 * META_WAVES) hist_t[(size_t)e * NS + s] = hist[e];
}

__global__ __launch_bounds__(256) void meta_scan_kernel(const int32_t* __restrict__ hist_t, int E, int NS,
                                                        int32_t* __restrict__ base_t, int32_t* __restrict__ freq) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int e = blockIdx.x * 4 + wave;
  if (e >= E) return;
  int32_t carry = 0;
  for (int s0 = 0; s0 < NS; s0 += 64) {
    const int s = s0 + lane;
    const int32_t h = s < NS ? hist_t[(size_t)e * NS + s] : 0;
    int32_t v = h;
    for (int d = 1; d < 64; d <<= 1) {
      int32_t o = __shfl_up(v, d, 64);
      if (lane >= d) v += o;
    }
    if (s < NS) base_t[(size_t)e * NS + s] = carry + v - h;
    carry += __shfl(v, 63, 64);
  }
  if (lane == 0) freq[e] = carry;
}

__global__ __launch_bounds__(64 * META_WAVES) void meta_scatter_kernel(
    const int32_t* __restrict__ expert_idx, const int32_t* __restrict__ token_idx, int TK, int64_t T, int E,
    int K, int NS, int ebits, const int32_t* __restrict__ freq, const int32_t* __restrict__ base_t,
    int32_t* __restrict__ off, int32_t* __restrict__ gidx, int32_t* __restrict__ sidx, int32_t* __restrict__ ridx,
    int32_t* __restrict__ tok_off, const TileMapPair maps) {
  extern __shared__ int32_t lds[];  // META_WAVES x E, then a word per wavefront
  if ((int)blockIdx.x >= NS) {  // behind the segments: the tile maps, where the caller wants them
    const int which = blockIdx.x - NS;
    write_tile_map<META_WAVES, true>(freq, nullptr, nullptr, E, tile_map_rows(which), maps.gmax, maps.snake,
                                     which == 0 ? maps.map[0] : maps.map[1], lds);
    return;
  }
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  int32_t* cursor = lds + (size_t)wave * E;
  int32_t* wave_total = lds + (size_t)META_WAVES * E;
  const int s = blockIdx.x;
  const int lo = s * SEG + wave * (SEG / META_WAVES);
  int ids[SEG_STEPS];
  load_segment(expert_idx, lo, TK, lane, ids);
  for (int e = lane; e < E; e += 64) cursor[e] = 0;
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int i = 0; i < SEG_STEPS; i++)
    if (ids[i] >= 0 && ids[i] < E) atomicAdd(&cursor[ids[i]], 1);

  // exclusive scan of freq -> off (every segment needs it; segment 0 also publishes it), 256 experts at a time; thread e
  // turns the wavefronts' counts of expert e into their cursors
  int32_t carry = 0;
  for (int e0 = 0; e0 < E; e0 += 64 * META_WAVES) {
    const int e = e0 + tid;
    const int32_t f = e < E ? freq[e] : 0;
    const int32_t base = e < E ? base_t[(size_t)e * NS + s] : 0;
    int32_t v = f;
    for (int d = 1; d < 64; d <<= 1) {
      int32_t o = __shfl_up(v, d, 64);
      if (lane >= d) v += o;
    }
    if (lane == 63) wave_total[wave] = v;
    __syncthreads();  // (the first one also: every wavefront's counts are there)
    int32_t excl = carry + v - f;
#pragma unroll
    for (int w = 0; w < META_WAVES; w++) {
      if (w < wave) excl += wave_total[w];
      carry += wave_total[w];
    }
    if (e < E) {
      int32_t at = excl + base;
#pragma unroll
      for (int w = 0; w < META_WAVES; w++) {
        const int32_t n = lds[(size_t)w * E + e];
        lds[(size_t)w * E + e] = at;
        at += n;
      }
      if (s == 0) off[e] = excl;
    }
    __syncthreads();
  }
  if (s == 0 && tid == 0) off[E] = carry;

#pragma unroll
  for (int i = 0; i < SEG_STEPS; i++) {
    const uint32_t j0 = (uint32_t)lo + i * 64;
    if (j0 < (uint32_t)TK)
      place_slots(ids[i], (int)(j0 + lane), j0 + lane < (uint32_t)TK, lane, token_idx, TK, T, E, K, ebits, cursor, gidx,
                  sidx, ridx, tok_off);
  }
  if (tok_off && TK == 0 && s == 0)
    for (int64_t u = tid; u <= T; u += 64 * META_WAVES) tok_off[u] = 0;
}

// The three passes as one workgroup, for few slots: what they cost there is launches and one round trip to memory after
// the other.  Wavefront w owns M1_STEPS * 64 consecutive slots at most, whose expert ids it reads once, all at the start;
// histograms, scan and cursors stay in LDS.  The line at M1_SLOTS: one compute unit ranks 64 slots of each of its 16
// wavefronts in about a microsecond, the three launches and their dependent reads take 10 to 11 us: one workgroup takes 4.7
// for 512 slots, 7.6 for 3108 (E = 48), 13.5 for 8192.
constexpr int M1_WAVES = 16, M1_STEPS = 4, M1_SLOTS = M1_WAVES * M1_STEPS * 64, M1_MAX_E = 512;

__global__ __launch_bounds__(64 * M1_WAVES) void meta_one_kernel(
    const int32_t* __restrict__ expert_idx, const int32_t* __restrict__ token_idx, int TK, int64_t T, int E, int K,
    int ebits, int steps, int32_t* __restrict__ freq, int32_t* __restrict__ off, int32_t* __restrict__ gidx,
    int32_t* __restrict__ sidx, int32_t* __restrict__ ridx, int32_t* __restrict__ tok_off, const TileMapPair maps) {
  extern __shared__ int32_t lds[];  // M1_WAVES x E
  __shared__ int32_t map_part[2][2 * M1_WAVES];
  __shared__ int32_t wave_total[M1_WAVES];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int32_t* cursor = lds + wave * E;
  const int first = wave * steps * 64 + lane;
  int ids[M1_STEPS];
#pragma unroll
  for (int i = 0; i < M1_STEPS; i++) {
    const int j = first + i * 64;
    ids[i] = i < steps && TK > 0 ? expert_idx[j < TK ? j : TK - 1] : -1;  // (no condition per lane: no wait per load)
  }
#pragma unroll
  for (int i = 0; i < M1_STEPS; i++) ids[i] = first + i * 64 < TK ? (int)opaque(ids[i]) : -1;
  for (int e = lane; e < E; e += 64) cursor[e] = 0;
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int i = 0; i < M1_STEPS; i++)
    if (ids[i] >= 0 && ids[i] < E) atomicAdd(&cursor[ids[i]], 1);
  __syncthreads();
  counts_to_cursors<M1_WAVES>(lds, E, wave_total, freq, off);
#pragma unroll
  for (int i = 0; i < M1_STEPS; i++) {
    const int j = first + i * 64;
    if (i < steps && j - lane < TK)
      place_slots(ids[i], j, j < TK, lane, token_idx, TK, T, E, K, ebits, cursor, gidx, sidx, ridx, tok_off);
  }
  if (tok_off && TK == 0)
    for (int64_t u = tid; u <= T; u += 64 * M1_WAVES) tok_off[u] = 0;
  // (off was written before the last barrier.  3108 slots, E = 48: 10.6 us with the two maps, 8.4 + 3.7 apart)
  if (maps.map[0].header != nullptr)
    for (int which = 0; which < 2; which++)
      write_tile_map<M1_WAVES, false>(nullptr, off, nullptr, E, tile_map_rows(which), maps.gmax, maps.snake,
                                      which == 0 ? maps.map[0] : maps.map[1], map_part[which]);
}

}  // namespace smoe

using namespace smoe;

extern "C" int smoe_count_cumsum(const void* x, int x_is_int64, int64_t n, int E, int32_t* count, int32_t* cumsum,
                                 void* stream) {
  SMOE_REQUIRE(count != nullptr && (x != nullptr || n == 0), SMOE_ERR_INVALID, "count_cumsum: null pointer");
  SMOE_REQUIRE(n >= 0, SMOE_ERR_INVALID, "count_cumsum: negative length");
  SMOE_REQUIRE(E >= 1 && E <= 65536, SMOE_ERR_UNSUPPORTED, "count_cumsum: E=%d outside [1, 65536]", E);
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL(fill_i32_kernel, dim3((unsigned)ceil_div(E, 256)), dim3(256), 0, st, count, (int64_t)E, 0);
  SMOE_LAUNCH_CHECK();
  if (n > 0) {
    const bool use_lds = E <= 8192;
    int blocks = (int)(ceil_div(n, 1024 * 8) < 256 ? ceil_div(n, 1024 * 8) : 256);
    if (blocks < 1) blocks = 1;
    const size_t smem = use_lds ? (size_t)E * 4 : 0;
    if (x_is_int64) {
      if (use_lds)
        hipLaunchKernelGGL((count_kernel<int64_t, true>), dim3(blocks), dim3(1024), smem, st, (const int64_t*)x, n,
                           E, count);
      else
        hipLaunchKernelGGL((count_kernel<int64_t, false>), dim3(blocks), dim3(1024), 0, st, (const int64_t*)x, n, E,
                           count);
    } else {
      if (use_lds)
        hipLaunchKernelGGL((count_kernel<int32_t, true>), dim3(blocks), dim3(1024), smem, st, (const int32_t*)x, n,
                           E, count);
      else
        hipLaunchKernelGGL((count_kernel<int32_t, false>), dim3(blocks), dim3(1024), 0, st, (const int32_t*)x, n, E,
                           count);
    }
    SMOE_LAUNCH_CHECK();
  }
  if (cumsum) {
    hipLaunchKernelGGL(inclusive_scan_kernel, dim3(1), dim3(1024), 0, st, count, E, cumsum);
    SMOE_LAUNCH_CHECK();
  }
  return SMOE_OK;
}

extern "C" int smoe_topk_softmax_fwd(const void* logits, int dtype, int64_t T, int E, int K, int64_t row_stride,
                                     float* scores, int32_t* indices, int softmax, void* stream) {
  SMOE_REQUIRE(T >= 0, SMOE_ERR_INVALID, "topk: negative T");
  if (T == 0) return SMOE_OK;
  SMOE_REQUIRE(logits && scores && indices, SMOE_ERR_INVALID, "topk: null pointer");
  SMOE_REQUIRE(E >= 1 && E <= 4096, SMOE_ERR_UNSUPPORTED, "topk: E=%d outside [1, 4096]", E);
  SMOE_REQUIRE(K >= 1 && K <= E && K <= 64, SMOE_ERR_UNSUPPORTED, "topk: K=%d outside [1, min(E, 64)]", K);
  SMOE_REQUIRE(row_stride >= E, SMOE_ERR_INVALID, "topk: row stride %lld < E", (long long)row_stride);
  hipStream_t st = (hipStream_t)stream;
  uint32_t p2 = 1;
  while ((int)p2 < E) p2 <<= 1;
  switch (dtype) {
    case SMOE_DT_BF16:
      return launch_topk<uint16_t>(logits, T, E, K, row_stride, scores, indices, softmax, 0xffffffffu, st);
    case SMOE_DT_F16:
      return launch_topk<__half>(logits, T, E, K, row_stride, scores, indices, softmax, ~(p2 - 1), st);
    case SMOE_DT_F32:
      return launch_topk<float>(logits, T, E, K, row_stride, scores, indices, softmax, ~(p2 - 1), st);
  }
  set_error("topk: unknown dtype %d", dtype);
  return SMOE_ERR_INVALID;
}

extern "C" int smoe_softmax_topk_bwd(void* dlogits, int dtype, int64_t row_stride, const void* dlogits_add,
                                     const float* dscores, const float* scores, const int32_t* indices, int64_t T, int K,
                                     void* stream) {
  SMOE_REQUIRE(T >= 0 && K >= 1, SMOE_ERR_INVALID, "softmax_topk_bwd: bad sizes");
  if (T == 0) return SMOE_OK;
  SMOE_REQUIRE(dlogits && dscores && scores && indices, SMOE_ERR_INVALID, "softmax_topk_bwd: null pointer");
  hipStream_t st = (hipStream_t)stream;
  const dim3 grid((unsigned)ceil_div(T, 256)), block(256);
  switch (dtype) {
    case SMOE_DT_BF16:
      hipLaunchKernelGGL(softmax_topk_bwd_kernel<uint16_t>, grid, block, 0, st, (uint16_t*)dlogits, row_stride,
                         (const uint16_t*)dlogits_add, dscores, scores, indices, T, K);
      break;
    case SMOE_DT_F16:
      hipLaunchKernelGGL(softmax_topk_bwd_kernel<__half>, grid, block, 0, st, (__half*)dlogits, row_stride,
                         (const __half*)dlogits_add, dscores, scores, indices, T, K);
      break;
    case SMOE_DT_F32:
      hipLaunchKernelGGL(softmax_topk_bwd_kernel<float>, grid, block, 0, st, (float*)dlogits, row_stride,
                         (const float*)dlogits_add, dscores, scores, indices, T, K);
      break;
    default:
      set_error("softmax_topk_bwd: unknown dtype %d", dtype);
      return SMOE_ERR_INVALID;
  }
  SMOE_LAUNCH_CHECK();
  return SMOE_OK;
}

extern "C" int smoe_router_logit_grad(void* dlogits, int dtype, int64_t row_stride, const void* outside,
                                      int64_t outside_stride, const float* dscores, const float* scores,
                                      const int32_t* indices, int64_t T, int E, int K, void* stream) {
  SMOE_REQUIRE(T >= 0 && T < (1ll << 31) && E >= 1 && K >= 1, SMOE_ERR_INVALID, "router_logit_grad: bad sizes");
  if (T == 0) return SMOE_OK;
  SMOE_REQUIRE(dlogits && dscores && scores && indices, SMOE_ERR_INVALID, "router_logit_grad: null pointer");
  SMOE_REQUIRE(row_stride >= E && (outside == nullptr || outside_stride >= E || T == 1), SMOE_ERR_INVALID,
               "router_logit_grad: row stride below E");
  hipStream_t st = (hipStream_t)stream;
  switch (dtype) {
    case SMOE_DT_BF16:
      launch_router_logit_grad<uint16_t>(dlogits, row_stride, outside, outside_stride, dscores, scores, indices, T, E, K, st);
      break;
    case SMOE_DT_F16:
      launch_router_logit_grad<__half>(dlogits, row_stride, outside, outside_stride, dscores, scores, indices, T, E, K, st);
      break;
    case SMOE_DT_F32:
      launch_router_logit_grad<float>(dlogits, row_stride, outside, outside_stride, dscores, scores, indices, T, E, K, st);
      break;
    default:
      set_error("router_logit_grad: unknown dtype %d", dtype);
      return SMOE_ERR_INVALID;
  }
  SMOE_LAUNCH_CHECK();
  return SMOE_OK;
}

extern "C" int smoe_topk_bwd(void* dlogits, int dtype, int64_t row_stride, const float* dvalues, const int32_t* indices,
                             int64_t T, int K, void* stream) {
  SMOE_REQUIRE(T >= 0 && K >= 1, SMOE_ERR_INVALID, "topk_bwd: bad sizes");
  if (T == 0) return SMOE_OK;
  SMOE_REQUIRE(dlogits && dvalues && indices, SMOE_ERR_INVALID, "topk_bwd: null pointer");
  hipStream_t st = (hipStream_t)stream;
  const dim3 grid((unsigned)ceil_div(T, 256)), block(256);
  switch (dtype) {
    case SMOE_DT_BF16:
      hipLaunchKernelGGL(topk_bwd_kernel<uint16_t>, grid, block, 0, st, (uint16_t*)dlogits, row_stride, dvalues, indices,
                         T, K);
      break;
    case SMOE_DT_F16:
      hipLaunchKernelGGL(topk_bwd_kernel<__half>, grid, block, 0, st, (__half*)dlogits, row_stride, dvalues, indices, T,
                         K);
      break;
    case SMOE_DT_F32:
      hipLaunchKernelGGL(topk_bwd_kernel<float>, grid, block, 0, st, (float*)dlogits, row_stride, dvalues, indices, T, K);
      break;
    default:
      set_error("topk_bwd: unknown dtype %d", dtype);
      return SMOE_ERR_INVALID;
  }
  SMOE_LAUNCH_CHECK();
  return SMOE_OK;
}

static inline int meta_segments(int64_t TK) {
  int64_t ns = ceil_div(TK, smoe::SEG);
  return (int)(ns < 1 ? 1 : ns);
}

extern "C" size_t smoe_routing_metadata_workspace_bytes(int64_t TK, int E) {
  if (TK < 0 || E < 1) return 0;
  return (size_t)2 * (size_t)E * (size_t)meta_segments(TK) * sizeof(int32_t);
}

// argument checks shared by the two metadata entry points (everything but the scratch memory)
static int check_routing_metadata_args(const int32_t* expert_idx, const int32_t* token_idx, int64_t TK, int64_t T, int E,
                                       int K, const int32_t* freq, const int32_t* off, const int32_t* x_gather_idx,
                                       const int32_t* s_scatter_idx, const int32_t* s_reverse_scatter_idx) {
  SMOE_REQUIRE(TK >= 0 && T >= 0, SMOE_ERR_INVALID, "routing_metadata: negative size");
  SMOE_REQUIRE(TK < (1ll << 31), SMOE_ERR_UNSUPPORTED, "routing_metadata: TK does not fit int32");
  SMOE_REQUIRE(E >= 1 && E <= 4096, SMOE_ERR_UNSUPPORTED, "routing_metadata: E=%d outside [1, 4096]", E);
  SMOE_REQUIRE(freq && off, SMOE_ERR_INVALID, "routing_metadata: null pointer");
  SMOE_REQUIRE(TK == 0 || (expert_idx && x_gather_idx && s_scatter_idx && s_reverse_scatter_idx), SMOE_ERR_INVALID,
               "routing_metadata: null pointer");
  SMOE_REQUIRE(token_idx != nullptr || K >= 1, SMOE_ERR_INVALID, "routing_metadata: K must be >= 1 without token_idx");
  return SMOE_OK;
}

// The maps need the counts only, which the scan has left: two workgroups behind the segments write them while the slots are
// placed.  6001 tokens, E = 128, K = 8: 7.4 us, 7.7 without the maps and 4.6 for a launch of them.  MAPS_MAX_E: as many
// experts as the 256 threads of a map's workgroup list at once.
constexpr int MAPS_MAX_E = 64 * META_WAVES;

// the three passes of the counting sort, and with `maps` the tile maps in the last one's launch; `workspace` holds the two
// (E, NS) int32 tables, both written in full by the first two passes before they are read (nothing in it has to start at
// zero)
static int launch_routing_metadata(const int32_t* expert_idx, const int32_t* token_idx, int64_t TK, int64_t T, int E,
                                   int K, int32_t* freq, int32_t* off, int32_t* x_gather_idx, int32_t* s_scatter_idx,
                                   int32_t* s_reverse_scatter_idx, int32_t* tok_off, void* workspace, hipStream_t st,
                                   const TileMapPair* maps = nullptr, bool* maps_written = nullptr) {
  const int NS = meta_segments(TK);
  int32_t* hist_t = (int32_t*)workspace;
  int32_t* base_t = hist_t + (size_t)E * NS;
  int ebits = 0;
  while ((1 << ebits) < E) ebits++;
  if (TK <= M1_SLOTS && E <= M1_MAX_E) {
    const int steps = (int)ceil_div(TK, 64 * M1_WAVES);
    hipLaunchKernelGGL(meta_one_kernel, dim3(1), dim3(64 * M1_WAVES), (size_t)M1_WAVES * E * sizeof(int32_t), st, expert_idx,
                       token_idx, (int)TK, T, E, K, ebits, steps, freq, off, x_gather_idx, s_scatter_idx,
                       s_reverse_scatter_idx, tok_off, maps ? *maps : TileMapPair{});
    SMOE_LAUNCH_CHECK();
    if (maps) *maps_written = true;
    return SMOE_OK;
  }
  const dim3 grid_seg((unsigned)NS), block_seg(64 * META_WAVES);
  const size_t smem = (size_t)META_WAVES * (E + 1) * sizeof(int32_t);
  static LdsLimitOnce lds_limit;  // E = 4096 is the first size beyond 64 KiB
  const int rc_attr = lds_limit.ensure((const void*)meta_scatter_kernel, META_WAVES * (4096 + 1) * (int)sizeof(int32_t));
  if (rc_attr) return rc_attr;
  hipLaunchKernelGGL(meta_hist_kernel, grid_seg, block_seg, (size_t)E * sizeof(int32_t), st, expert_idx, (int)TK, E, NS,
                     hist_t);
  SMOE_LAUNCH_CHECK();
  hipLaunchKernelGGL(meta_scan_kernel, dim3((unsigned)ceil_div(E, 4)), dim3(256), 0, st, hist_t, E, NS, base_t, freq);
  SMOE_LAUNCH_CHECK();
  const bool write_maps = maps != nullptr && E <= MAPS_MAX_E;
  hipLaunchKernelGGL(meta_scatter_kernel, dim3((unsigned)NS + (write_maps ? 2 : 0)), block_seg, smem, st, expert_idx,
                     token_idx, (int)TK, T, E, K, NS, ebits, freq, base_t, off, x_gather_idx, s_scatter_idx,
                     s_reverse_scatter_idx, tok_off, write_maps ? *maps : TileMapPair{});
  SMOE_LAUNCH_CHECK();
  if (write_maps) *maps_written = true;
  return SMOE_OK;
}

extern "C" int smoe_routing_metadata(const int32_t* expert_idx, const int32_t* token_idx, int64_t TK, int64_t T,
                                     int E, int K, int32_t* freq, int32_t* off, int32_t* x_gather_idx,
                                     int32_t* s_scatter_idx, int32_t* s_reverse_scatter_idx, int32_t* tok_off,
                                     void* workspace, size_t workspace_bytes, void* stream) {
  const int rc = check_routing_metadata_args(expert_idx, token_idx, TK, T, E, K, freq, off, x_gather_idx, s_scatter_idx,
                                             s_reverse_scatter_idx);
  if (rc) return rc;
  SMOE_REQUIRE(workspace != nullptr, SMOE_ERR_INVALID, "routing_metadata: null pointer");
  SMOE_REQUIRE(workspace_bytes >= smoe_routing_metadata_workspace_bytes(TK, E), SMOE_ERR_WORKSPACE,
               "routing_metadata: workspace too small");
  return launch_routing_metadata(expert_idx, token_idx, TK, T, E, K, freq, off, x_gather_idx, s_scatter_idx,
                                 s_reverse_scatter_idx, tok_off, workspace, (hipStream_t)stream);
}

int smoe::routing_metadata_and_maps(const int32_t* expert_idx, int64_t TK, int64_t T, int E, int K, int32_t* freq,
                                    int32_t* off, int32_t* x_gather_idx, int32_t* s_scatter_idx, int32_t* s_reverse_scatter_idx,
                                    int32_t* tok_off, void* workspace, size_t workspace_bytes, const TileMapPair* maps,
                                    bool* maps_written, hipStream_t st) {
  const int rc = check_routing_metadata_args(expert_idx, nullptr, TK, T, E, K, freq, off, x_gather_idx, s_scatter_idx,
                                             s_reverse_scatter_idx);
  if (rc) return rc;
  SMOE_REQUIRE(workspace != nullptr, SMOE_ERR_INVALID, "routing_metadata: null pointer");
  SMOE_REQUIRE(workspace_bytes >= smoe_routing_metadata_workspace_bytes(TK, E), SMOE_ERR_WORKSPACE,
               "routing_metadata: workspace too small");
  return launch_routing_metadata(expert_idx, nullptr, TK, T, E, K, freq, off, x_gather_idx, s_scatter_idx,
                                 s_reverse_scatter_idx, tok_off, workspace, st, maps, maps_written);
}

// ---- the same operator for callers that cannot allocate ------------------------------------------------------
// The two tables live in a device array that is part of the library image: one copy per GPU, at an address of its
// own on each, looked up once per device.  In host code the array's NAME is only a handle for that look-up; the
// kernels get the looked-up pointer.
static __device__ __align__(256) unsigned char scratch[SMOE_ROUTING_METADATA_STATIC_BYTES];

namespace {
constexpr int MAX_DEVICES = 64;
std::mutex scratch_mutex;
void* scratch_ptr[MAX_DEVICES] = {};  // device address of `scratch` on each GPU, null = not looked up yet
}  // namespace

// device address of this GPU's copy of `scratch`
static int static_scratch(void** out) {
  int dev = 0;
  SMOE_HIP_CHECK(hipGetDevice(&dev));
  SMOE_REQUIRE(dev >= 0 && dev < MAX_DEVICES, SMOE_ERR_UNSUPPORTED, "routing_metadata_static: device %d out of range",
               dev);
  std::lock_guard<std::mutex> lock(scratch_mutex);
  if (scratch_ptr[dev] == nullptr) {
    void* p = nullptr;
    SMOE_HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    SMOE_REQUIRE(p != nullptr, SMOE_ERR_HIP, "routing_metadata_static: no device address for the scratch array");
    scratch_ptr[dev] = p;
  }
  *out = scratch_ptr[dev];
  return SMOE_OK;
}

extern "C" size_t smoe_routing_metadata_static_capacity(void) { return SMOE_ROUTING_METADATA_STATIC_BYTES; }

extern "C" int smoe_routing_metadata_static(const int32_t* expert_idx, const int32_t* token_idx, int64_t TK, int64_t T,
                                            int E, int K, int32_t* freq, int32_t* off, int32_t* x_gather_idx,
                                            int32_t* s_scatter_idx, int32_t* s_reverse_scatter_idx, int32_t* tok_off,
                                            void* stream) {
  int rc = check_routing_metadata_args(expert_idx, token_idx, TK, T, E, K, freq, off, x_gather_idx, s_scatter_idx,
                                       s_reverse_scatter_idx);
  if (rc) return rc;
  const size_t need = smoe_routing_metadata_workspace_bytes(TK, E);
  SMOE_REQUIRE(need <= (size_t)SMOE_ROUTING_METADATA_STATIC_BYTES, SMOE_ERR_WORKSPACE,
               "routing_metadata_static: TK=%lld, E=%d need %zu bytes of scratch, the built-in array holds %zu; use "
               "smoe_routing_metadata with a workspace of your own",
               (long long)TK, E, need, (size_t)SMOE_ROUTING_METADATA_STATIC_BYTES);
  void* ws = nullptr;
  rc = static_scratch(&ws);
  if (rc) return rc;
  return launch_routing_metadata(expert_idx, token_idx, TK, T, E, K, freq, off, x_gather_idx, s_scatter_idx,
                                 s_reverse_scatter_idx, tok_off, ws, (hipStream_t)stream);
}
