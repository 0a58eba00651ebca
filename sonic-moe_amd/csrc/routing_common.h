// What the routing kernels and the load-balancing loss share: sort keys of the top-K, one step of the counting sort, row
// softmax and sums over a wavefront or workgroup.
#pragma once
#include <hip/hip_fp16.h>

#include "common.h"
#include "tile_map.h"

namespace smoe {

// ---- reductions ----------------------------------------------------------------------------------------------------------
// Reductions over a wavefront in six steps of the vector pipe: neighbours, pairs and quads inside rows of 16 lanes by DPP,
// the rows by lane swaps.  Through __shfl_xor each step is a round trip to LDS of some 60 cycles, and a top-K of 8 is 48 of
// them in a row.  Every lane gets the result.
template <int CTRL>
SMOE_DEV uint32_t dpp(uint32_t v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true);
}
constexpr int DPP_XOR1 = 0xb1, DPP_XOR2 = 0x4e, DPP_HALF_MIRROR = 0x141, DPP_MIRROR = 0x140;
// op over lanes whose numbers differ in the bits below G (a power of two up to 64, the same for all lanes)
template <class V, class Op>
SMOE_DEV V group_reduce(V v, int G, Op op) {
  auto bits = [](V x) { return __builtin_bit_cast(uint32_t, x); };
  auto value = [](uint32_t x) { return __builtin_bit_cast(V, x); };
  if (G > 1) v = op(v, value(dpp<DPP_XOR1>(bits(v))));
  if (G > 2) v = op(v, value(dpp<DPP_XOR2>(bits(v))));
  if (G > 4) v = op(v, value(dpp<DPP_HALF_MIRROR>(bits(v))));  // (a quad's lanes agree by now: any lane of the other one)
  if (G > 8) v = op(v, value(dpp<DPP_MIRROR>(bits(v))));
  if (G > 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(bits(v), bits(v), false, false);
    v = op(value(r[0]), value(r[1]));
  }
  if (G > 32) {
    const auto r = __builtin_amdgcn_permlane32_swap(bits(v), bits(v), false, false);
    v = op(value(r[0]), value(r[1]));
  }
  return v;
}
SMOE_DEV uint32_t group_max(uint32_t v, int G) {
  return group_reduce(v, G, [](uint32_t a, uint32_t b) { return a > b ? a : b; });
}
SMOE_DEV float wave_max(float v) {
  return group_reduce(v, 64, [](float a, float b) { return fmaxf(a, b); });
}
SMOE_DEV float wave_sum(float v) {
  return group_reduce(v, 64, [](float a, float b) { return a + b; });
}

// ---- top-K keys (layout: routing.hip) ------------------------------------------------------------------------------------
SMOE_DEV uint32_t orderable(uint32_t bits) { return bits ^ ((bits >> 31) ? 0xffffffffu : 0x80000000u); }
SMOE_DEV uint32_t unorderable(uint32_t o) { return o ^ ((o >> 31) ? 0x80000000u : 0xffffffffu); }

template <typename T>
SMOE_DEV uint32_t load_as_f32_bits(const T* p);
template <>
__device__ __forceinline__ uint32_t load_as_f32_bits<uint16_t>(const uint16_t* p) {  // bf16
  return (uint32_t)(*p) << 16;
}
template <>
__device__ __forceinline__ uint32_t load_as_f32_bits<__half>(const __half* p) {
  return __float_as_uint(__half2float(*p));
}
template <>
__device__ __forceinline__ uint32_t load_as_f32_bits<float>(const float* p) {
  return __float_as_uint(*p);
}

template <typename T>
struct TopkKey;
template <>
struct TopkKey<float> {
  // Two words, compared one after the other.  As one 64-bit key a maximum was a compare and two selects, each waiting for the
  // one before, and went from lane to lane through LDS; us, that / this: E = 16, K = 16, 8192 rows 16.8/10.0; E = 256, K = 16
  // one row 17.7/8.3, 8192 rows 26.6/16.7; E = 4096, K = 32, 1000 rows 104/58.
  struct Key {
    uint32_t hi, lo;
  };
  static __device__ __forceinline__ uint32_t load(const float* p, uint32_t clear_mask) {
    return __float_as_uint(*p) & clear_mask;
  }
  static __device__ __forceinline__ Key make(uint32_t bits, int col) { return {orderable(bits), 0xffffffffu - (uint32_t)col}; }
  static __device__ __forceinline__ Key none() { return {0, 0}; }
  static __device__ __forceinline__ float value(Key k) { return __uint_as_float(unorderable(k.hi)); }
  static __device__ __forceinline__ int column(Key k) { return (int)(0xffffffffu - k.lo); }
  template <int COLS>
  static __device__ __forceinline__ Key best(const Key (&key)[COLS], int G) {
    uint32_t hi = key[0].hi, lo = 0;
#pragma unroll
    for (int i = 1; i < COLS; i++) hi = key[i].hi > hi ? key[i].hi : hi;
    hi = group_max(hi, G);
#pragma unroll
    for (int i = 0; i < COLS; i++) {
      const uint32_t c = key[i].hi == hi ? key[i].lo : 0;
      lo = c > lo ? c : lo;
    }
    return {hi, group_max(lo, G)};
  }
  static __device__ __forceinline__ bool same(Key a, Key b) { return a.lo == b.lo; }  // (columns of a row differ)
};
// (clearing the low bits of the fp32 image, log2(E) <= 12 of them, does not touch a 16-bit value)
template <typename T>
struct TopkKey16 {
  typedef uint32_t Key;
  static __device__ __forceinline__ uint32_t load(const T* p, uint32_t) { return *(const uint16_t*)p; }
  static __device__ __forceinline__ Key make(uint32_t bits, int col) {
    return (bits ^ ((bits >> 15) ? 0xffffu : 0x8000u)) << 16 | (0xffffu - (uint32_t)col);
  }
  static __device__ __forceinline__ float value(Key k) {
    const uint16_t o = (uint16_t)(k >> 16), bits = o ^ ((o >> 15) ? 0x8000u : 0xffffu);
    return __uint_as_float(load_as_f32_bits<T>((const T*)&bits));
  }
  static __device__ __forceinline__ int column(Key k) { return (int)(0xffffu - (k & 0xffffu)); }
  static __device__ __forceinline__ Key none() { return 0; }
  template <int COLS>
  static __device__ __forceinline__ Key best(const Key (&key)[COLS], int G) {
    Key k = key[0];
#pragma unroll
    for (int i = 1; i < COLS; i++) k = key[i] > k ? key[i] : k;
    return group_max(k, G);
  }
  static __device__ __forceinline__ bool same(Key a, Key b) { return a == b; }
};
template <>
struct TopkKey<uint16_t> : TopkKey16<uint16_t> {};
template <>
struct TopkKey<__half> : TopkKey16<__half> {};

// The K winners of a row whose keys G consecutive lanes hold (G a power of two up to 64, the same for all lanes of the
// wavefront; g = the lane's number in its row): K rounds of "arg-max over the row, retire the winner".  Lane g keeps the
// winners g, G + g, ...: their softmax, which needs one exponential per winner, is evaluated outside the rounds.  picks:
// nullable, the columns once more.
template <class Top, int COLS>
SMOE_DEV void pick_winners(typename Top::Key (&key)[COLS], int G, int g, int lane, bool row_ok, int K, bool softmax,
                           float* scores, int32_t* indices, int32_t* picks) {
  typedef typename Top::Key Key;
  float vmax = 0.f, esum = 0.f;
  for (int r0 = 0; r0 < K; r0 += G) {
    const int n = K - r0 < G ? K - r0 : G;
    Key mine = Top::none();
    for (int r = 0; r < n; r++) {
      const Key best = Top::best(key, G);
#pragma unroll
      for (int i = 0; i < COLS; i++) key[i] = Top::same(key[i], best) ? Top::none() : key[i];
      mine = g == r ? best : mine;
    }
    float out = Top::value(mine);
    if (softmax) {
      if (r0 == 0) vmax = __shfl(out, lane - g, 64);
      out = expf(out - vmax);
      for (int r = 0; r < n; r++) esum += __shfl(out, lane - g + r, 64);  // one after the other, as the winners come
    }
    if (row_ok && g < n) {
      const int col = Top::column(mine);
      indices[r0 + g] = col;
      if (picks != nullptr) picks[r0 + g] = col;
      scores[r0 + g] = out;  // (still to be divided by the sum)
    }
  }
  if (softmax && row_ok)
    for (int r = g; r < K; r += G) scores[r] = scores[r] / esum;  // the lane's own stores
}

// ---- counting sort ---------------------------------------------------------------------------------------------------------
// One step of the counting sort for a wavefront: lane l holds slot j (consecutive over the lanes, `valid` a prefix of them)
// of expert e.  Slots of the same expert take consecutive positions from that expert's cursor, in lane order.
SMOE_DEV void place_slots(int e, int j, bool valid, int lane, const int32_t* __restrict__ token_idx, int TK,
                          int64_t T, int E, int K, int ebits, int32_t* cursor, int32_t* __restrict__ gidx,
                          int32_t* __restrict__ sidx, int32_t* __restrict__ ridx, int32_t* __restrict__ tok_off) {
  const uint64_t lt_mask = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  const bool in_range = valid && e >= 0 && e < E;
  if (!in_range) e = 0;
  uint64_t peers = __ballot(in_range);
  for (int b = 0; b < ebits; b++) {
    const uint64_t bal = __ballot((e >> b) & 1);
    peers &= ((e >> b) & 1) ? bal : ~bal;
  }
  int32_t pos = 0;
  if (in_range) {
    pos = cursor[e] + __popcll(peers & lt_mask);
  }
  __builtin_amdgcn_wave_barrier();
  if (in_range && (peers >> lane) >> 1 == 0) cursor[e] = pos + 1;  // highest peer lane advances the cursor
  __builtin_amdgcn_wave_barrier();
  // (past the end j may not fit a token: nothing is read or written for it)
  int32_t t = 0;
  if (token_idx == nullptr)
    t = (int32_t)((uint32_t)j / (uint32_t)K);
  else if (valid)
    t = token_idx[j];
  if (in_range) {
    sidx[pos] = j;
    ridx[j] = pos;
    gidx[pos] = t;
  }
  if (tok_off && valid) {
    if (token_idx) {
      const int32_t tprev = j == 0 ? -1 : token_idx[j - 1];
      for (int32_t u = tprev + 1; u <= t; u++) tok_off[u] = j;
      if (j == TK - 1)
        for (int64_t u = (int64_t)t + 1; u <= T; u++) tok_off[u] = TK;
    } else {
      if (j == t * K) tok_off[t] = j;
      if (j == TK - 1) tok_off[T] = TK;
    }
  }
}

// The step between the counts and the ranking, of one workgroup whose thread e has expert e (E <= 64 * WAVES).  cursors: WAVES x
// E words of LDS, the wavefronts' counts, all written before; they become the positions at which each wavefront's slots of an
// expert begin.  Counts and offsets go to freq and off; returned is the expert's count (0 past the end).  total_of: WAVES words
// of LDS.  Begins without a barrier and ends with one.
template <int WAVES>
SMOE_DEV int32_t counts_to_cursors(int32_t* cursors, int E, int32_t* total_of, int32_t* __restrict__ freq,
                                   int32_t* __restrict__ off) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int32_t total = 0;
  if (tid < E) {
#pragma unroll
    for (int w = 0; w < WAVES; w++) {
      const int32_t n = cursors[w * E + tid];
      cursors[w * E + tid] = total;
      total += n;
    }
  }
  int32_t upto = total;
  for (int d = 1; d < 64; d <<= 1) {
    const int32_t o = __shfl_up(upto, d, 64);
    if (lane >= d) upto += o;
  }
  if (lane == 63) total_of[wave] = upto;
  __syncthreads();
  int32_t begin = upto - total;
  for (int w = 0; w < wave; w++) begin += total_of[w];
  if (tid < E) {
    freq[tid] = total;
    off[tid] = begin;
    if (tid == E - 1) off[E] = begin + total;
#pragma unroll
    for (int w = 0; w < WAVES; w++) cursors[w * E + tid] += begin;
  }
  __syncthreads();
  return total;
}

// ---- softmax of a row, sums --------------------------------------------------------------------------------------------------
template <typename T>
SMOE_DEV float sl_load(const T* p);
template <>
__device__ __forceinline__ float sl_load<uint16_t>(const uint16_t* p) {  // bf16
  return __uint_as_float((uint32_t)(*p) << 16);
}
template <>
__device__ __forceinline__ float sl_load<__half>(const __half* p) {
  return __half2float(*p);
}
template <>
__device__ __forceinline__ float sl_load<float>(const float* p) {
  return *p;
}

// softmax of one row held as VPL values per lane (columns lane + 64 i); columns >= E hold -inf and come out as 0
template <int VPL>
SMOE_DEV void row_softmax(float (&v)[VPL]) {
  float m = v[0];
#pragma unroll
  for (int i = 1; i < VPL; i++) m = fmaxf(m, v[i]);
  m = wave_max(m);
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < VPL; i++) {
    v[i] = __expf(v[i] - m);
    s += v[i];
  }
  s = wave_sum(s);
  const float inv = 1.0f / s;
#pragma unroll
  for (int i = 0; i < VPL; i++) v[i] *= inv;
}

template <typename T, int VPL>
SMOE_DEV void load_row(const T* row, int E, int lane, float (&v)[VPL]) {
#pragma unroll
  for (int i = 0; i < VPL; i++) {
    const int c = lane + 64 * i;
    v[i] = sl_load<T>(row + (c < E ? c : E - 1));
  }
}
// the columns past the end, once all of a wavefront's loads are under way
template <int VPL>
SMOE_DEV void mask_row(int E, int lane, float (&v)[VPL]) {
#pragma unroll
  for (int i = 0; i < VPL; i++) {
    const float x = __uint_as_float(opaque(__float_as_uint(v[i])));
    v[i] = lane + 64 * i < E ? x : -INFINITY;
  }
}

// block-wide sum of three values; every thread gets the totals
SMOE_DEV void block_sum3(float& a, float& b, float& c, float* scratch /* 3 * 16 floats */) {
  a = wave_sum(a);
  b = wave_sum(b);
  c = wave_sum(c);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  if (lane == 0) {
    scratch[wave] = a;
    scratch[16 + wave] = b;
    scratch[32 + wave] = c;
  }
  __syncthreads();
  a = b = c = 0.f;
  for (int w = 0; w < nw; w++) {
    a += scratch[w];
    b += scratch[16 + w];
    c += scratch[32 + w];
  }
  __syncthreads();
}

// The load-balancing loss of the sums of the softmax columns (s), of the counts (f) and of their products (d)
SMOE_DEV float switch_loss_value(int E, float s, float f, float d) {
  return (float)E * d / (fmaxf(s, 1e-12f) * fmaxf(f, 1e-12f));
}

// router_logits, top-K, metadata and loss of few tokens: route_few.hip
bool route_few_takes(int64_t T, int H, int E, int K);
size_t route_few_workspace_bytes(int64_t T, int E);
int launch_route_few(const void* x, const void* wr, int64_t T, int H, int E, int K, void* logits, float* scores,
                     int32_t* indices, int32_t* freq, int32_t* off, int32_t* gidx, int32_t* sidx, int32_t* ridx,
                     int32_t* tok_off, float* loss_acc, float* loss, void* workspace, hipStream_t st);

// smoe_routing_metadata of a top-K router's picks; the tile maps (nullable) too where they cost no launch of their
// own: routing.hip
int routing_metadata_and_maps(const int32_t* expert_idx, int64_t TK, int64_t T, int E, int K, int32_t* freq, int32_t* off,
                              int32_t* x_gather_idx, int32_t* s_scatter_idx, int32_t* s_reverse_scatter_idx,
                              int32_t* tok_off, void* workspace, size_t workspace_bytes, const TileMapPair* maps,
                              bool* maps_written, hipStream_t st);

}  // namespace smoe
