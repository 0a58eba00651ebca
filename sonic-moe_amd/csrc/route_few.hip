// The routing of few tokens in two launches instead of four or five: at 1 to 64 tokens each of those is a few memory latencies
// long, and they stand in a row in front of the experts.
//   router_logits_kernel   logits = x Wr^T, the weights spread over the chip
//   route_few_kernel       top-K softmax, counting sort and the load-balancing loss in one workgroup
#include "gemm_common.h"
#include "routing_common.h"

namespace smoe {

// ---- router GEMM ----------------------------------------------------------------------------------------------------------
// 16 experts x 16 tokens, the contraction in 16 consecutive parts, one to a wavefront, which loads fragments of both operands
// straight into registers, eight k-steps of 32 at once (all that a part has at H <= 4096).  The parts are added four by four in
// a fixed order.  What it costs is latency and the 256 KiB (at H = 4096) that one compute unit draws for such a tile, so for
// the fused routing four workgroups share a tile (SPLIT: four wavefronts each, fp32 sums to `partial` (4, T, E), which the
// routing kernel adds); alone it is one workgroup of sixteen wavefronts with the same sums.
constexpr int RL_PARTS = 16, RL_GROUP = 4, RL_AHEAD = 8;

template <bool SPLIT>
__global__ __launch_bounds__(64 * (SPLIT ? RL_GROUP : RL_PARTS)) void router_logits_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ wr, int T, int H, int E, uint16_t* __restrict__ logits,
    float* __restrict__ partial) {
  constexpr int WAVES = SPLIT ? RL_GROUP : RL_PARTS;
  __shared__ f32x4 red[WAVES][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int e0 = blockIdx.x * 16, t0 = blockIdx.y * 16;
  const int e = e0 + (lane & 15), t = t0 + (lane & 15);
  // (experts and tokens past the end repeat the last one; their products are not stored)
  const uint16_t* wp = wr + (int64_t)(e < E ? e : E - 1) * H + 8 * (lane >> 4);
  const uint16_t* xp = x + (int64_t)(t < T ? t : T - 1) * H + 8 * (lane >> 4);
  const int steps = H / 32, per = (steps + RL_PARTS - 1) / RL_PARTS;
  const int first = (blockIdx.z * RL_GROUP + wave) * per, last = first + per < steps ? first + per : steps;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int s = first; s < last; s += RL_AHEAD) {
    elemx8 w[RL_AHEAD], p[RL_AHEAD];
#pragma unroll
    for (int i = 0; i < RL_AHEAD; i++) {
      const int at = (s + i < last ? s + i : last - 1) * 32;
      w[i] = *(const elemx8*)(wp + at);
      p[i] = *(const elemx8*)(xp + at);
    }
    __builtin_amdgcn_sched_barrier(0);  // all loads before the first product
#pragma unroll
    for (int i = 0; i < RL_AHEAD; i++)
      if (s + i < last) acc = ElemMma16::run(w[i], p[i], acc);
  }
  red[wave][lane] = acc;
  __syncthreads();
  if (tid >= 64) return;
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int g = 0; g < WAVES / RL_GROUP; g++) {
    f32x4 group = red[g * RL_GROUP][tid];
#pragma unroll
    for (int w = 1; w < RL_GROUP; w++) group += red[g * RL_GROUP + w][tid];
    v = g == 0 ? group : v + group;
  }
  const int col = e0 + 4 * (tid >> 4), row = t0 + (tid & 15);
  if (row >= T) return;
  if constexpr (SPLIT) {
    float* out = partial + ((int64_t)blockIdx.z * T + row) * E + col;
#pragma unroll
    for (int i = 0; i < 4; i++)
      if (col + i < E) out[i] = v[i];
  } else {
    uint16_t* out = logits + (int64_t)row * E + col;
    const uint32_t lo = pack_elem2(v[0], v[1]), hi = pack_elem2(v[2], v[3]);
    if (col < E) out[0] = (uint16_t)lo;
    if (col + 1 < E) out[1] = (uint16_t)(lo >> 16);
    if (col + 2 < E) out[2] = (uint16_t)hi;
    if (col + 3 < E) out[3] = (uint16_t)(hi >> 16);
  }
}

// ---- top-K, metadata and loss ----------------------------------------------------------------------------------------------
// One workgroup of 16 wavefronts, in three steps:
//   a wavefront owns the rows w, w + 16, ...: it adds a row's four partial sums, stores the logits, leaves them in LDS as they
//   are stored, and adds the row's softmax to its column sums (the arithmetic and order of softmax_colsum_kernel)
//   16 lanes own a row: K rounds of an arg-max over them (the keys and the arithmetic of topk_softmax_kernel); at 64 rows the
//   compute unit's issue slots are what it takes, and four rows to an instruction save them (the kernel 17.8 -> 11.7 us)
//   the picks meet in LDS, every wavefront ranks 64 of them as meta_one_kernel does, and the loss follows from the counts
// Same bits as the three kernels.  The line: all picks in one step of the sort (1024), 256 experts in 52 KiB of LDS, and the
// loss's own line at 64 tokens, up to which the rows of a wavefront are added in this order.  Both kernels against the four
// they stand for (the library's GEMM 10 to 15 us of it), us: one token, H = 4096, E = 128, K = 8 28 -> 11; 23 tokens, H = 1536
// 27 -> 13; 64 tokens, H = 4096 35 -> 17.
constexpr int RF_WAVES = 16, RF_MAX_T = 64, RF_MAX_E = 256, RF_MAX_SLOTS = 1024;

#ifdef SMOE_ELEM_F16
typedef __half route_t;
#else
typedef uint16_t route_t;  // bf16 bits
#endif

// VPL: columns per lane of a wavefront that owns a row (E <= 64 * VPL)
template <int VPL>
__global__ __launch_bounds__(64 * RF_WAVES) void route_few_kernel(
    const float* __restrict__ partial, uint16_t* __restrict__ logits, int Trows, int E, int K, int ebits,
    float* __restrict__ scores, int32_t* __restrict__ indices, int32_t* __restrict__ freq, int32_t* __restrict__ off,
    int32_t* __restrict__ gidx, int32_t* __restrict__ sidx, int32_t* __restrict__ ridx, int32_t* __restrict__ tok_off,
    float* __restrict__ loss_acc, float* __restrict__ loss) {
  extern __shared__ int32_t lds[];  // column sums RF_WAVES x E, picks, and rows of logits or (afterwards) cursors RF_WAVES x E
  __shared__ int32_t wave_total[RF_WAVES];
  __shared__ float scratch[48];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, TK = Trows * K;
  float* sums = (float*)lds;
  int32_t* picks = lds + RF_WAVES * E;
  int32_t* cursors = picks + RF_MAX_SLOTS;
  int32_t* cursor = cursors + wave * E;
  uint16_t* rows = (uint16_t*)cursors;

  float acc[VPL];
#pragma unroll
  for (int i = 0; i < VPL; i++) acc[i] = 0.f;
  for (int row = wave; row < Trows; row += RF_WAVES) {
    float part[RL_GROUP][VPL], v[VPL];
#pragma unroll
    for (int z = 0; z < RL_GROUP; z++)
#pragma unroll
      for (int i = 0; i < VPL; i++) {
        const int c = lane + 64 * i;
        part[z][i] = partial[(z * Trows + row) * E + (c < E ? c : E - 1)];
      }
#pragma unroll
    for (int i = 0; i < VPL; i++) {
      const int c = lane + 64 * i;
      float sum = part[0][i];
#pragma unroll
      for (int z = 1; z < RL_GROUP; z++) sum += part[z][i];
      const uint16_t b = (uint16_t)pack_elem2(sum, sum);
      if (c < E) {
        logits[row * E + c] = b;
        rows[row * E + c] = b;
      }
      v[i] = c < E ? __uint_as_float(load_as_f32_bits<route_t>((const route_t*)&b)) : -INFINITY;
    }
    if (loss != nullptr) {
      row_softmax<VPL>(v);
#pragma unroll
      for (int i = 0; i < VPL; i++) acc[i] += v[i];
    }
  }
#pragma unroll
  for (int i = 0; i < VPL; i++) {
    const int c = lane + 64 * i;
    if (c < E) sums[wave * E + c] = acc[i];
  }
  __syncthreads();
  if (wave * 4 < Trows) {  // (the same for all lanes of a wavefront)
    const int g = lane & 15, row = wave * 4 + lane / 16;
    const bool row_ok = row < Trows;
    const uint16_t* src = rows + (row_ok ? row : Trows - 1) * E;
    typedef TopkKey<route_t> Top;
    uint32_t key[4 * VPL];
#pragma unroll
    for (int i = 0; i < 4 * VPL; i++) {
      const int c = g + 16 * i;
      key[i] = c < E ? Top::make(src[c], c) : 0;
    }
    pick_winners<Top>(key, 16, g, lane, row_ok, K, true, scores + row * K, indices + row * K, picks + row * K);
  }
  __syncthreads();
  for (int e = lane; e < E; e += 64) cursor[e] = 0;
  __syncthreads();
  const int j = wave * 64 + lane;
  const int id = j < TK ? picks[j] : -1;
  if (id >= 0 && id < E) atomicAdd(&cursor[id], 1);
  __syncthreads();
  const int32_t total = counts_to_cursors<RF_WAVES>(cursors, E, wave_total, freq, off);
  if (wave * 64 < TK)
    place_slots(id, j, j < TK, lane, nullptr, TK, Trows, E, K, ebits, cursor, gidx, sidx, ridx, tok_off);
  if (loss == nullptr) return;
  float sum = 0.f;
  if (tid < E) {
    for (int w = 0; w < RF_WAVES; w++) sum += sums[w * E + tid];
    loss_acc[tid] = sum;
  }
  const float fc = tid < E ? (float)total : 0.f;
  float f = fabsf(fc), d = sum * fc;
  block_sum3(sum, f, d, scratch);
  if (tid == 0) loss[0] = switch_loss_value(E, sum, f, d);
}

bool route_few_takes(int64_t T, int H, int E, int K) {
  return T <= RF_MAX_T && E <= RF_MAX_E && K <= 64 && K <= E && T * K <= RF_MAX_SLOTS && H % 32 == 0;
}
size_t route_few_workspace_bytes(int64_t T, int E) {
  return T <= RF_MAX_T && E <= RF_MAX_E ? (size_t)RL_GROUP * T * E * sizeof(float) : 0;
}

int launch_route_few(const void* x, const void* wr, int64_t T, int H, int E, int K, void* logits, float* scores,
                     int32_t* indices, int32_t* freq, int32_t* off, int32_t* gidx, int32_t* sidx, int32_t* ridx,
                     int32_t* tok_off, float* loss_acc, float* loss, void* workspace, hipStream_t st) {
  SMOE_REQUIRE(T >= 1 && E >= 1 && K >= 1 && H >= 32 && route_few_takes(T, H, E, K), SMOE_ERR_UNSUPPORTED,
               "route_few: sizes out of range");
  SMOE_REQUIRE(x && wr && logits && scores && indices && freq && off && gidx && sidx && ridx && tok_off && workspace &&
                   (!loss || loss_acc), SMOE_ERR_INVALID, "route_few: null pointer");
  SMOE_REQUIRE_ALIGNED("route_few", x, wr);
  float* partial = (float*)workspace;
  hipLaunchKernelGGL(router_logits_kernel<true>, dim3((unsigned)ceil_div(E, 16), (unsigned)ceil_div(T, 16), RL_PARTS / RL_GROUP),
                     dim3(64 * RL_GROUP), 0, st, (const uint16_t*)x, (const uint16_t*)wr, (int)T, H, E, nullptr, partial);
  SMOE_LAUNCH_CHECK();
  int ebits = 0;
  while ((1 << ebits) < E) ebits++;
  const int rows_words = (int)ceil_div(T * E, 2), cursor_words = RF_WAVES * E;
  const size_t smem = (size_t)(RF_WAVES * E + RF_MAX_SLOTS + (rows_words > cursor_words ? rows_words : cursor_words)) * 4;
  auto kernel = E <= 64 ? route_few_kernel<1> : E <= 128 ? route_few_kernel<2> : route_few_kernel<4>;
  hipLaunchKernelGGL(kernel, dim3(1), dim3(64 * RF_WAVES), smem, st, (const float*)partial, (uint16_t*)logits, (int)T, E, K,
                     ebits, scores, indices, freq, off, gidx, sidx, ridx, tok_off, loss_acc, loss);
  SMOE_LAUNCH_CHECK();
  return SMOE_OK;
}

}  // namespace smoe

using namespace smoe;

extern "C" int smoe_router_logits(const void* x, const void* wr, int64_t T, int H, int E, void* logits, void* stream) {
  SMOE_REQUIRE(T >= 1 && T < (1ll << 31) && E >= 1 && E <= (1 << 20), SMOE_ERR_INVALID, "router_logits: bad sizes");
  SMOE_REQUIRE(H >= 32 && H % 32 == 0, SMOE_ERR_UNSUPPORTED, "router_logits: H=%d must be a multiple of 32", H);
  SMOE_REQUIRE(ceil_div(T, 16) < 65536, SMOE_ERR_UNSUPPORTED, "router_logits: too many tokens");
  SMOE_REQUIRE(x && wr && logits, SMOE_ERR_INVALID, "router_logits: null pointer");
  SMOE_REQUIRE_ALIGNED("router_logits", x, wr);
  hipLaunchKernelGGL(router_logits_kernel<false>, dim3((unsigned)ceil_div(E, 16), (unsigned)ceil_div(T, 16)),
                     dim3(64 * RL_PARTS), 0, (hipStream_t)stream, (const uint16_t*)x, (const uint16_t*)wr, (int)T, H, E,
                     (uint16_t*)logits, nullptr);
  SMOE_LAUNCH_CHECK();
  return SMOE_OK;
}
