// Forward grouped GEMM for few token rows per expert (decode, short prompts):
//     C[m, n] = sum_k P[row(m), k] * Q_e[n, k]
// What bounds it is reading the weights of the picked experts once, so the kernel is built around the weight stream
// instead of around the matrix cores: no LDS ring, no barrier and no shared state in the contraction.
#include "gemm_common.h"

namespace smoe {

// A workgroup owns 64 weight rows (output columns) of one expert and up to 32 of its token rows.  Its four
// wavefronts split the contraction: wavefront w takes the pieces w, w + 4, ... of 64 elements (128 bytes of every row), so
// that together they walk through each weight row front to back.  A wavefront loads the matrix-core fragments of weights
// and tokens straight from memory into registers, DEPTH - 1 pieces ahead (two or three, one for blocks of more than 16
// rows), and the partial sums of the four are added in LDS in a fixed order.
constexpr int SK_NW = 4, SK_FN = 4, SK_BN = 16 * SK_FN, SK_PIECE = 64, SK_FM_MAX = 2;

constexpr int SK_ROWS = 16 * SK_FM_MAX;

// The experts' rows are cut into blocks of SK_ROWS.  With at least as many rows as experts, workgroup row y < E takes the
// first block of expert y (if it has one) and the workgroup rows behind them the further blocks of all experts in order;
// with fewer rows than experts workgroup row y takes the y-th block of all.  A block is found by counting, 256 experts at
// a time: a table would be a launch of its own.
struct SkinnyBlock {
  int e, row0, row_end;  // e < 0: there is no such block
};
// the y-th block that is not among the first `skip` of its expert
SMOE_DEV SkinnyBlock count_blocks(const int32_t* __restrict__ off, int E, int y, int skip, int lane) {
  for (int e0 = 0; e0 < E; e0 += 256) {  // lane l counts the experts e0 + 4 l .. e0 + 4 l + 3
    int lo[5], blocks = 0;
#pragma unroll
    for (int i = 0; i < 5; i++) {
      const int e = e0 + 4 * lane + i;
      lo[i] = off[e < E ? e : E];
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int n = (lo[i + 1] - lo[i] + SK_ROWS - 1) / SK_ROWS - skip;
      blocks += n > 0 ? n : 0;
    }
    int upto = blocks;  // of this and the lanes before
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int o = __shfl_up(upto, d, 64);
      upto += lane >= d ? o : 0;
    }
    const uint64_t past = __ballot(upto > y);
    if (past != 0) {
      const int src = __builtin_ctzll(past);  // the lane whose experts hold the block
      y -= __builtin_amdgcn_readlane(upto - blocks, src);
      SkinnyBlock b = {-1, 0, 0};
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int begin = __builtin_amdgcn_readlane(lo[i], src), end = __builtin_amdgcn_readlane(lo[i + 1], src);
        const int n = (end - begin + SK_ROWS - 1) / SK_ROWS - skip;
        if (b.e < 0 && y < n) b = {e0 + 4 * src + i, begin + (skip + y) * SK_ROWS, end};
        y -= n > 0 ? n : 0;
      }
      return b;
    }
    y -= __builtin_amdgcn_readlane(upto, 63);
  }
  return {-1, 0, 0};
}

SMOE_DEV elemx8 buffer_read16(const void* base, uint32_t bytes, uint32_t voff, uint32_t soff) {
  const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000);
  return __builtin_bit_cast(elemx8, __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, (int)soff, 0));
}

// Rows row0 .. row0 + 16 * FM - 1 (those below row_end) of one expert.
template <int FM, int DEPTH, bool WITH_ACT, int ACT>
SMOE_DEV void skinny_rows(const SkinnyGemm& g, const uint16_t* qe, const uint16_t* bias, f32x4* red, int n0, int row0,
                          int row_end, int wave, int lane) {
  constexpr int FN = SK_FN, KS = SK_NW;
  constexpr uint32_t NOWHERE = 0x80000000u;  // the launcher keeps both operands below 2 GiB: dropped by the range check
  const int pieces = g.Kdim / SK_PIECE;
  const uint32_t q_bytes = (uint32_t)((int64_t)g.N * g.q_stride_row * 2), p_bytes = (uint32_t)(g.p_rows * g.p_stride * 2);
  const uint32_t q_row = (uint32_t)(g.q_stride_row * 2);
  const uint32_t q_off = (uint32_t)(n0 + (lane & 15)) * q_row + (lane >> 4) * 16;
  uint32_t p_off[FM];
#pragma unroll
  for (int fm = 0; fm < FM; fm++) {
    const int m = row0 + fm * 16 + (lane & 15);
    int row = m < row_end ? m : row_end - 1;
    if (g.gidx != nullptr) row = g.gidx[row];
    p_off[fm] = m < row_end ? (uint32_t)row * (uint32_t)(g.p_stride * 2) + (lane >> 4) * 16 : NOWHERE;
  }

  f32x4 acc[FN][FM];
#pragma unroll
  for (int fn = 0; fn < FN; fn++)
#pragma unroll
    for (int fm = 0; fm < FM; fm++) acc[fn][fm] = f32x4{0.f, 0.f, 0.f, 0.f};

  elemx8 q[DEPTH][2][FN], pf[DEPTH][2][FM];
  const int n = pieces > wave ? (pieces - wave + KS - 1) / KS : 0;
  auto load = [&](auto slot_c, int i) {
    constexpr int slot = decltype(slot_c)::value % DEPTH;
    const uint32_t at = (uint32_t)(wave + i * KS) * (SK_PIECE * 2);
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {
#pragma unroll
      for (int fn = 0; fn < FN; fn++) q[slot][ks][fn] = buffer_read16(qe, q_bytes, q_off + ks * 64, at + fn * 16 * q_row);
#pragma unroll
      for (int fm = 0; fm < FM; fm++) pf[slot][ks][fm] = buffer_read16(g.P, p_bytes, p_off[fm] + ks * 64, at);
    }
    __builtin_amdgcn_sched_barrier(0);  // the compiler would sink the loads to their uses
  };
  auto multiply = [&](auto slot_c) {
    constexpr int slot = decltype(slot_c)::value % DEPTH;
#pragma unroll
    for (int ks = 0; ks < 2; ks++)
#pragma unroll
      for (int fn = 0; fn < FN; fn++)
#pragma unroll
        for (int fm = 0; fm < FM; fm++) acc[fn][fm] = ElemMma16::run(q[slot][ks][fn], pf[slot][ks][fm], acc[fn][fm]);
    __builtin_amdgcn_sched_barrier(0);
  };
  static_for<DEPTH - 1>([&](auto s) {
    if (decltype(s)::value < n) load(s, decltype(s)::value);
  });
  int i = 0;
  for (; i + 2 * DEPTH - 1 <= n; i += DEPTH) {  // every load is one of the wavefront's pieces
    static_for<DEPTH>([&](auto s) {
      load(std::integral_constant<int, decltype(s)::value + DEPTH - 1>{}, i + decltype(s)::value + DEPTH - 1);
      multiply(s);
    });
  }
  static_for<2 * DEPTH - 2>([&](auto s) {
    constexpr int ahead = decltype(s)::value + DEPTH - 1;
    if (ahead < 2 * DEPTH - 2 && i + ahead < n) load(std::integral_constant<int, ahead>{}, i + ahead);
    if (i + decltype(s)::value < n) multiply(s);
  });

  auto finish = [&](int fn, int fm, f32x4 v) {
    const int col = n0 + fn * 16 + 4 * (lane >> 4), m = row0 + fm * 16 + (lane & 15);
    if (bias != nullptr) {
      const u32x2 b = *(const u32x2*)(bias + col);
      v[0] += elem_lo(b[0]);
      v[1] += elem_hi(b[0]);
      v[2] += elem_lo(b[1]);
      v[3] += elem_hi(b[1]);
    }
    if (m < row_end) {
      if (!WITH_ACT || g.out0 != nullptr)
        *(u32x2*)(g.out0 + (int64_t)m * g.out0_stride + col) = u32x2{pack_elem2(v[0], v[1]), pack_elem2(v[2], v[3])};
      if constexpr (WITH_ACT) {
        constexpr int PW = act_pointwise(ACT);
        if constexpr (act_is_glu(ACT)) {
          *(uint32_t*)(g.out1 + (int64_t)m * g.out1_stride + col / 2) =
              pack_elem2(pointwise<PW>(v[0]) * v[1], pointwise<PW>(v[2]) * v[3]);
        } else {
          *(u32x2*)(g.out1 + (int64_t)m * g.out1_stride + col) =
              u32x2{pack_elem2(pointwise<PW>(v[0]), pointwise<PW>(v[1])), pack_elem2(pointwise<PW>(v[2]), pointwise<PW>(v[3]))};
        }
      }
    }
  };
#pragma unroll
  for (int fn = 0; fn < FN; fn++)
#pragma unroll
    for (int fm = 0; fm < FM; fm++) red[((fn * FM + fm) * KS + wave) * 64 + lane] = acc[fn][fm];
  __syncthreads();
#pragma unroll 1
  for (int f = wave; f < FN * FM; f += KS) {  // wavefront w finishes the fragments w, w + KS, ...
    f32x4 v = red[(f * KS) * 64 + lane];
#pragma unroll
    for (int w = 1; w < KS; w++) v += red[(f * KS + w) * 64 + lane];
    finish(f / FM, f % FM, v);
  }
}

template <int DEPTH, bool WITH_ACT, int ACT>
__global__ __launch_bounds__(SK_NW * 64, DEPTH >= 4 ? 2 : 3) void skinny_gemm_kernel(const SkinnyGemm g) {
  __shared__ f32x4 red[SK_FN * SK_FM_MAX * SK_NW * 64];  // one quad per lane, wavefront and fragment: 32 KiB
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  SkinnyBlock b;
  if (!g.first_blocks) {
    b = count_blocks(g.off, g.E, blockIdx.y, 0, lane);
  } else if ((int)blockIdx.y < g.E) {
    b = {(int)blockIdx.y, g.off[blockIdx.y], g.off[blockIdx.y + 1]};
  } else {
    b = count_blocks(g.off, g.E, blockIdx.y - g.E, 1, lane);
  }
  if (b.e < 0 || b.row0 >= b.row_end) return;
  const int n0 = blockIdx.x * SK_BN;
  const uint16_t* qe = g.Q + (int64_t)b.e * g.q_stride_e;
  const uint16_t* bias = g.bias ? g.bias + (int64_t)b.e * g.N : nullptr;
  if (b.row_end - b.row0 <= 16) {
    skinny_rows<1, DEPTH, WITH_ACT, ACT>(g, qe, bias, red, n0, b.row0, b.row_end, wave, lane);
  } else {
    skinny_rows<2, 2, WITH_ACT, ACT>(g, qe, bias, red, n0, b.row0, b.row_end, wave, lane);
  }
}

// the most blocks that TK rows of E experts can make
static int64_t skinny_blocks(const SkinnyGemm& g, int64_t TK) { return TK / SK_ROWS + (TK < g.E ? TK : g.E); }

// Where the line to the tile kernels lies, in token rows per expert on average.  A tile costs the same for one row as for
// 128 or 256, and a kernel of tiles needs some of them per compute unit; but it reads the weights of an expert with many
// rows once, where this kernel reads them from the caches again for every 32 rows.  SwiGLU, us, the tile kernel that would
// run / this kernel: even load, popularity by Zipf's law, all tokens with the same K experts.
//   (H, I)        E    rows   up                             down
//   (4096, 1024)  128   1     275/250  171/116   74/24       157/119   83/55    29/14
//                       4     368/360  174/174   76/50       209/176   96/86    29/28
//                       8     369/374  190/237   78/92       210/182  111/118   29/50
//   (4096,  256)  256   2     183/176   82/79    73/26       111/80    43/34    15/18
//                       4     194/188   86/103   73/48       120/91    55/46    15/26
//                       8     194/192  109/136   74/49       124/99    66/68    16/41
//                      16     195/200  177/190   74/94       130/117   84/108   22/71
//   (3072, 1408)  256   2     689/649  203/185   62/58       367/319  103/91    34/36
//                       4     761/729  216/263   64/108      400/357  111/128   33/52
//   (2048,  512)  256   4     209/187   65/69    44/30       109/93    33/32    13/18
//                      16     208/200  101/155   45/99       114/109   56/81    18/58
//   (1536,  256)  128   4      44/38    26/28    21/21        30/20    17/14    10/10
//                      16      45/43    37/42    22/29        31/23    22/24    10/16
//   (1472,  704)   48  16      54/44    40/46    21/29        31/24    24/27    14/17
//   (512,   256)    8  16      12/6     12/7     11/7          9/5      9/5      9/5
// Where the matrices fill the chip (512 tiles and more) the gain at an even load is small, and how many rows the most
// popular experts get grows with the rows of the launch: there the line is also drawn by those, sooner for a long
// contraction, whose workgroups take longer over a second block of rows.
bool skinny_gemm_takes(const SkinnyGemm& g, int64_t TK) {
  const int64_t lim = 1ll << 31;
  const int most = tuning().gemm_skinny_rows;
  int64_t rows = most;
  if (g.E * ceil_div(g.N, 256) >= 512) {
    rows = (16ll << 20) / ((int64_t)g.N * g.Kdim);
    rows = rows < most / 4 ? most / 4 : rows > most ? most : rows;
    if (TK > (g.Kdim >= 1024 ? 32ll : 128ll) * most) return false;
  }
  return TK <= rows * g.E && skinny_blocks(g, TK) <= 65535 && g.N % SK_BN == 0 && g.Kdim % SK_PIECE == 0 &&
         g.q_stride_row > 0 && g.N * g.q_stride_row * 2 < lim && g.p_rows * g.p_stride * 2 < lim;
}

template <bool WITH_ACT, int ACT>
static int launch_skinny(const SkinnyGemm& gin, int64_t TK, hipStream_t st) {
  SkinnyGemm g = gin;
  g.first_blocks = TK >= g.E;
  const dim3 grid((unsigned)(g.N / SK_BN), (unsigned)skinny_blocks(g, TK));
  // (pieces per wavefront; 16 or 6 at K = 4096, 1536, 4 or 1 at K = 1024, 256)
  if (g.Kdim >= 2048) {
    hipLaunchKernelGGL((skinny_gemm_kernel<4, WITH_ACT, ACT>), grid, dim3(SK_NW * 64), 0, st, g);
  } else {
    hipLaunchKernelGGL((skinny_gemm_kernel<3, WITH_ACT, ACT>), grid, dim3(SK_NW * 64), 0, st, g);
  }
  SMOE_LAUNCH_CHECK();
  return SMOE_OK;
}

int launch_skinny_gemm(const SkinnyGemm& g, int act, int64_t TK, hipStream_t st) {
  switch (act) {
    case -1: return launch_skinny<false, SMOE_ACT_RELU>(g, TK, st);
    case SMOE_ACT_SWIGLU: return launch_skinny<true, SMOE_ACT_SWIGLU>(g, TK, st);
    case SMOE_ACT_GEGLU: return launch_skinny<true, SMOE_ACT_GEGLU>(g, TK, st);
    case SMOE_ACT_REGLU: return launch_skinny<true, SMOE_ACT_REGLU>(g, TK, st);
    case SMOE_ACT_RELU_SQ: return launch_skinny<true, SMOE_ACT_RELU_SQ>(g, TK, st);
    case SMOE_ACT_RELU: return launch_skinny<true, SMOE_ACT_RELU>(g, TK, st);
    case SMOE_ACT_GELU: return launch_skinny<true, SMOE_ACT_GELU>(g, TK, st);
    case SMOE_ACT_SILU: return launch_skinny<true, SMOE_ACT_SILU>(g, TK, st);
  }
  set_error("unknown activation code %d", act);
  return SMOE_ERR_INVALID;
}

}  // namespace smoe
