// The token-choice layer's launches behind the router GEMM as one call per direction: the entry points of this library in
// the order in which the operators of the Python layer call them, on scratch memory that is carved here out of one buffer.
// No kernel of its own; the GEMMs of a direction share one tile map and one order of the experts (GemmScratch).  What it is
// for: a call of an operator from Python (argument checks, allocations, ctypes) costs 8 to 15 us of host time, more than
// most of the kernels take on a few tokens; a launch from here costs 3.
#include "gemm_common.h"
#include "routing_common.h"

namespace smoe {

// Scratch memory in pieces of whole 256 bytes
struct Carver {
  char* base;
  size_t used = 0;
  void* take(size_t bytes) {
    char* at = base + used;
    used += (bytes + 255) / 256 * 256;
    return at;
  }
};

struct ForwardScratch {
  void *y1, *y2, *map, *small_map, *metadata, *loss, *few;
  size_t metadata_bytes, loss_bytes, total;
  ForwardScratch(void* base, int64_t T, int H, int I, int E, int K) {
    Carver c{(char*)base};
    const int64_t TK = T * K;
    metadata_bytes = smoe_routing_metadata_workspace_bytes(TK, E);
    loss_bytes = smoe_switch_loss_workspace_bytes(T, E);
    map = c.take(smoe_gemm_workspace_bytes(TK, E));
    small_map = c.take(smoe_gemm_workspace_bytes(TK, E));
    metadata = c.take(metadata_bytes);
    loss = c.take(loss_bytes);
    few = c.take(route_few_workspace_bytes(T, E));
    y1 = c.take((size_t)TK * I * 2);
    y2 = c.take((size_t)TK * H * 2);
    total = c.used;
  }
};

struct BackwardScratch {
  void *dz, *y1s, *dx_expanded, *partial, *map, *small_map, *sorted;
  float *ds, *ds_partial;
  size_t sorted_bytes, total;
  BackwardScratch(void* base, int64_t T, int H, int I, int E, int K, int N1, int64_t chunks) {
    Carver c{(char*)base};
    const int64_t TK = T * K;
    map = c.take(smoe_gemm_workspace_bytes(TK, E));
    small_map = c.take(smoe_gemm_workspace_bytes(TK, E));
    sorted_bytes = (size_t)E * sizeof(int32_t);
    sorted = c.take(sorted_bytes);
    ds = (float*)c.take((size_t)TK * 4);
    // dz is done with when the chunks of the router's weight gradient are written (one chunk is the gradient itself)
    const size_t at_dz = c.used;
    partial = c.take((size_t)(chunks > 1 ? chunks : 0) * E * H * 2);
    const size_t behind_partial = c.used;
    c.used = at_dz;
    dz = c.take((size_t)TK * N1 * 2);
    if (c.used < behind_partial) c.used = behind_partial;
    // y1s and the score gradient's partial sums are done with when dx_expanded is written
    const size_t shared = c.used;
    y1s = c.take((size_t)TK * I * 2);
    ds_partial = (float*)c.take((size_t)TK * smoe_dz_partial_cols(I) * 4);
    total = c.used;
    c.used = shared;
    dx_expanded = c.take((size_t)TK * H * 2);
    if (c.used > total) total = c.used;
  }
};

#ifdef SMOE_ELEM_F16
constexpr int ELEM_DTYPE = SMOE_DT_F16;
#else
constexpr int ELEM_DTYPE = SMOE_DT_BF16;
#endif

static bool layer_sizes_ok(int64_t T, int64_t H, int64_t I, int64_t E, int64_t K) {
  const int64_t lim = 1ll << 31;
  return T > 0 && T < lim && H > 0 && H < (1 << 24) && I > 0 && I < (1 << 24) && E > 0 && E <= 4096 && K > 0 && K <= E &&
         T * K < lim;
}

}  // namespace smoe

using namespace smoe;

extern "C" size_t smoe_layer_forward_workspace_bytes(int64_t T, int H, int I, int E, int K) {
  return layer_sizes_ok(T, H, I, E, K) ? ForwardScratch(nullptr, T, H, I, E, K).total : 0;
}

extern "C" int smoe_layer_forward(const smoe_layer_forward_args* a, void* stream) {
  SMOE_REQUIRE(a != nullptr, SMOE_ERR_INVALID, "layer_forward: null pointer");
  SMOE_REQUIRE(layer_sizes_ok(a->T, a->H, a->I, a->E, a->K), SMOE_ERR_UNSUPPORTED, "layer_forward: sizes out of range");
  const int H = (int)a->H, I = (int)a->I, E = (int)a->E, K = (int)a->K;
  const int64_t T = a->T, TK = T * K;
  const ForwardScratch s(a->workspace, T, H, I, E, K);
  SMOE_REQUIRE(a->workspace != nullptr && a->workspace_bytes >= (int64_t)s.total, SMOE_ERR_WORKSPACE,
               "layer_forward: workspace too small");
  int rc = SMOE_OK;
  bool maps_written = false;
  SMOE_REQUIRE(a->router_w == nullptr || (a->logits_row_stride == E && a->logits_dtype == ELEM_DTYPE), SMOE_ERR_INVALID,
               "layer_forward: logits to be computed are contiguous, of the library's type");
  const bool few = a->router_w != nullptr && route_few_takes(T, H, E, K);
  if (few) {  // logits, top-K, metadata and loss in two launches, the same results
    rc = launch_route_few(a->x, a->router_w, T, H, E, K, a->logits, a->scores, a->indices, a->freq, a->off, a->x_gather_idx,
                          a->s_scatter_idx, a->s_reverse_scatter_idx, a->tok_off, a->loss_acc, a->loss, s.few,
                          (hipStream_t)stream);
    if (rc) return rc;
  } else {
    if (a->router_w != nullptr) {
      rc = smoe_router_logits(a->x, a->router_w, T, H, E, a->logits, stream);
      if (rc) return rc;
    }
    rc = smoe_topk_softmax_fwd(a->logits, (int)a->logits_dtype, T, E, K, a->logits_row_stride, a->scores, a->indices, 1,
                               stream);
    if (rc) return rc;
    // (to that many rows per expert the GEMMs may be the ones that walk no map)
    const TileMapPair maps = tile_map_pair(s.map, s.small_map, TK, E);
    const bool want_maps = TK > (int64_t)tuning().gemm_skinny_rows * E;
    rc = routing_metadata_and_maps(a->indices, TK, T, E, K, a->freq, a->off, a->x_gather_idx, a->s_scatter_idx,
                                   a->s_reverse_scatter_idx, a->tok_off, s.metadata, s.metadata_bytes,
                                   want_maps ? &maps : nullptr, &maps_written, (hipStream_t)stream);
    if (rc) return rc;
  }
  GemmScratch ws(s.map, s.small_map, nullptr, 0);
  if (maps_written) ws.map_rows = 256;
  rc = up_projection_forward(a->x, a->w1, a->w1_stride_e, a->w1_stride_row, a->b1, a->z, s.y1, a->off, nullptr,
                             a->x_gather_idx, T, TK, H, I, E, (int)a->activation, ws, stream);
  if (rc) return rc;
  rc = down_projection_forward(s.y1, a->w2, a->w2_stride_e, a->w2_stride_row, a->b2, s.y2, a->off, nullptr, TK, H, I, E, ws,
                               stream);
  if (rc) return rc;
  rc = smoe_gather_sum(s.y2, a->o, a->scores, a->s_reverse_scatter_idx, nullptr, T, K, H, stream);
  if (rc || few || a->loss == nullptr) return rc;
  return smoe_switch_loss_fwd(a->logits, (int)a->logits_dtype, a->logits_row_stride, T, E, a->freq, a->loss_acc, a->loss,
                              s.loss, s.loss_bytes, stream);
}

extern "C" size_t smoe_layer_backward_workspace_bytes(int64_t T, int H, int I, int E, int K, int activation, int chunks) {
  if (!layer_sizes_ok(T, H, I, E, K) || chunks < 0) return 0;
  return BackwardScratch(nullptr, T, H, I, E, K, activation <= SMOE_ACT_REGLU ? 2 * I : I, chunks).total;
}

extern "C" int smoe_layer_backward(const smoe_layer_backward_args* a, void* stream) {
  SMOE_REQUIRE(a != nullptr, SMOE_ERR_INVALID, "layer_backward: null pointer");
  SMOE_REQUIRE(layer_sizes_ok(a->T, a->H, a->I, a->E, a->K) && a->router_chunks >= 0 && a->router_chunks < 65536,
               SMOE_ERR_UNSUPPORTED, "layer_backward: sizes out of range");
  SMOE_REQUIRE(a->loss_grad == nullptr || a->outside == nullptr, SMOE_ERR_INVALID,
               "layer_backward: one gradient of the logits from outside, the loss's or another");
  const int H = (int)a->H, I = (int)a->I, E = (int)a->E, K = (int)a->K, act = (int)a->activation;
  const int64_t T = a->T, TK = T * K;
  const BackwardScratch s(a->workspace, T, H, I, E, K, act <= SMOE_ACT_REGLU ? 2 * I : I, a->router_chunks);
  SMOE_REQUIRE(a->workspace != nullptr && a->workspace_bytes >= (int64_t)s.total, SMOE_ERR_WORKSPACE,
               "layer_backward: workspace too small");
  GemmScratch ws(s.map, s.small_map, s.sorted, s.sorted_bytes);
  int rc = down_projection_backward(a->dout, a->z, a->w2, a->w2_stride_e, a->w2_stride_row, a->b2, a->dw2,
                                         a->dw2_stride_e, a->dw2_stride_row, a->db2, s.dz, s.y1s, s.ds, s.ds_partial,
                                         a->scores, a->off, nullptr, a->x_gather_idx, a->s_scatter_idx, T, TK, H, I, E, act,
                                         ws, stream);
  if (rc) return rc;
  rc = up_projection_backward(a->x, a->w1, a->w1_stride_e, a->w1_stride_row, s.dz, a->dw1, a->dw1_stride_e,
                                   a->dw1_stride_row, a->db1, s.dx_expanded, a->off, nullptr, a->x_gather_idx, T, TK, H, I, E,
                                   act, ws, stream);
  if (rc) return rc;
  if (a->router_w == nullptr) {
    rc = smoe_gather_sum(s.dx_expanded, a->dx, nullptr, a->s_reverse_scatter_idx, nullptr, T, K, H, stream);
    if (rc) return rc;
  }
  const void* outside = a->outside;
  int64_t outside_stride = a->outside_row_stride;
  if (a->loss_grad != nullptr) {
    rc = smoe_switch_loss_bwd(a->logits, (int)a->logits_dtype, a->logits_row_stride, T, E, a->freq, a->loss_acc, a->loss_grad,
                              a->dlogits, E, stream);
    if (rc) return rc;
    outside = a->dlogits;  // (the top-K's share is added in place)
    outside_stride = E;
  }
  rc = smoe_router_logit_grad(a->dlogits, (int)a->logits_dtype, E, outside, outside_stride, s.ds, a->scores, a->indices, T, E,
                              K, stream);
  if (rc) return rc;
  if (a->router_w != nullptr) {
    rc = smoe_gather_sum_router(s.dx_expanded, a->dx, a->s_reverse_scatter_idx, T, K, H, a->dlogits, E, a->router_w, stream);
    if (rc) return rc;
  }
  if (a->router_chunks == 0) return rc;
  if (a->router_chunks == 1) return smoe_router_weight_grad(a->dlogits, a->x, a->dwr, T, E, H, 1, stream);
  rc = smoe_router_weight_grad(a->dlogits, a->x, s.partial, T, E, H, (int)a->router_chunks, stream);
  if (rc) return rc;
  return smoe_sum_chunks(s.partial, (int)a->router_chunks, (int64_t)E * H, a->dwr, stream);
}
