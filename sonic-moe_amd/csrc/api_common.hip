// Library-wide pieces of the C ABI: version, thread-local error text, and the tile-map builder that turns the
// expert offsets into a list of token tiles on the device (no host synchronisation anywhere on the hot path).
#include <stdarg.h>
#include <stdlib.h>
#include <string.h>

#include <mutex>

#include "gemm_common.h"

namespace smoe {

static thread_local char g_error[512] = "";

void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_error, sizeof(g_error), fmt, ap);
  va_end(ap);
}

namespace {
std::once_flag g_tuning_once;
Tuning g_tuning = {1, 0, 2, 1, 1, 8, 1, 1, -1, 16};

struct Knob {
  const char* name;
  const char* env;
  int Tuning::*field;
  int lo, hi, def;
};
const Knob g_knobs[] = {
    {"gemm_stream", "SMOE_GEMM_STREAM", &Tuning::gemm_stream, 0, 1, 1},
    {"gemm_stream_grid", "SMOE_GEMM_STREAM_GRID", &Tuning::gemm_stream_grid, 0, 1 << 30, 0},
    {"varlen_k_tile_order", "SMOE_VARLEN_K_TILE_ORDER", &Tuning::varlen_k_tile_order, 0, 2, 2},
    {"dz_stream", "SMOE_DZ_STREAM", &Tuning::dz_stream, 0, 1, 1},
    {"gemm_asm", "SMOE_GEMM_ASM", &Tuning::gemm_asm, 0, 1, 1},
    {"gemm_group_tiles", "SMOE_GEMM_GROUP_TILES", &Tuning::gemm_group_tiles, 1, TILE_GROUP_MAX, 8},
    {"gemm_group_snake", "SMOE_GEMM_GROUP_SNAKE", &Tuning::gemm_group_snake, 0, 1, 1},
    {"gemm_small_tiles", "SMOE_GEMM_SMALL_TILES", &Tuning::gemm_small_tiles, 0, 2, 1},
    {"varlen_k_stream_rows", "SMOE_VARLEN_K_STREAM_ROWS", &Tuning::varlen_k_stream_rows, 0, 1 << 30, -1},
    {"gemm_skinny_rows", "SMOE_GEMM_SKINNY_ROWS", &Tuning::gemm_skinny_rows, 0, 1 << 20, 16},
};

void read_tuning_env() {
  for (const Knob& k : g_knobs) {
    const char* v = getenv(k.env);
    if (v == nullptr || *v == 0) continue;
    const long x = strtol(v, nullptr, 10);
    g_tuning.*(k.field) = x < k.lo || x > k.hi ? k.def : (int)x;
  }
}
}  // namespace

const Tuning& tuning() {
  std::call_once(g_tuning_once, read_tuning_env);
  return g_tuning;
}

int device_compute_units(int* out) {
  static int cus[64] = {};
  int dev = 0;
  SMOE_HIP_CHECK(hipGetDevice(&dev));
  if (dev < 0 || dev >= 64 || cus[dev] == 0) {
    int n = 0;
    SMOE_HIP_CHECK(hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev));
    if (dev < 0 || dev >= 64) {
      *out = n;
      return SMOE_OK;
    }
    cus[dev] = n;
  }
  *out = cus[dev];
  return SMOE_OK;
}

// workgroup 0 and, with a pair, 1: the maps; 2: the experts' order
__global__ __launch_bounds__(1024) void build_tile_map_kernel(const int32_t* __restrict__ off,
                                                              const int32_t* __restrict__ order, int E, int BM,
                                                              const TileMapPair maps, int32_t* __restrict__ sorted) {
  __shared__ int32_t lds[TILE_SORT_MAX_E];
  static_assert(TILE_SORT_MAX_E >= 32, "write_tile_map's words");
  const int which = blockIdx.x;
  if (which == 2) {
    sort_experts(off, order, E, sorted, lds);
    return;
  }
  write_tile_map<16, false>(nullptr, off, order, E, which == 0 ? BM : tile_map_rows(1), maps.gmax, maps.snake,
                            which == 0 ? maps.map[0] : maps.map[1], lds);
}

int launch_build_tile_map(const int32_t* off, const int32_t* order, int E, int BM, TileMap tm, hipStream_t st,
                          const TileMapPair* pair, int32_t* sorted) {
  const TileMapPair one = {{tm, tm}, tuning().gemm_group_tiles, tuning().gemm_group_snake};
  const int grid = pair == nullptr ? 1 : sorted == nullptr ? 2 : 3;
  hipLaunchKernelGGL(build_tile_map_kernel, dim3(grid), dim3(1024), 0, st, off, order, E, BM,
                     pair ? *pair : one, sorted);
  SMOE_LAUNCH_CHECK();
  return SMOE_OK;
}

}  // namespace smoe

extern "C" int smoe_version(void) { return 310; }
extern "C" const char* smoe_last_error(void) { return smoe::g_error; }

extern "C" int smoe_set_tuning(const char* name, int value) {
  SMOE_REQUIRE(name != nullptr, SMOE_ERR_INVALID, "set_tuning: null name");
  smoe::tuning();  // the environment is read first, so that it cannot overwrite this call later
  for (const smoe::Knob& k : smoe::g_knobs) {
    if (strcmp(name, k.name) != 0) continue;
    if (value < 0) value = k.def;
    SMOE_REQUIRE(value == k.def || (value >= k.lo && value <= k.hi), SMOE_ERR_INVALID, "set_tuning: %s = %d outside [%d, %d]",
                 name, value, k.lo, k.hi);
    smoe::g_tuning.*(k.field) = value;
    return SMOE_OK;
  }
  smoe::set_error("set_tuning: unknown knob '%s'", name);
  return SMOE_ERR_INVALID;
}
