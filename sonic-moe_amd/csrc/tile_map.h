// The list of token tiles that the grouped GEMMs walk, and the order of the experts that the weight-gradient streams walk.
#pragma once
#include "common.h"

namespace smoe {

// ---- tile map ------------------------------------------------------------------------------------------------
// Built on the device from the expert offsets; header[0] = number of token tiles.  Entry i = (expert, first row) and
// the group of token tiles entry i belongs to: the token tiles of an expert are cut into groups of nearly equal height
// (at most gemm_group_tiles), and a group's tiles are walked feature tile by feature tile, so that the workgroups of an
// XCD that run at the same time share few operand panels.  group[i] = first entry of the group | height << 24 |
// (sweep direction) << 31.
struct TileMap {
  int32_t* header;  // [4]
  int32_t* expert;  // [max_tiles]
  int32_t* row0;    // [max_tiles]
  int32_t* group;   // [max_tiles]
};
constexpr int TILE_GROUP_MAX = 127;  // 7 bits of height

static inline int64_t max_token_tiles(int64_t TK, int E, int BM) { return TK / BM + E; }

static inline size_t tile_map_bytes(int64_t TK, int E) {
  // sized for the smallest token tile any kernel uses (64 rows)
  return (size_t)(4 + 3 * max_token_tiles(TK, E, 64)) * sizeof(int32_t);
}

static inline TileMap carve_tile_map(void* ws, int64_t TK, int E, int BM) {
  TileMap t;
  t.header = (int32_t*)ws;
  t.expert = t.header + 4;
  t.row0 = t.expert + max_token_tiles(TK, E, BM);
  t.group = t.row0 + max_token_tiles(TK, E, BM);
  return t;
}

// the maps of one routing for tiles of 256 and of 128 rows
struct TileMapPair {
  TileMap map[2];
  int gmax, snake;
};
SMOE_DEV int tile_map_rows(int which) { return which == 0 ? 256 : 128; }

// One workgroup of WAVES wavefronts writes one map; part: 2 * WAVES words of LDS.  SCAN: counts are the experts' row counts,
// whose sums it forms itself, experts listed 0, 1, ...; otherwise off, and with an order, position i of the list holds
// expert order[i].
template <int WAVES, bool SCAN>
SMOE_DEV void write_tile_map(const int32_t* __restrict__ counts, const int32_t* __restrict__ off,
                             const int32_t* __restrict__ order, int E, int BM, int gmax, int snake, const TileMap& tm,
                             int32_t* part) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int32_t base = 0, row_base = 0;
  for (int e0 = 0; e0 < E; e0 += 64 * WAVES) {
    int e = e0 + tid;
    int32_t lo = 0, cnt = 0;
    if (e < E) {
      if constexpr (SCAN) {
        cnt = counts[e];
      } else {
        if (order != nullptr) e = order[e];
        lo = off[e];
        cnt = off[e + 1] - lo;
      }
    }
    const int32_t tiles = (cnt + BM - 1) / BM;
    int32_t v = tiles, rows = cnt;
    for (int d = 1; d < 64; d <<= 1) {
      const int32_t o = __shfl_up(v, d, 64);
      if (lane >= d) v += o;
      if constexpr (SCAN) {
        const int32_t r = __shfl_up(rows, d, 64);
        if (lane >= d) rows += r;
      }
    }
    __syncthreads();  // part is used again
    if (lane == 63) {
      part[wave] = v;
      if constexpr (SCAN) part[WAVES + wave] = rows;
    }
    __syncthreads();
    int32_t wbase = 0, tot = 0, wrows = 0, tot_rows = 0;
    for (int w = 0; w < WAVES; w++) {
      if (w < wave) wbase += part[w];
      tot += part[w];
      if constexpr (SCAN) {
        if (w < wave) wrows += part[WAVES + w];
        tot_rows += part[WAVES + w];
      }
    }
    const int32_t start = base + wbase + v - tiles;
    if constexpr (SCAN) lo = row_base + wrows + rows - cnt;
    // groups of nearly equal height: the first `taller` of them have one token tile more
    const int32_t ngroups = (tiles + gmax - 1) / gmax;
    const int32_t hbase = ngroups ? tiles / ngroups : 0, taller = ngroups ? tiles % ngroups : 0;
    const int32_t split = taller * (hbase + 1);
    for (int32_t i = 0; i < tiles; i++) {
      tm.expert[start + i] = e;
      tm.row0[start + i] = lo + i * BM;
      int32_t g, first, h;
      if (i < split) {
        h = hbase + 1;
        g = i / h;
        first = g * h;
      } else {
        h = hbase;
        g = (i - split) / h;
        first = split + g * h;
        g += taller;
      }
      tm.group[start + i] = (int32_t)((uint32_t)(start + first) | (uint32_t)h << 24 | (uint32_t)(snake & g & 1) << 31);
    }
    base += tot;
    row_base += tot_rows;
  }
  if (tid == 0) tm.header[0] = base;
}

// The experts by their row counts, largest first, equal ones by number (or in the caller's order), by one workgroup of 1024;
// cost: E words of LDS.  Every expert counts the ones before it, E steps for each 1024 experts: up to TILE_SORT_MAX_E that is
// done beside the maps in their launch.  E = 128: 5.6 us for the two maps and the order, 4.6 + 5.9 as two launches.
constexpr int TILE_SORT_MAX_E = 256;
SMOE_DEV void sort_experts(const int32_t* __restrict__ off, const int32_t* __restrict__ order, int E,
                           int32_t* __restrict__ sorted, int32_t* cost) {
  const int tid = threadIdx.x;
  for (int e = tid; e < E; e += 1024) cost[e] = off[e + 1] - off[e];
  __syncthreads();
  for (int e = tid; e < E; e += 1024) {
    if (order != nullptr) {
      sorted[e] = order[e];
    } else {
      int pos = 0;
      const int c = cost[e];
#pragma unroll 8
      for (int o = 0; o < E; o++) pos += (cost[o] > c || (cost[o] == c && o < e)) ? 1 : 0;
      sorted[pos] = e;
    }
  }
}

}  // namespace smoe
