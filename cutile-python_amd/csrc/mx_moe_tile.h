// Interface of the mixture-of-experts layer at medium sizes (mx_moe_tile.hip): experts of some 24 to 128 rows each.
#pragma once
#include "mx_common.h"

namespace mx {

constexpr int kMoeTileCols = 128;   // of a workgroup, 64 or 128 rows high; the up projection's are 64 of the gate and 64 of the up half
constexpr int kMoeTileMaxIds = 16384, kMoeTileMaxExperts = 1024;

// One row tile of an expert: written by moe_tiles_kernel for every tile of the worst routing (rows == 0: not in use).
struct MoeTile {
  int32_t expert, rows;     // rows of the expert from this tile on
  int32_t run, run_tiles;   // the expert's first tile and its number of tiles
};
inline int64_t moe_tiles_max(int64_t num_ids, int64_t experts, int tile_rows) {
  const int64_t used = experts < num_ids ? experts : num_ids;
  return (num_ids + used * (tile_rows - 1)) / tile_rows;
}
// tiles[max_tiles], slots[max_tiles * tile_rows]: the routed copies of every expert, in tiles of their own (entries behind
// an expert's last copy are not written)
int launch_moe_tiles(const void* ids, int ids64, int64_t num_ids, int num_experts, int tile_rows, MoeTile* tiles, int32_t* slots, int64_t max_tiles,
                     hipStream_t stream);

struct MoeTileArgs {
  const uint8_t* X; const uint8_t* Xs; const uint8_t* W; const uint8_t* Ws;   // Ws: MX_SCALE_NATIVE
  const MoeTile* tiles; const int32_t* slots;
  uint8_t* q; uint8_t* qs;             // up: activation [copy][F] and its scales [copy][F / 32]
  float* C; int64_t c_split;           // down: fp32 partial products [split][copy][N], elements from split to split
  int64_t ldx, ldxs, ldw, w_es, ws_es; // bytes; *_es: between experts
  int32_t x_rows, N, K, F;             // N: rows of an expert's W (up: 2 F)
  int32_t n_ids, E, max_tiles, tile_rows, replicas;         // a routed copy `id` reads row id / replicas of X
  int32_t w_fmt, scale_mode, splits;   // ranges of K (down)
};
int moe_tile_rows(int64_t num_ids, int64_t experts, int64_t H, int w_fmt);
int moe_tile_splits(int64_t num_ids, int64_t experts, int tile_rows, int64_t N, int64_t K);
int launch_moe_tile(const MoeTileArgs& a, bool up, hipStream_t stream);

}  // namespace mx
