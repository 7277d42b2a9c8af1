// Pieces shared by the persistent ping-pong GEMM kernels (mx_gemm_pp.hip: 16x16x128 MFMA tiles, all element
// formats; mx_gemm_pp32.hip: 32x32x64 MFMA tiles, 8-bit formats): LDS budget, tile walk, launch helpers.
#pragma once
#include "mx_gemm_tile.h"

namespace mx {

// s_waitcnt immediate that waits for vmcnt <= n only (gfx9 encoding: vmcnt in bits 3:0 and 15:14)
constexpr int vmcnt_imm(int n) { return 0x0F70 | (n & 15) | ((n >> 4) << 14); }

template <class C>
struct PP {
  static_assert((C::BM == 256 || C::BM == 192) && C::BN == 256, "ping-pong kernel is 256 (192) x 256");
  static constexpr int A_BUFS = 3, B_BUFS = 2;
  static constexpr int B_BASE = A_BUFS * C::A_STAGE;
  static constexpr int LDS_BYTES = B_BASE + B_BUFS * C::B_STAGE;
  static constexpr int A_RPI = 64 / C::A_CPR, B_RPI = 64 / C::B_CPR;   // rows per DMA instruction
  static constexpr int AL = C::WTM / A_RPI / 4;              // A loads per wave and stage
  static constexpr int BL = 64 / B_RPI;                     // B loads per team-1 wave and stage
  static_assert(LDS_BYTES <= 160 * 1024, "LDS budget");
};

// Tiles a workgroup walks: linear tile ids first, first + step, ... below end, then possibly (the ping-pong kernel with room
// for partial sums) some K-quads of one more tile, `tail`.  Linear ids map to (tile row, tile column) in groups of 4
// tile rows walked column by column (the 32 tiles an XCD works on at a time are 4 tile rows x 8 tile columns, which
// its L2 serves).
constexpr int kNoTile = 0x7FFFFFFF;
struct TileWalk {
  int first, step, end, tiles_m, tiles_n;
  int tail = kNoTile;
  int quads = 0;   // of the tail: first K-quad | number << 16
  template <int ROWS = 256>   // of a tile
  __device__ void origin(int lid, int& m0, int& n0) const {
    constexpr int GM = 4;   // measured: 4 rows is 1 - 3 % faster than 8 (2, 3, 6, 16 are slower than either)
    const int in_group = GM * tiles_n;
    const int gid = lid / in_group, first_m = gid * GM;
    const int gsz = (tiles_m - first_m) < GM ? (tiles_m - first_m) : GM;
    const int in = lid % in_group;
    m0 = (first_m + in % gsz) * ROWS;
    n0 = (in / gsz) * 256;
  }
  // the walk including the tail tile: kNoTile after the last one
  __device__ int head() const { return first < end ? first : tail; }
  __device__ int next(int lid) const { return lid >= end ? kNoTile : lid + step < end ? lid + step : tail; }
};

// The same for a grouped product: groups of tile rows that don't cross from one expert to the next, so that the rows walked
// together share their W tiles (a group of 4 over two experts reads twice the W for the same work: 8192 slots of 8 experts,
// 4 or 5 tile rows each, 28672 x 4096 MXFP8: 873 -> 838 us, 4096 x 14336: 416 -> 402 us).  An expert's tile rows are cut
// into groups of nearly 4: 5 stay together, 6 are 3 + 3.  The 64 lanes look at 64 tile rows at a time (an expert is cut where
// they end): bit i of `first` is set if tile row 64 * chunk + i begins an expert.
struct ExpertRuns {
  const int32_t* ids;   // of each tile_m slots
  int tile_m, tiles_m, tiles_n;
  int chunk = -1;
  uint64_t first = 0;
  __device__ void origin(int lid, int& m0, int& n0) {   // (all lanes of the wave)
    int tiles_n = this->tiles_n;
    asm volatile("" : "+s"(tiles_n));   // (no reciprocal of it is kept in registers from one tile to the next)
    const int row = lid / tiles_n, bit = row & 63;
    if ((row >> 6) != chunk) {
      chunk = row >> 6;
      const int lane = __lane_id(), at = chunk * 64 + lane;
      const int e = at < tiles_m ? ids[(int64_t)at * 256 / tile_m] : -1;
      const int before = __builtin_amdgcn_ds_bpermute((lane + 63 & 63) * 4, e);
      first = __builtin_amdgcn_ballot_w64(lane == 0 || at == tiles_m || e != before);
    }
    const int begin = 63 - __builtin_clzll(first & (~0ull >> (63 - bit)));
    const uint64_t above = first >> bit >> 1;
    const int end = above ? bit + 1 + __builtin_ctzll(above) : tiles_m - chunk * 64 < 64 ? tiles_m - chunk * 64 : 64;
    const int count = end - begin, parts = count < 3 ? 1 : (count + 2) >> 2, size = (count + parts - 1) / parts;
    const int g0 = begin + (bit - begin) / size * size, rows = size < end - g0 ? size : end - g0;
    const int in = lid - (chunk * 64 + g0) * tiles_n;
    m0 = (chunk * 64 + g0 + in % rows) * 256;
    n0 = in / rows * 256;
  }
};

// XCD x (workgroup ids are dealt round-robin to the 8 XCDs, each with its own L2) owns a contiguous range of the linear
// tile ids: [start, start + count), which its `wgs` workgroups walk with a stride of their count.
struct XcdShare { int start, count, wgs; };
__device__ inline XcdShare xcd_share(int total, int grid, int xcd) {
  const int per = total >> 3, rem = total & 7;
  return {xcd * per + (xcd < rem ? xcd : rem), per + (xcd < rem ? 1 : 0), (grid - xcd + 7) >> 3};
}

// Ways a tile of the last, partly filled round of an XCD is split along K (1: not).  A K-quad takes a workgroup 5.8 us with
// 8-bit operands, 3.6 us with FP4 ones; against that stand a launch that adds the partial sums up (6 us) and 256 KiB per
// workgroup written and read again (22 us when every workgroup has some: 1531 x 14336 x 4096, 80 tiles three ways,
// 46 us of stages saved 31 and cost 27).  The cheapest number of ways that the XCD's workgroups allow is taken if it
// gains 5 us or more.  In whole tenths of a us, so that the kernel and the launch behind it agree.
constexpr int kTailMax = 16;   // split tiles per XCD
__host__ __device__ inline int tail_tenths(int S, int rest, int wgs, int KQ, bool fp4) {
  const int quad = fp4 ? 36 : 58;
  return S == 1 ? KQ * quad : (KQ + S - 1) / S * quad + 60 + 220 * rest * S / wgs;
}
__host__ __device__ inline int tail_splits(int rest, int wgs, int KQ, bool fp4) {
  if (rest <= 0 || rest > kTailMax) return 1;
  int best = tail_tenths(1, rest, wgs, KQ, fp4) - 50, S = 1;
  for (int s = 2; s <= 8 && s <= KQ && s * rest <= wgs; ++s) {
    const int c = tail_tenths(s, rest, wgs, KQ, fp4);
    if (c <= best) { best = c; S = s; }
  }
  return S;
}

__device__ inline TileWalk make_tile_walk(int M, int N, int rows = 256) {
  TileWalk walk;
  walk.tiles_m = (M + rows - 1) / rows;
  walk.tiles_n = (N + 255) / 256;
  const XcdShare x = xcd_share(walk.tiles_m * walk.tiles_n, gridDim.x, blockIdx.x & 7);
  walk.step = x.wgs;
  walk.first = x.start + (blockIdx.x >> 3);
  walk.end = x.start + x.count;
  return walk;
}

// the same with the last round's tiles split along K where that pays
__device__ inline TileWalk make_split_walk(int M, int N, int KQ, bool fp4) {
  TileWalk walk = make_tile_walk(M, N);
  const XcdShare x = xcd_share(walk.tiles_m * walk.tiles_n, gridDim.x, blockIdx.x & 7);
  const int rest = x.count % x.wgs, S = tail_splits(rest, x.wgs, KQ, fp4), loc = blockIdx.x >> 3;
  if (S > 1) {
    walk.end = x.start + x.count - rest;
    if (loc < rest * S) {
      walk.tail = walk.end + loc / S;
      const int q0 = loc % S * KQ / S;
      walk.quads = q0 | ((loc % S + 1) * KQ / S - q0) << 16;
    }
  }
  return walk;
}

inline int num_cus() {
  static int cus = [] {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 256;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) return 256;
    return n;
  }();
  return cus;
}

// grid of a persistent ping-pong launch: one workgroup per CU walking several tiles when the stage pipeline can
// run across tile boundaries (at least two stages per tile, whole K-quads); otherwise one workgroup per tile
inline int64_t pp_grid(int M, int N, int K, int ksub, int rows = 256) {
  const int64_t tiles = (int64_t)((M + rows - 1) / rows) * ((N + 255) / 256);
  const int ksteps = (K + 127) / 128;
  const int nstages = (ksteps + ksub - 1) / ksub;
  const bool can_walk = nstages >= 2 && ksteps % 4 == 0;
  return (can_walk && tiles > num_cus()) ? num_cus() : tiles;
}

// Partial sums of the split last round of a ping-pong launch: one 256 x 256 fp32 tile per workgroup.  0 where no split is
// possible (a K that is not whole K-quads) or none pays: for this number of tiles, or (tiles_known false: M is an upper bound)
// for a typical one.
inline int64_t pp_tail_bytes(int64_t M, int64_t N, int64_t K, bool fp4, bool tiles_known) {
  const int64_t tiles = ((M + 255) / 256) * ((N + 255) / 256), KQ = K / 512;
  if (K % 512 != 0 || KQ >= 1 << 15 || tiles <= 0 || tiles > 0x7FFFFFFF) return 0;
  const int cus = num_cus(), w = cus / 8;
  if (w == 0) return 0;
  if (tiles_known) {   // the XCDs' shares differ by at most one tile
    const int64_t lo = tiles / 8, hi = (tiles + 7) / 8;
    if (tail_splits((int)(lo % w), w, (int)KQ, fp4) == 1 && tail_splits((int)(hi % w), w, (int)KQ, fp4) == 1) return 0;
  } else {   // a quarter of a round, as a typical one: worth the launch behind it and the extra scalars if it saves 20 us
    const int S = tail_splits(w / 4, w, (int)KQ, fp4);
    if (tail_tenths(1, w / 4, w, (int)KQ, fp4) - tail_tenths(S, w / 4, w, (int)KQ, fp4) < 200) return 0;
  }
  return (int64_t)cus * 256 * 256 * 4;
}

// the ping-pong kernels of one element-format pair (mx_gemm_pp.hip, compiled once per pair)
template <int AF, int BF>
int launch_pp_pair(const GemmArgs& g, hipStream_t stream);

}  // namespace mx
