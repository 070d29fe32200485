// Which tile of the expert GEMM pipeline, and which of its K steps, a workgroup takes: moe_pipe.hip on the GPU, and the host where the
// rule is checked.
//
// Each XCD runs its tiles in rounds of one per CU.  The tiles past the last whole round are cut over K where that pays: every
// piece leaves its fp32 sums in a workspace, and the one that finishes last -- a counter, nobody waits -- adds them in the order of the pieces.
#pragma once
#include <hip/hip_runtime.h>

namespace dsse {
namespace moe_cut {

constexpr int kCUs = 32;      // per XCD
constexpr int kMostCut = 8;   // pieces of a tile
constexpr int kPieces = 16;   // pieces per XCD
constexpr int kCutTiles = 4;  // cut tiles per XCD
constexpr int kLeast = 2;     // K steps of a piece: the pipeline's last two are always run

struct Cut {
  int left, pieces;  // most tiles past the last whole round that are cut, pieces of each
};

// steps_r, steps_s: K steps of a routed and of a shared tile (steps_r where there is none); forced: 0, or pieces by force (1: no tile is cut).
// Pieces pay where they are few -- tiles of a round that is half empty run faster than those of a full one -- and long, and where no
// shared expert's longer walk is what the launch waits for (down products).  Without / with, one MI355X, work list and both products, us, mean of six random
// choices: 16 experts, top 2 and a shared one, 2048 x 1408, 1024 rows (264 tiles, one left per XCD) 164 / 154; 4096 x 3584, 1300 rows 553 / 526, 1500
// 592 / 568, 3000 1017 / 1005; 200 and 700 rows, whose experts' tiles are not left over, 311 and 405 in both.  With more than these left it turns (forced): 2048 x
// 1408, three or four tiles left, 1100 rows 151 / 154, five to eight 1300 rows 154 / 163, 1500 165 / 170; 16 K steps, 1024 x 2048, 2500 rows 174 / 178.
__host__ __device__ inline Cut most_cut(int steps_r, int steps_s, int forced) {
  if (forced) {
    const int fit = (steps_r < steps_s ? steps_r : steps_s) / kLeast;
    return Cut{kCutTiles, forced < fit ? forced : fit};
  }
  const int left = steps_r / 16 < kCutTiles ? steps_r / 16 : kCutTiles;
  return Cut{steps_r < 32 || steps_s > steps_r ? 0 : left, kMostCut};
}

// Workgroups per XCD beyond one for each tile
__host__ __device__ inline int pieces_room(Cut most) { return most.left > 0 && most.pieces > 1 ? kPieces : 0; }

struct Item {
  int u;          // the tile, or the count of them: none
  int piece, of;  // its piece
  int whole;      // tiles before the first cut one
};

// Workgroup `item` of an XCD with `tiles` tiles
__host__ __device__ inline Item item_of(int item, int tiles, Cut most) {
  const int left = tiles % kCUs;
  const int fit = left ? kPieces / left : 1, cut = left < 1 || left > most.left ? 1 : most.pieces < fit ? most.pieces : fit;
  const int whole = cut > 1 ? tiles - left : tiles;
  if (item < whole) return Item{item, 0, 1, whole};
  const int u = whole + (item - whole) / cut;
  return u < tiles ? Item{u, (item - whole) % cut, cut, whole} : Item{tiles, 0, 1, whole};
}

// Tile `at` of an expert of T row tiles and nb column blocks: groups of 8 row tiles swept column by column
struct Spot {
  int row_tile, block;
};
__host__ __device__ inline Spot spot_of(int at, int T, int nb) {
  const int grp = at / (8 * nb), gsz = T - 8 * grp < 8 ? T - 8 * grp : 8, in = at - grp * 8 * nb;
  return Spot{8 * grp + in % gsz, in / gsz};
}

// Whether a tile of kn K steps is cut.  The last tiles of an XCD may be a shared expert's, whose walk may be short.  And a routed tile is cut only with
// all T row tiles of its column block: which of them holds a row is up to the atomics that made the work list, so where one had another order of sums, the
// same call would not give the same bits again.  (A shared expert's rows are in order.)  ns, tiles: the XCD's shared tiles, all of its tiles.
__host__ __device__ inline bool cuts(const Item& it, int kn, int ns, int tiles, int row_tile, int T) {
  if (it.of == 1 || kn < kLeast * it.of) return false;
  const int block = it.u - row_tile;  // the block's first tile: T <= 8 follow each other, and no more than kCutTiles are cut
  return it.u < ns || (block >= it.whole && block >= ns && block + T <= tiles);
}

struct Walk {
  int first, steps;
};

// K steps of piece `piece` of `of`, of the walk [k0, k0 + kn)
__host__ __device__ inline Walk walk_of(int k0, int kn, int piece, int of) {
  const int first = kn * piece / of;
  return Walk{k0 + first, kn * (piece + 1) / of - first};
}

}  // namespace moe_cut
}  // namespace dsse
