// Elimination schedule of the coarse-level tiled Cholesky (host code, no
// device calls): the storage order of the DOFs, the workgroup tasks of every
// launch, and the non-zero tile rows of W = L^{-1}.
#pragma once

#include <string>
#include <vector>

namespace t3d {

constexpr int kTile = 64;   // tile size of the coarse factorization
constexpr int kMaxSrc = 4;  // tile columns updating one tile in one launch
constexpr int kTaskFactor = 1;

// One workgroup task: tile (I, J), I >= J, minus the updates of the tile
// columns K[0..nsrc) eliminated in this launch; kTaskFactor: the (diagonal)
// tile is complete afterwards and is factored in place.  nsrc = 0 with
// kTaskFactor factors the tile as it is.
struct CholTask {
  int I, J, nsrc, flags;
  int K[kMaxSrc];
};

struct CoarseSchedule {
  int n = 0, np = 0, nblk = 0;         // logical size, storage size (64 nblk)
  std::vector<int> pos;                // logical DOF -> storage index
  std::vector<CholTask> tasks;         // all launches, concatenated
  std::vector<int> launch_first, launch_count;
  // W = L^{-1}: tile column J has colinfo[2J+1] rows starting at row
  // colinfo[2J]; row r is (I, klist offset, klist count, klist entries of a
  // lower level than I) at rows[4r..]; klist holds the K < I of the column's
  // earlier rows with L_IK != 0, in ascending order
  std::vector<int> colinfo, rows, klist;
  // Levels of the elimination (the levels of the dissection; one for a
  // band): after launch level_launch[v] the diagonal tiles of level v are
  // factored and its rows of L written as far as the level's own columns,
  // after the next one (if any) all rows of L in its columns.  Tile column J
  // has lcolinfo[2 (v nblk + J) + 1] rows of W in level v, from row
  // lcolinfo[2 (v nblk + J)].
  int nlevels = 0;
  std::vector<int> tile_level, level_launch, lcolinfo;
  // the tiles of each tile row of W, and of W^T, that can be non-zero:
  // list_stride entries per tile row, the count, then the tile columns in
  // ascending order, then -1
  int list_stride = 0;
  std::vector<int> wlist, wtlist;
  std::string error;
};

// planes > 1 with n divisible by planes: the DOFs form `planes` consecutive
// blocks coupled only to adjacent blocks (x-planes of a grid), eliminated in
// nested-dissection order, each plane padded to whole tiles.  Otherwise the
// matrix is taken as banded (half bandwidth bw) in its own order.
bool build_coarse_schedule(int n, int bw, int planes, CoarseSchedule &out);

}  // namespace t3d
