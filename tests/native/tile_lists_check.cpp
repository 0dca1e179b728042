// CPU check of the tile lists of W and W^T (coarse_schedule.cpp): each tile
// row lists exactly the tiles in the reach of the columns, ascending, its
// diagonal tile among them, and -1 behind them.
// Usage: tile_lists_check n bw planes
#include <cstdio>
#include <cstdlib>
#include <set>

#include "../../topopt-in-openmp-gpu_amd/csrc/coarse_schedule.hpp"

using namespace t3d;

int main(int argc, char **argv) {
  if (argc < 4) return 2;
  CoarseSchedule cs;
  if (!build_coarse_schedule(std::atoi(argv[1]), std::atoi(argv[2]), std::atoi(argv[3]), cs))
    return 1;
  const int nb = cs.nblk, st = cs.list_stride;
  if (st < nb + 1 || (int)cs.wlist.size() != nb * st || (int)cs.wtlist.size() != nb * st) return 1;
  std::set<std::pair<int, int>> nz, got[2];
  for (int J = 0; J < nb; J++) {
    nz.insert({J, J});
    for (int q = 0; q < cs.colinfo[2 * J + 1]; q++)
      nz.insert({cs.rows[4 * (cs.colinfo[2 * J] + q)], J});
  }
  for (int t = 0; t < 2; t++)
    for (int R = 0; R < nb; R++) {
      const int *l = (t ? cs.wtlist.data() : cs.wlist.data()) + (size_t)R * st;
      for (int q = 1; q < st; q++) {
        if (q > l[0] ? l[q] != -1 : (l[q] < 0 || (q > 1 && l[q] <= l[q - 1]))) return 1;
        if (q <= l[0]) got[t].insert(t ? std::make_pair(l[q], R) : std::make_pair(R, l[q]));
      }
    }
  if (got[0] != nz || got[1] != nz) return 1;
  std::printf("OK tiles %d nonzero %zu\n", nb, nz.size());
  return 0;
}
