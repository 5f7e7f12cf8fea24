// Host check of the interface nodes' places (hirensi_amd/csrc/hr_split.h): every node
// of the regular-domain box that a PML element holds has a place of its own below the
// count, and none is left over.
#include <cstdio>
#include <initializer_list>
#include <vector>
#include "../../hirensi_amd/csrc/hr_split.h"

int main() {
  using namespace hr;
  long checked = 0;
  for (int ex : {1, 2, 3, 7})
    for (int ey : {1, 2, 5})
      for (int ez : {1, 2, 4}) {
        const int lo[3] = {2, 1, 3}, hi[3] = {2 + ex, 1 + ey, 3 + ez};      // one PML layer above in x, y
        const int bn[3] = {2 * ex + 1, 2 * ey + 1, 2 * ez + 1};
        std::vector<int> seen(sp_iface_count(bn[0], bn[1], bn[2]), 0);
        for (int k = 0; k < 2 * hi[2] + 1; ++k)
          for (int j = 0; j < 2 * hi[1] + 3; ++j)
            for (int i = 0; i < 2 * hi[0] + 3; ++i) {
              const SpAxis X = sp_axis(i, hi[0] + 1, lo[0], hi[0]), Y = sp_axis(j, hi[1] + 1, lo[1], hi[1]),
                           Z = sp_axis(k, hi[2], lo[2], hi[2]);
              const bool pml = !(i > 2 * lo[0] && i < 2 * hi[0] && j > 2 * lo[1] && j < 2 * hi[1] && k > 2 * lo[2]);
              if (!pml || !sp_iface(X, Y, Z)) continue;
              const unsigned q = sp_iface_column(i - 2 * lo[0], j - 2 * lo[1], bn[0], bn[1], bn[2]) +
                                 sp_rim(bn[0], bn[1]) * (unsigned)(k - 2 * lo[2]);
              if (q >= seen.size() || seen[q]++) { std::printf("node %d %d %d: place %u\n", i, j, k, q); return 1; }
              ++checked;
            }
        for (int s : seen)
          if (s != 1) { std::printf("%d x %d x %d: places left over\n", ex, ey, ez); return 1; }
      }
  std::printf("interface nodes %ld\n", checked);
  return checked > 0 ? 0 : 1;
}
