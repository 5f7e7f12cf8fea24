// Host check of the displacement addresses (hirensi_amd/csrc/hr_index.h): corner and
// middle nodes of lattices around and past 2^32 / 24 nodes, where a 32-bit byte offset
// from the vector's start wraps, up to the largest lattice a context takes.
#include <cstdio>
#include <initializer_list>
#include "../../hirensi_amd/csrc/hr_index.h"

int main() {
  using namespace hr;
  const int lat[][3] = {{5, 5, 5}, {129, 129, 65}, {563, 563, 563}, {565, 565, 563}, {781, 781, 781},
                        {9765, 9765, 5}, {5, 9765, 9765}, {9765, 5, 9765}, {21, 4001, 5001}};
  long wrapped = 0, checked = 0;
  for (const auto& N : lat) {
    const long long nn = (long long)N[0] * N[1] * N[2];
    if (nn > LATTICE_NODES) { std::printf("%d x %d x %d: beyond the limit\n", N[0], N[1], N[2]); return 1; }
    for (int k : {0, 1, N[2] / 2, N[2] - 1})
      for (int j : {0, N[1] / 2, N[1] - 1})
        for (int i : {0, N[0] / 2, N[0] - 1}) {
          const long long n = i + (long long)N[0] * (j + (long long)N[1] * k);
          const long long at = 8 * plane_doubles(N[0], N[1], k) + (long long)in_plane_bytes(N[0], i, j);
          if (at != 24 * n) { std::printf("%d x %d x %d node %d %d %d: %lld\n", N[0], N[1], N[2], i, j, k, at); return 1; }
          wrapped += (long long)((unsigned)n * 24u) != 24 * n;
          ++checked;
        }
  }
  std::printf("addresses %ld, of them past 32 bits %ld\n", checked, wrapped);
  // a plane of the largest lattice of five planes, and the slots
  if (24ll * (LATTICE_NODES / 5) >= 1ll << 32 || 9 * LATTICE_NODES + 1 >= 1ll << 32) return 1;
  return wrapped > 0 ? 0 : 1;
}
