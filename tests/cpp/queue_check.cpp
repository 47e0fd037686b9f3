// Queue places of the tracks that may become loopers (kf_queue.hpp), on the
// host: every place taken once, whatever their number; a wavefront apart where
// they fit so; with the layer navigator from two batches of the resident lanes
// on 16 to a wavefront; in one block in the largest batches.
#include <cstdio>
#include <cstdlib>
#include <initializer_list>
#include <vector>

#include "../../acts_amd/csrc/kf_queue.hpp"

using namespace kf;

int main() {
  const int64_t lanes = 65536;
  int failures = 0;
  for (bool layers : {false, true})
    for (int64_t n : {65, 100, 4096, 5000, 65536, 100000, 131072, 131073, 175000, 196608, 196609,
                      200000, 250000, 262144, 262145, 300001})
      for (int64_t nSeam : {int64_t{0}, int64_t{1}, int64_t{3}, n / 1000, n / 300, n / 100, n / 17,
                            n / 3, n - 1, n}) {
        const Spread s = spreadOf(n, lanes, layers);
        std::vector<char> taken(n, 0), wave((n + 63) / 64, 0);
        bool ok = true;
        int64_t waves = 0;
        for (int64_t i = 0; i < n && ok; ++i) {
          const int64_t at = spreadPlace(static_cast<int32_t>(i), static_cast<int32_t>(nSeam), s);
          ok = at >= 0 && at < n && !taken[at];
          if (!ok) break;
          taken[at] = 1;
          if (i < nSeam && !wave[at / 64]) {
            wave[at / 64] = 1;
            ++waves;
          }
        }
        const int64_t block = (nSeam + 63) / 64;
        if (n > 4 * lanes)
          ok = ok && waves == block;
        else if (layers && n > 2 * lanes)
          ok = ok && waves <= (nSeam + 15) / 16;
        else if (64 * nSeam <= (n < lanes ? n : lanes))
          ok = ok && waves == nSeam;
        if (!ok) {
          ++failures;
          std::printf("FAILED layers %d n %lld candidates %lld: in %lld wavefronts\n", layers,
                      static_cast<long long>(n), static_cast<long long>(nSeam),
                      static_cast<long long>(waves));
        }
      }
  if (failures == 0) std::printf("ok\n");
  return failures ? 1 : 0;
}
