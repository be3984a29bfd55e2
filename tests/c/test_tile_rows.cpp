// Host check of the row store of a full tile (store_rows_full in ptq2_device.h): for every row count and first
// plane that the kernels use, every lane reads its row's value, and no lane, storing or not, reads past the
// tile's 3 TCS values.
#include <cstdio>

#include "ptq2_device.h"

using namespace ptq2;

template <int ROWS>
static int check(int z0) {
  int bad = 0;
  for (int lane = 0; lane < BEL; lane++) {
    const FastLane L = fast_lane(Box{}, lane);
    for (int it = 0; it < (ROWS + 1) / 2; it++) {
      const int o = TPS * z0 + fast_loff<ROWS>(L, it);
      if (o < 0 || o >= 3 * TCS) bad++;
      const int r = 2 * it + L.p;
      if (L.p > 1 || r >= ROWS) continue;
      if (o != L.c * TCS + tx(L.ii) + TRS * (r % TN) + TPS * (z0 + r / TN)) bad++;
    }
  }
  if (bad) std::printf("%d rows from plane %d: %d bad offsets\n", ROWS, z0, bad);
  return bad;
}

int main() {
  int bad = check<2 * BE * TN>(0) + check<TN>(2 * BE) + check<WPLANES * TN>(0) + check<WPLANES * TN>(WPLANES) +
            check<2 * TN>(2 * WPLANES);
  for (int z = 0; z < TN; z++) bad += check<TN>(z);
  if (bad) return 1;
  std::printf("tile rows ok\n");
  return 0;
}
