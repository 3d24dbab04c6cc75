// Products with rows that no float4 fits: the loaders that need 4-byte alignment only. A row-major B takes any tile
// shape (its columns are few as often as they are many), a transposed one those of small and middling
// products.
#include "gemm_host.h"

using namespace tfhip;

int tfhip::launch_ragged_gemm(GemmParams &p, bool transpose_b) {
  if (!transpose_b) return launch_gemm_shape<kLoadKAny, kLoadXVec>(choose_tile_shape(p.M, p.N, p.K, p.batch, num_cus()), p);
  static const int shapes[] = {9, 11, 12};
  int best = shapes[0];
  double best_us = 0;
  for (const int s : shapes) {
    const double us = estimate_us(kTileShapes[s], p.M, p.N, p.K, p.batch, num_cus());
    if (s == shapes[0] || us < best_us) {
      best_us = us;
      best = s;
    }
  }
  if (best == 9) return launch_gemm<64, 64, 32, 2, 2, kLoadKAny, kLoadKAny>(p);
  if (best == 11) return launch_gemm<32, 64, 32, 2, 2, kLoadKAny, kLoadKAny>(p);
  return launch_gemm<32, 32, 32, 2, 2, kLoadKAny, kLoadKAny>(p);
}
