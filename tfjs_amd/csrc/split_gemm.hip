// Which products the kernel of split_gemm.h takes, with which tile, and its launch.
#include "gemm_host.h"
#include "split_gemm.h"

namespace tfhip {
namespace {

// The tiles, and what a product takes with them: `launch` microseconds, and for every compute unit's round of workgroups
// (one, or two side by side where they fit) `per_tile` for each k tile of 32 a group works through and `fixed` for the rest.
// Least squares on 3700 products and 1900 convolutions of random extents, every tile timed on each (operands in the
// caches): root mean square error 4 to 7% for products, 2% for windows, and the tile with the least estimate is on average 0.7%
// slower than the fastest. (Fitted before operands were scaled, 3% of a k tile: left as it is, since the estimate for gemm_kernel is
// low by more than that on few k tiles, where 128 x (512 x 512 x 64) takes 56 us with it and 44 here.)
struct SplitShape {
  int gw, tn, kg;
  double launch, per_tile, fixed, per_tile_two, fixed_two;   // (_two: two workgroups on a compute unit; 0: one fits)
};
constexpr SplitShape kSplitShapes[] = {
    {4, 4, 1, 2.5, 1.09, 5.2, 2.17, 6.0}, {4, 4, 2, 0.0, 1.79, 7.6, 0, 0}, {4, 3, 1, 3.3, 0.93, 3.8, 1.71, 4.6}, {4, 3, 2, 0.7, 1.42, 6.4, 0, 0},
    {4, 2, 1, 4.0, 0.77, 2.0, 1.30, 2.6}, {4, 2, 2, 1.3, 1.17, 4.9, 0, 0}, {2, 2, 4, 1.5, 1.37, 4.4, 0, 0},   {2, 1, 4, 1.9, 0.97, 3.4, 0, 0},
};
constexpr int kNumSplitShapes = sizeof(kSplitShapes) / sizeof(kSplitShapes[0]);
constexpr int kMaxSlices = 8;
constexpr int kEndWindows = 400;   // K to which tiled_end_us was fitted to windows

// Whether the knob names a tile and its slices.
bool split_forced() { return tuning(kTuneSplit) >= 0 && tuning(kTuneSplit) < 80; }

// The windows of an image cost their address arithmetic, ragged ones also what mends them.
double split_estimate_us(const SplitShape &s, const GemmParams &p, int slices, double windows) {
  const long long tiles = ((p.M + 32 * s.gw - 1) / (32 * s.gw)) * (long long)((p.N + 32 * s.tn - 1) / (32 * s.tn)) * p.batch * slices;
  const int k_tiles = ((p.K + 31) / 32 + slices - 1) / slices, rounds_of_k = (k_tiles + s.kg - 1) / s.kg;
  const long long cus = num_cus();
  const double one = rounds_of_k * s.per_tile + s.fixed, two = rounds_of_k * s.per_tile_two + s.fixed_two;
  double us;
  if (s.per_tile_two == 0) {
    us = (double)((tiles + cus - 1) / cus) * one;
  } else {
    const long long full = tiles / (2 * cus), rest = tiles % (2 * cus);
    us = (double)full * two + (rest == 0 ? 0 : (rest <= cus ? one : two));
  }
  return s.launch + us * windows + finish_us(p, slices);
}

// The fourth root of the fourth powers' sum. (With pow, 0.1 us of host time in every call that comes this far.)
double longer_of(double a, double b) { return sqrt(sqrt(a * a * a * a + b * b * b * b)); }

// What the same product takes with gemm_kernel, whatever tile and slices that chooses: the launch, the matrix instructions at
// 77% of their rate or the way of k through the pipeline, whichever is longer, and what fills and empties the chip. Least
// squares on 8800 products and 4300 convolutions of random extents, root mean square error 16%.
double tiled_estimate_us(const GemmParams &p, double windows) {
  const double blocks = (double)((p.M + 31) / 32) * ((p.N + 31) / 32) * p.batch, peak_us = blocks * 2048.0 * p.K / 155e6;
  const double pipeline_us = 0.0044 * p.K * (blocks < 256 ? pow(blocks / 256, 0.27) : 1.0);
  return 4.4 + windows * (longer_of(peak_us / 0.77, pipeline_us) + 1.4 * sqrt(peak_us));
}

// The same with a term for each tile's end, which counts for more than k where there are a few k tiles: 1200 products of random extents,
// K 16 to 6144, error 13% (20% without it), up to K = 32 1.1 to 1.4 times what it says; 750 convolutions of K 16 to 400, 13% and, ragged, 21%.
double tiled_end_us(const GemmParams &p, int a_kind, bool transposed_b) {
  static constexpr double kTerms[5][4] = {   // float4s fit both operands, they do not, a transposed B; windows, ragged windows
      {3.49, 0.94, 0.76, 0.156}, {2.74, 0.99, 1.52, 0.215}, {3.44, 1.02, 0.20, 0.229}, {4.25, 1.02, 0.54, 0.255}, {1.51, 1.21, 2.37, 0.461}};
  const int kind = a_kind == kLoadWindows ? 3 : (a_kind == kLoadWindowsAny ? 4 : (transposed_b ? 2 : (p.K % 4 == 0 && p.N % 4 == 0 ? 0 : 1)));
  const double *t = kTerms[kind];
  const double blocks = (double)((p.M + 31) / 32) * ((p.N + 31) / 32) * p.batch, peak_us = blocks * 2048.0 * p.K / 155e6;
  const double pipeline_us = 0.0044 * p.K * (blocks < 256 ? pow(blocks / 256, 0.27) : 1.0);
  const double us = t[0] + t[1] * longer_of(peak_us / 0.77, pipeline_us) + t[2] * sqrt(peak_us) + t[3] * blocks / 256;
  return p.K <= 32 && a_kind == kLoadKAny ? 1.2 * us : us;
}

// The same for products of at most 32 columns, which gemm_kernel takes in tiles of 32 x 32 and, where these are few, in up to 16 slices.
double tiled_narrow_us(const GemmParams &p, int a_kind) {
  const bool windows = a_kind != kLoadKAny, vec = windows ? a_kind == kLoadWindows : p.K % 4 == 0 && p.N % 4 == 0;
  double best = tiles_of_32_us(p, windows, vec);
  for (int slices = 2; slices <= 16 && p.K >= 256 * slices; ++slices) best = fmin(best, tiles_of_32_us(p, windows, vec, slices));
  return best;
}

template <int GW, int TN, int KG, int A_KIND, int B_KIND>
int launch_shape(GemmParams &p, int slices) {
  using T = SplitTile<GW, TN, KG>;
  p.tiles_m = (p.M + T::BM - 1) / T::BM;
  p.tiles_n = (p.N + T::BN - 1) / T::BN;
  p.splits = 1;
  p.k_per_split = p.K;
  p.ws = nullptr;
  std::unique_lock<std::mutex> held;
  const int fits = fit_fixed_scratch(p, slices, split_forced());
  if (fits != kOk) return fits;
  if (slices > 1) {
    const size_t bytes = (size_t)slices * p.batch * p.M * p.N * sizeof(float);
    held = lock_workspace();
    p.ws = bytes <= (size_t(1) << 30) ? static_cast<float *>(workspace(bytes)) : nullptr;
    if (p.ws) {
      p.splits = slices;
      p.k_per_split = ((p.K + 31) / 32 + slices - 1) / slices * 32;
    }
  }
  note_splits(p.splits);
  const long long grid = (long long)p.tiles_m * p.tiles_n * p.batch * p.splits;
  if (grid > 0x7fffffffLL) return fail(kBadArgument, "split_gemm: %lld tiles exceed the grid limit", grid);
  p.group_m = tile_rows_per_panel(grid, T::BM, T::BN, p.tiles_m);
  number_tiles(p, grid);
  const auto kernel = split_gemm<GW, TN, KG, A_KIND, B_KIND>;
  if (T::LDS_BYTES > 64 * 1024) {
    static std::atomic<int> raised{0};
    const int rc = raise_lds_limit(raised, reinterpret_cast<const void *>(kernel), T::LDS_BYTES);
    if (rc != kOk) return rc;
  }
  note_kernel("split_gemm<%d, %d, %d, %d, %d>", GW, TN, KG, A_KIND, B_KIND);
  p.inline_epilogue = p.splits == 1 && p.epi.channel_operands && p.epi.activation <= TFHIP_LEAKYRELU;
  const dim3 blocks((unsigned)grid), threads(T::kThreads);
  if (p.inline_epilogue) {
    TFHIP_LAUNCH((kernel<<<blocks, threads, T::LDS_BYTES, stream()>>>(p)));
  } else {
    TFHIP_LAUNCH((kernel<<<blocks, threads, T::LDS_BYTES, stream()>>>(p), enqueue_finish(p)));
  }
  return kOk;
}

template <int A_KIND, int B_KIND>
int launch_kind(SplitChoice c, GemmParams &p) {
  switch (c.shape) {
    case 0: return launch_shape<4, 4, 1, A_KIND, B_KIND>(p, c.slices);
    case 1: return launch_shape<4, 4, 2, A_KIND, B_KIND>(p, c.slices);
    case 2: return launch_shape<4, 3, 1, A_KIND, B_KIND>(p, c.slices);
    case 3: return launch_shape<4, 3, 2, A_KIND, B_KIND>(p, c.slices);
    case 4: return launch_shape<4, 2, 1, A_KIND, B_KIND>(p, c.slices);
    case 5: return launch_shape<4, 2, 2, A_KIND, B_KIND>(p, c.slices);
    case 6: return launch_shape<2, 2, 4, A_KIND, B_KIND>(p, c.slices);
    default: return launch_shape<2, 1, 4, A_KIND, B_KIND>(p, c.slices);
  }
}

}  // namespace

// What goes here, in this order: nothing that the offsets or the epilogue cannot hold; what the knob names; nothing below `least` FLOP or of
// few rows; of what is left the tile and slices with the least estimate, if that is 8% below the tiled kernel's (narrow: below that in tiles
// of 32 x 32); and of a few k tiles what the estimate with a tile's end leaves.
SplitChoice split_gemm_choice(const GemmParams &p, int a_kind, bool transposed_b) {
  SplitChoice best = {-1, 1, 0};
  const int forced = tuning(kTuneSplit);
  if (forced == 99 || tuning(kTuneTile) >= 0 || tuning(kTuneSplitK) >= 0 || tuning(kTuneKGroups) >= 0) return best;
  // 32-bit offsets, also of the rows behind the last one that a k tile reaches; bias and PReLU weights per column or one for all
  constexpr unsigned kMaxBytes = 0x7fffffffu;
  if (p.K <= 0 || p.a_bytes == 0 || p.a_bytes > kMaxBytes || p.b_bytes == 0 || p.b_bytes > kMaxBytes || p.N > (1 << 22) || p.c_bytes == 0 ||
      p.epi.addressing == kConv)
    return best;
  if (p.epi.channel_operands && (p.epi.bias_s[3] > 1 || p.epi.prelu_s[3] > 1)) return best;
  if (split_forced()) return {forced % 10 % kNumSplitShapes, forced / 10 + 1, 0};
  const bool narrow = forced < 0 && p.N <= 32;
  // Below 0.45 GFLOP the fixed part decides, and that of the other kernels is shorter (0.1 to 0.2 GFLOP 1.2 times slower here, of 39
  // products and convolutions of 0.3 to 0.45 1.02 times; 0.8 to 1.2 0.88 of the time, from 4 on 0.7), but for products of a few k tiles,
  // whose results are most of the work: those of K up to 128 from 0.06 GFLOP on, and windows from 0.2, go by the last lines below (1454 x 4277 x 23
  // 17 us there and 11 here; of a transposed B 32 of 200 gain and 7 lose up to 28%). So it is with tiles that
  // are mostly padding: few columns, few rows of each product of a batch. Under 448 rows only half of the products gain.
  const double flops = 2.0 * p.batch * p.M * (double)p.N * p.K;
  const bool small = forced < 0 && flops < 4.5e8;
  const double least = narrow ? 4.5e8
                              : (a_kind == kLoadKAny && !transposed_b && p.K <= 128 ? 0.6e8 : (a_kind == kLoadWindows && p.K <= kEndWindows ? 2e8 : 4.5e8));
  if (forced < 0 && (flops < least || p.M < 64 || (long long)p.batch * p.M < 448)) return best;
  // 17 to 32 columns are one strip of the 64 x 32 tile. Of 520 such products and convolutions (K 200 to 12500) 187 are taken, on average at
  // 0.85 (products) and 0.77 (windows) of the time, two of them 3 and 5% slower; us, before and here: 3982 x 25 x 8604 40.6 and 28.8,
  // 14871 x 28 x 2168 33.1 and 24.6, [2,29,116,200] 5x5 -> 21 64.7 and 38.8. Few rows mean slices, of which gemm_kernel has more
  // (1232 x 31 x 8036 windows 24.6 and 26.6); up to 16 columns it has a tile of 256 x 16 (53900 x 8 x 774 windows 49.4 and 50.6).
  if (narrow && (p.N <= 16 || transposed_b || (long long)p.batch * p.M < 1536)) return best;
  const double windows = a_kind == kLoadWindows ? 1.08 : (a_kind == kLoadWindowsAny ? 1.35 : 1.0);
  double best_us = 0;
  // (Of a fixed scratch the slices that it holds, with the tile that suits those: 536 x 1768 x 13978 takes 164 us in seven, 242 in the
  // four that fit with the same tile and 165 as it is chosen; 1500 x 1024 x 6000 107.)
  const size_t slice_bytes = (size_t)p.batch * p.M * p.N * sizeof(float);
  for (int i = narrow ? kNumSplitShapes - 1 : 0; i < kNumSplitShapes; ++i) {
    for (int slices = 1; slices <= kMaxSlices; ++slices) {
      if (slices > 1 && workspace_is_fixed() && slices * slice_bytes > fixed_workspace_bytes()) break;
      if (slices > 1 && p.K < 32 * 4 * kSplitShapes[i].kg * slices) break;
      const double us = split_estimate_us(kSplitShapes[i], p, slices, windows);
      if (best.shape < 0 || us < best_us * (slices > 1 ? 0.97 : 1.0)) {
        best_us = us;
        best = {i, slices, us};
      }
    }
  }
  // The lead that makes up for the estimates' errors: of the 13000, half are taken, on average at 0.78 of the time; 2% of
  // those are 5% slower than with gemm_kernel and more.
  // gemm_kernel is faster on a transposed B than on a row-major one (from K = 129 on 0.86 of its estimate): of 400 such products, with
  // the estimate as it is, 28 took 3 to 27% longer here than there, with 0.9 of it nine.
  const double tiled = narrow ? tiled_narrow_us(p, a_kind)
                              : tiled_estimate_us(p, a_kind == kLoadWindows ? 1.24 : (a_kind == kLoadWindowsAny ? 1.82 : 1.0)) *
                                    (transposed_b && p.K > 128 ? 0.9 : 1.0);
  if (forced >= 0 || (!small && best_us <= 0.92 * tiled)) return best;
  // What that line leaves, by the estimate that knows of a tile's end: 5300 of 7600 products of K 8 to 1024 and 0.06 to 10 GFLOP at 0.77
  // of the time, 500 of 1500 windows of K up to 400 at 0.74, but not:
  //  * what gemm_kernel has tiles of 64 x 64 or 64 x 48 for, which it has where they fill the chip and pad little: small products
  //    (700, 1.0 of the time at the median) and windows (86, 1.06) there; larger products only with more of a lead (0.85).
  //  * small products whose results are below 20 MB, but for a larger lead (0.81): 16% of them were slower, at 0.92 on average.
  // Of what is left, 2% of the small products, 1% of the others, 1.6% of a transposed B and 1% of the windows are 3% slower and more (before
  // these two 8, 1.4, 3.5 and 10%, up to a third: 11616 x 368 x 14 6.7 and 8.8, 32474 x 112 x 16 5.7 and 7.3, [7,96,98,3] 5x5 -> 61 17.6
  // and 23.0). us, before and here: 4282 x 3818 x 32 34 and 21, 18 x (1007 x 860 x 20) of a transposed B 30 and 19, 3991 x 1333 x 71
  // 20 and 13, 130032 x 224 x 72 (windows) 94 and 54, 81125 x 100 x 40 (ragged) 39 and 24. (By that estimate alone, 3% of the products that
  // the line above takes were not taken any more, and up to 1.3 times slower.)
  const double part = best_us / tiled_end_us(p, a_kind, transposed_b);
  double lead = a_kind == kLoadKAny ? (small ? 0.92 : 0.97) : (small ? 0.87 : 0.91);
  if (small && a_kind == kLoadKAny && (double)p.batch * p.M * p.N < 5e6) lead = 0.81;
  if (!narrow && (a_kind == kLoadKAny || p.K <= kEndWindows) && part <= lead) {
    const TileShape &t = kTileShapes[choose_tile_shape(p.M, p.N, p.K, p.batch, num_cus())];
    const bool suits = t.bm == 64 && t.bn <= 64;
    if (!suits || (!small && a_kind == kLoadKAny && part <= 0.85)) return best;
  }
  best.shape = -1;
  return best;
}

int launch_split_gemm(SplitChoice choice, GemmParams &p, int a_kind, bool transposed_b) {
  if (transposed_b) return launch_kind<kLoadKAny, kLoadKVec>(choice, p);
  if (a_kind == kLoadWindows) return launch_kind<kLoadWindows, kLoadXVec>(choice, p);
  if (a_kind == kLoadWindowsAny) return launch_kind<kLoadWindowsAny, kLoadFilter>(choice, p);
  return launch_kind<kLoadKAny, kLoadXVec>(choice, p);
}

}  // namespace tfhip
