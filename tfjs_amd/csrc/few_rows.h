// Small products: C[M x N] = A[M x K] * B[K x N], row-major, any extents and any 4-byte alignment (a dense layer on a
// handful of examples, an encoder on a short sentence, the late layers of a mobile network on one picture).
//
// Such a product is bound by latency: the launch, one trip to memory, the sum; with very few rows and a large B, by
// fetching B once. So there is no LDS stage and no k loop to speak of. A workgroup of eight wavefronts takes 16 MB
// rows of a strip of 16 CB columns, its wavefronts take k groups of 16 in turn, and each has the fetches of U groups
// out before it waits for the first.
//  * lane (g, r) (g = lane / 16, r = lane % 16) feeds k = 16 T + 4 g + j in the j-th of the four matrix instructions
//    (v_mfma_f32_16x16x4_f32) of group T: of A a float4 of row r, of B columns CB r .. CB r + CB - 1 of row k, 16
//    lanes side by side. Buffer loads need 4-byte alignment only, and what lies beyond an operand reads as zero, dword
//    by dword.
//  * A can be the windows of an NHWC image (KIND kLoadWindows, kLoadWindowsAny: a float4 is a unit of four k of a
//    segment, see ConvGeom): the small convolutions of a network's later stages.
//  * the wavefronts' sums meet in LDS and are added in order.
//  * where the tiles leave compute units idle, `splits` workgroups share one and cut its k: each leaves its sums in
//    scratch, the last to arrive (a counter per tile) adds them in the order of k and finishes. One launch instead of
//    two, and the bits do not depend on who is last.
#pragma once

#include <hip/hip_runtime.h>

#include "common.h"
#include "gemm_host.h"
#include "gemm_kernel.h"

namespace tfhip {

struct FewRowsArgs {
  const float *a, *b, *bias, *prelu, *residual;
  float *c, *ws;
  int *counters;
  long long bias_stride, prelu_stride;
  double leaky_alpha;
  int M, N, K;
  unsigned a_bytes, b_bytes;
  int groups;               // of 16 k
  // Tiles side by side in the order of the workgroups: the row tiles of a strip (of 16 MB rows), or, negative, the strips of a row
  // tile. The two divisors' magic numbers (magic_of).
  int inner;
  int splits, groups_per_split;
  unsigned inner_magic, splits_magic;
  int finish_apart;         // another launch adds the slices
  ConvGeom conv;            // A gathered from an image (k counted as there)
  int activation;
};

constexpr int kFewRowsWaves = 8;
// Offsets no descriptor here covers, also when a smaller one is added (operands are at most 1 GiB).
constexpr unsigned kOutside = 0x80000000u, kOutsideRow = 0x40000000u;
constexpr long long kFewRowsMaxBytes = 0x40000000LL;

// Sums over wavefronts are written through to memory and read past the reader's L2, which does not see other XCDs'
// lines (a fence at device scope would write back and drop whole caches instead).
constexpr int kThrough = 16;   // sc1

// Strip and row tile of a tile. The operand of the longer side is what the XCDs fetch in parts: all of the shorter one each
// (5967 x 1788 x 64 in 748 tiles, row tiles and strips side by side: 34.2 and 23.7 us).
__device__ __forceinline__ void tile_place(const FewRowsArgs &p, int tile, int &strip, int &row_tile) {
  const int outer = by_magic(tile, p.inner_magic), in = tile - outer * abs(p.inner);
  strip = p.inner > 0 ? outer : in;
  row_tile = p.inner > 0 ? in : outer;
}

// Sum over the slices (or, of one, over the wavefronts' sums in `lds`), bias, activation, residual and store of the
// outputs of a tile; `bias` and `alpha` belong to the thread's column.
template <int MB, int CB>
__device__ __forceinline__ void finish_tile(const FewRowsArgs &p, int tile, float bias, float alpha, const float *lds) {
  constexpr int W = kFewRowsWaves, kCols = 16 * CB, kOut = 256 * MB * CB;
  static_assert((64 * W) % kCols == 0, "a thread keeps its column");
  const __amdgpu_buffer_rsrc_t rsrc_ws = __builtin_amdgcn_make_buffer_rsrc(
      (void *)uniform_pointer(p.ws + (long long)tile * p.splits * kOut), 0, p.splits * kOut * 4, 0x00020000);
  int strip, row_tile;
  tile_place(p, tile, strip, row_tile);
  const int m0 = row_tile * 16 * MB;
  const int col = strip * kCols + (int)threadIdx.x % kCols;
  const int live = min(kOut, (p.M - m0) * kCols);   // elements of the tile that exist (its rows come first)
#pragma unroll 1
  for (int i = threadIdx.x; i < live; i += 64 * W) {
    float v = 0.f;
    if (p.splits > 1) {
#pragma unroll 1
      for (int s0 = 0; s0 < p.splits; s0 += 8) {
        float part[8];
#pragma unroll
        for (int s = 0; s < 8; ++s)   // (beyond the last slice: outside the descriptor, zero)
          part[s] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsrc_ws, 4 * ((s0 + s) * kOut + i), 0, kThrough));
#pragma unroll
        for (int s = 0; s < 8; ++s) v += part[s];
      }
    } else {
      v = lds[i];
#pragma unroll
      for (int w = 1; w < W; ++w) v += lds[w * kOut + i];
    }
    if (col >= p.N) continue;
    v = activate(v + bias, p.activation, alpha, p.leaky_alpha);
    const long long at = (long long)(m0 + i / kCols) * p.N + col;
    p.c[at] = p.residual ? v + p.residual[at] : v;
  }
}

// U: k groups whose fetches a wavefront has out; when it has multiplied one, it asks for the one U further on, in the same
// registers. Issuing a group's fetches takes about 0.1 us, so the first ones are back before four have been asked for:
// with 8 at once, and the next 8 before the first are multiplied, that issue was most of the time. us, then and now:
// 196 x 384 x 64 4.7 and 3.2, 49 x 960 x 320 6.0 and 4.4, 16 x 1280 x 2048 7.1 and 5.3, 23 x 768 x 2304 6.7 and 4.9,
// 128 x 1536 x 768 10.3 and 8.5, 32 x 2304 x 8192 19.4 and 17.9; windows, [1,28,28,64] 5x5 -> 33 12.7 and 8.5. U = 1, 2, 4, 8:
// 16 x 2048 x 2048 6.0, 5.9, 6.0, 6.3; 5 x 2048 x 4096 7.3, 6.6, 6.6, 7.3; 64 x 1280 x 768 5.1, 5.1, 5.2, 6.0;
// with strips of 64 and two row blocks 32 x 1024 x 12288 12.5, 13.1, 14.6, -.
// ROW: the product of one row, multiplied with vector instructions, four per lane, column and group: a matrix instruction
// takes as long for one row as for sixteen, 128 cycles for a group. 1 x 1280 x 1000 6.4 and 3.5, 1 x 2048 x 4096 8.3 and 5.6.
// (Of two rows the vector form is behind, 5.1 and 4.9 with U = 8: all lanes of a group fetch each row's float4.)
template <int MB, int CB, int KIND, bool ROW>
__global__ __launch_bounds__(64 * kFewRowsWaves) void few_rows(FewRowsArgs p) {
  constexpr int U = MB * CB == 8 ? 1 : 2;
  constexpr bool kWindows = KIND != kLoadKAny;
  constexpr int W = kFewRowsWaves;
  static_assert(!ROW || (MB == 1 && !kWindows), "one row of a matrix");
  constexpr int kCols = 16 * CB, kRows = 16 * MB, kOut = kCols * kRows;
  __shared__ float lds[W * kOut];
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, r = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // What the first fetches need, asked for at once (left to itself, the compiler makes two trips of it, 0.2 us each).
  asm volatile("" : : "s"(p.a), "s"(p.b), "s"(p.M), "s"(p.N), "s"(p.K), "s"(p.a_bytes), "s"(p.b_bytes), "s"(p.groups), "s"(p.inner),
               "s"(p.inner_magic), "s"(p.splits), "s"(p.splits_magic), "s"(p.groups_per_split), "s"((int)gridDim.x));
  int id = blockIdx.x;   // neighbouring strips share cache lines: each XCD (ids i, i + 8, ..) gets a contiguous band
  {
    const int per_xcd = gridDim.x / 8;
    if (per_xcd > 0 && id < per_xcd * 8) id = (id % 8) * per_xcd + id / 8;
  }
  // the slices of a tile side by side
  const int tile = by_magic(id, p.splits_magic), split = id - tile * p.splits;
  int strip, row_tile;
  tile_place(p, tile, strip, row_tile);
  const int m0 = row_tile * kRows, n0 = strip * kCols;
  const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc((void *)p.a, 0, (int)p.a_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc((void *)p.b, 0, (int)p.b_bytes, 0x00020000);
  const int begin = split * p.groups_per_split + wave;
  const int end = min(p.groups, (split + 1) * p.groups_per_split);

  unsigned a_row[MB];
  int row_ih[MB], row_lin[MB];   // windows: image row and position in it of the first element
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    const int row = ROW ? 0 : m0 + 16 * m + r;   // (ROW: the same for all lanes)
    if (kWindows) {
      window_row(p.conv, row, p.M, row_ih[m], row_lin[m], a_row[m]);
    } else {
      a_row[m] = row < p.M ? 4u * (unsigned)row * (unsigned)p.K : kOutsideRow;
    }
  }
  const int col = n0 + CB * r;
  const unsigned b_col = col < p.N ? 4u * (unsigned)col : kOutsideRow;
  const unsigned pitch = 4u * (unsigned)p.N;

  struct {
    uint4_t a[U][MB];
    unsigned b[U][4][CB];
    int fix[U][MB];   // units to mend: what fix_up is to do
  } c;
  // group t = first + step * W, into slot u
  auto issue = [&](int u, int first, int step) __attribute__((always_inline)) {
    const unsigned k_first = (unsigned)(16 * first + 4 * g);
    const int t = first + step * W;
    unsigned kb;                   // where row k of B begins, in this lane's columns
    int live_rows = 4;             // of B, of the four
    if (kWindows) {
      const int k = 16 * t + 4 * g;
      const bool on = t < end && k < p.K;
      const ConvGeom &cg = p.conv;
      const int q = k >> 2;
      const int seg = cg.unit_magic ? (int)__umulhi((unsigned)q, (unsigned)cg.unit_magic) : q;
      const int in_seg = 4 * (q - seg * cg.units);
      int fr = seg, fs = 0;
      if (cg.taps > 1) {
        fr = seg / cg.taps;
        fs = seg - fr * cg.taps;
      }
      const int dh = fr * cg.dil_h, dl = fs * cg.seg_col + in_seg;
      const unsigned at = 4u * (unsigned)(fr * cg.seg_row + dl);
      live_rows = cg.seg_len - in_seg;
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        const bool row_in = on && (unsigned)(row_ih[m] + dh) < (unsigned)cg.in_h;
        const int lin = row_lin[m] + dl;
        const int before = KIND == kLoadWindowsAny && lin < 0 ? -lin : 0;
        const bool in = row_in && (KIND == kLoadWindowsAny ? before < 4 && lin < cg.row_len : (unsigned)lin < (unsigned)cg.row_len);
        c.a[u][m] = __builtin_amdgcn_raw_buffer_load_b128(rsrc_a, (int)(in ? a_row[m] + at + 4u * (unsigned)before : kNoOffset), 0, 0);
        if (KIND == kLoadWindowsAny) {
          const int real = min(cg.row_len - lin, live_rows);
          c.fix[u][m] = before << 16 | (real < 0 ? 0 : (real < 4 ? real : 4));
        }
      }
      kb = on ? (unsigned)(seg * cg.seg_len + in_seg) * pitch + b_col : kOutside;
    } else {
      // (a group that is not this slice's: outside both; what is asked for of k beyond the last lies behind B's last row)
      const unsigned gone = t < end ? 0u : kOutside;   // the same for the whole wavefront
#pragma unroll
      for (int m = 0; m < MB; ++m)
        c.a[u][m] = __builtin_amdgcn_raw_buffer_load_b128(rsrc_a, (int)(a_row[m] + 4u * k_first + 64u * (unsigned)(step * W) + gone), 0, 0);
      kb = k_first * pitch + b_col + ((unsigned)(16 * step * W) * pitch + gone);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {   // (rows beyond the last lie beyond the descriptor)
      const int at = (int)(KIND == kLoadWindowsAny && j >= live_rows ? kOutside : kb + (unsigned)j * pitch);
      if constexpr (CB == 4) {
        const uint4_t v = __builtin_amdgcn_raw_buffer_load_b128(rsrc_b, at, 0, 0);
#pragma unroll
        for (int q = 0; q < 4; ++q) c.b[u][j][q % CB] = v[q];
      } else {
        c.b[u][j][0] = __builtin_amdgcn_raw_buffer_load_b32(rsrc_b, at, 0, 0);
      }
    }
  };
  float4_t acc[MB][CB];
  float row_acc[CB];   // ROW: of this lane's k
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int q = 0; q < CB; ++q) acc[m][q] = (float4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int q = 0; q < CB; ++q) row_acc[q] = 0.f;
  auto multiply = [&](int u, int t) __attribute__((always_inline)) {
    const int k = 16 * t + 4 * g;
    float a4[MB][4];
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      float4 v = as_float4(c.a[u][m]);
      // (units of four that lie inside the image row or outside need no mending: the first a fetch gives, the others are zero)
      if (KIND == kLoadWindowsAny) v = fix_up<KIND>(v, c.fix[u][m]);
      else if (!kWindows && 16 * t + 16 > p.K) v = fix_up<KIND>(v, p.K - k);   // (the last float4 of a row may reach into the next one)
      a4[m][0] = v.x; a4[m][1] = v.y; a4[m][2] = v.z; a4[m][3] = v.w;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (ROW) {
#pragma unroll
        for (int q = 0; q < CB; ++q) row_acc[q] = fmaf(a4[0][j], __uint_as_float(c.b[u][j][q]), row_acc[q]);
      } else {
#pragma unroll
        for (int m = 0; m < MB; ++m)
#pragma unroll
          for (int q = 0; q < CB; ++q)
            acc[m][q] = __builtin_amdgcn_mfma_f32_16x16x4f32(a4[m][j], __uint_as_float(c.b[u][j][q]), acc[m][q], 0, 0, 0);
      }
    }
  };

#pragma unroll
  for (int u = 0; u < U; ++u) issue(u, begin, u);
  // what the column this thread finishes needs
  const int my_col = n0 + tid % kCols;
  const bool col_ok = my_col < p.N;
  const float bias = p.bias && col_ok ? p.bias[(long long)my_col * p.bias_stride] : 0.f;
  const float alpha = p.activation == TFHIP_PRELU && col_ok ? p.prelu[(long long)my_col * p.prelu_stride] : 0.f;
  int t = begin;
#pragma unroll 1
  for (; t + U * W < end; t += U * W)
#pragma unroll
    for (int u = 0; u < U; ++u) {
      multiply(u, t + u * W);
      issue(u, t, u + U);
    }
#pragma unroll
  for (int u = 0; u < U; ++u)
    if (t + u * W < end) multiply(u, t + u * W);   // (the same for the whole wavefront)

  // ---- the wavefronts' sums: lane holds rows 16 m + 4 g .. +3 of columns CB r + q (ROW: its k's share of the row)
  if (ROW) {
#pragma unroll
    for (int q = 0; q < CB; ++q) {
      float v = row_acc[q];
      v += __shfl_xor(v, 16);
      v += __shfl_xor(v, 32);
      if (g == 0) lds[wave * kOut + CB * r + q] = v;
    }
  } else {
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int q = 0; q < CB; ++q) lds[wave * kOut + (16 * m + 4 * g + e) * kCols + CB * r + q] = acc[m][q][e];
  }
  lds_barrier();
  auto wave_sum = [&](int i) __attribute__((always_inline)) {
    float v = lds[i];
#pragma unroll
    for (int w = 1; w < W; ++w) v += lds[w * kOut + i];
    return v;
  };
  // ---- k slices
  if (p.splits > 1) {
    const __amdgpu_buffer_rsrc_t rsrc_ws = __builtin_amdgcn_make_buffer_rsrc(
        (void *)uniform_pointer(p.ws + (long long)tile * p.splits * kOut), 0, p.splits * kOut * 4, 0x00020000);
#pragma unroll 1
    for (int i = tid; i < min(kOut, (p.M - m0) * kCols); i += 64 * W)
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(wave_sum(i)), rsrc_ws, 4 * (split * kOut + i), 0, kThrough);
    if (p.finish_apart) return;
    __builtin_amdgcn_s_waitcnt(0);   // the stores are in memory
    __syncthreads();
    int *last = reinterpret_cast<int *>(lds);
    if (tid == 0) {
      const int before = __hip_atomic_fetch_add(p.counters + tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (before == p.splits - 1) __hip_atomic_store(p.counters + tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *last = before == p.splits - 1;
    }
    __syncthreads();
    if (!*last) return;
  }
  finish_tile<MB, CB>(p, tile, bias, alpha, lds);
}

// The sums of the slices of one tile each, where few_rows leaves them (FewRowsArgs::finish_apart).
template <int MB, int CB>
__global__ __launch_bounds__(64 * kFewRowsWaves) void few_rows_finish(FewRowsArgs p) {
  int strip, row_tile;
  tile_place(p, blockIdx.x, strip, row_tile);
  const int col = strip * (16 * CB) + (int)threadIdx.x % (16 * CB);
  const float bias = p.bias && col < p.N ? p.bias[(long long)col * p.bias_stride] : 0.f;
  const float alpha = p.activation == TFHIP_PRELU && col < p.N ? p.prelu[(long long)col * p.prelu_stride] : 0.f;
  finish_tile<MB, CB>(p, blockIdx.x, bias, alpha, nullptr);
}

// How a product in tiles of 16 MB rows and 16 CB columns is cut over workgroups.
constexpr int kFewRowsCounters = 256;
struct FewRowsCut {
  int row_tiles, strips;
  long long tiles;
  int splits, groups_per_split;   // slices of k, and the k groups of 16 in one
};
inline FewRowsCut few_rows_cut(const GemmParams &p, int row_blocks, int col_blocks) {
  FewRowsCut cut;
  cut.row_tiles = row_blocks == 1 ? (p.M + 15) / 16 : (p.M + 31) / 32;
  cut.strips = col_blocks == 1 ? (p.N + 15) / 16 : (p.N + 63) / 64;
  cut.tiles = (long long)cut.row_tiles * cut.strips;
  const int groups = (p.K + 15) / 16;
  // Slices of 32 groups. With one row block a product stays whole up to 64, of one row up to 128: its workgroups have less to add
  // up. us, one slice and more: 1 x 1280 x 1000 3.9 and 5.0, 1 x 2048 x 1000 4.4 and 4.9, 1 x 3072 x 1000 6.1 and 5.3. Beyond, what a
  // compute unit can have out bounds the fetches (some 16 KB), so more units are ahead: with slices of 64, of 32 and the best of ten
  // counts, 16 x 2048 x 256 6.1, 5.3, 5.3, 40 x 2048 x 64 6.1, 4.8, 4.8, 16 x 4096 x 64 6.0, 5.0, 4.7, 1 x 3072 x 256 5.1, 5.0, 4.9; 140
  // products of 1 to 64 rows, 1040 to 4096 and 64 to 1024: 1.10, 1.03 and 1 on average (of 900 others, up to 4096 columns, 14 are more than 3%
  // slower with 32 than with 64). More workgroups than compute units only add to what goes through memory.
  const int whole = row_blocks != 1 ? 32 : (p.M == 1 ? 128 : 64);
  const int wanted = groups <= whole ? 1 : (groups + 31) / 32;
  const int most = cut.tiles * 2 > kFewRowsCounters ? 1 : kFewRowsCounters / (int)cut.tiles;
  cut.splits = wanted < most ? wanted : most;
  cut.groups_per_split = cut.splits == 1 ? groups : (groups + cut.splits - 1) / cut.splits;
  return cut;
}

// Strips of 64 columns, whole cache lines and a quarter of the tiles to share the slices among, where strips of 16
// (cut as `narrow` says) find no compute unit of their own each, or where a workgroup of theirs would fetch more than twice
// (with two row blocks three times) what it can have out at once; else strips of 16: as many workgroups as there are.
// us, strips of 16 and 64: 32 x 1536 x 2304 8.5 and 10.7, 32 x 3072 x 2304 16.3 and 11.5, 160 x 8192 x 256 24.1 and 12.0;
// 1 x 1024 x 4096 3.9 and 4.8. Just beyond the lines the strips of 16 are still ahead since their fetches are refilled one by one
// (1 x 1024 x 4112 5.0 and 5.9, 1 x 2304 x 4000 6.8 and 7.6, 48 x 2304 x 768 7.2 and 8.1); the tests of the dispatch have them here.
inline bool few_rows_wide(const FewRowsCut &narrow, int row_blocks) {
  return narrow.tiles > num_cus() || narrow.groups_per_split > (row_blocks == 1 ? 128 : 96);
}

// (32-bit offsets, no choice of another kernel with a knob)
inline bool few_rows_can(const GemmParams &p, bool windows) {
  if (tuning(kTuneSplit) >= 0 && tuning(kTuneSplit) != 99) return false;   // (99: only that split_gemm is not chosen)
  if (windows ? p.a_bytes > kFewRowsMaxBytes : (long long)p.M * p.K * 4 > kFewRowsMaxBytes) return false;
  return p.batch == 1 && p.K > 0 && p.N <= (1 << 24) && p.epi.channel_operands && p.epi.addressing != kConv && tuning(kTuneTile) < 0 &&
         tuning(kTuneSplitK) < 0 && (long long)p.K * p.N * 4 <= kFewRowsMaxBytes;
}

// Row blocks per workgroup that this kernel takes the product of two row-major operands with, or 0: it goes to the
// tiled kernel (`vec`: that one can fetch both operands in float4s). As long as every workgroup has a compute unit of its
// own, the fetches of a whole k range are out at once, where the tiled kernel goes round its pipeline once per 32 k (us,
// tiled and here: 49 x 960 x 160 9.2 and 4.2, 196 x 576 x 96 6.9 and 3.6, 80 x 768 x 768 8.1 and 4.2; windows,
// [2,35,34,120] 3x3/2 -> 16 11.5 and 5.8). The lines, each from a grid of extents on both sides, in the same form. Those from the
// third on were measured with eight groups out at once; with two, refilled one by one, this kernel has gained 10 to 40%, so they
// are on the safe side now (32 x 512 x 8192 in 5.6 with one row block, 128 x 3072 x 768 in 11.3), and are left where the tests
// of the dispatch have them:
//  * more than 32 rows, K < 320: 0.85 of the time at K = 16, 0.77 at 96, 0.6 at 300 (256 x 256 x 256 5.6 and 4.2, 784 x 192 x 32
//    4.5 and 2.9), except where the caller wants the sums of gemm_kernel (`float_bits`), and not for ragged rows, on which
//    the same is left: the tests of the ragged loader count on it there.
//  * windows of fewer than 256 floats (384 with units to mend): ahead from 48 on (0.84 of the time; [1,28,28,16] 3x3 -> 32 5.5 and 3.7),
//    but left for the same reason; above, 0.7 ([1,14,14,32] 3x3 -> 64 6.7 and 4.1).
//  * up to 32 rows always, from K = 2048 on with two row blocks: half the fetches of B, and slices enough to fill the
//    chip (23 x 3072 x 768 9.3 with one, 7.7 with two). Except 17 to 32 rows of 4097 to 8192 columns with K <= 1536
//    (where a float4 fits the rows, else 768): more strips than compute units, while each of the tiled kernel's 32-wide tiles
//    has one (32 x 512 x 8192 6.4 and 8.3, 32 x 1024 x 5000 8.9 and 11.2; 32 x 2048 x 5000 14.2 and 14.2,
//    32 x 1024 x 12288 17.9 and 13.9; ragged, 32 x 511 x 5001 7.3 and 8.4, 24 x 768 x 5001 9.3 and 9.5,
//    24 x 1280 x 5001 13.4 and 10.6).
//  * more than 32 rows with two row blocks, K <= 1536: 128 x 1024 x 1024 9.1 and 7.5, 128 x 1536 x 768 12.8 and 10.1;
//    128 x 3072 x 768 13.8 and 16.8. (128 x 1792 x 768, 14.4 and 11.4, is left on the wrong side.)
//  * windows have no strips of 64: with two strips and more, a workgroup on a third of the compute units and more, and
//    more than 192 groups for it (288 where the tiled kernel's loader has units to mend), the tiled kernel is ahead
//    ([1,10,10,256] 5x5 -> 256 14.5 and 15.4, [1,14,14,256] 7x7 -> 256 30.5 and 39.7; on 64 tiles [1,7,7,256] 7x7 -> 256
//    21.0 and 13.8; at 144 groups [1,10,10,512] 3x3 -> 256 12.8 and 13.0; of one strip [3,34,19,260] 7x7 -> 8 30.7 and
//    22.6; ragged, at 222 groups [3,33,22,141] 5x5/2 -> 111 22.2 and 20.3, at 399 [1,20,20,130] 7x7 -> 130 24.0 and 29.7).
inline int few_rows_blocks(const GemmParams &p, bool windows, bool vec, bool float_bits = false) {
  if (!few_rows_can(p, windows) || (windows && p.K < (vec ? 256 : 384))) return 0;
  const long long strips = (p.N + 15) / 16, cus = num_cus();
  int blocks = 0;
  if (p.M <= 16) blocks = 1;
  else if (p.M > 32 && p.K < 320 && !windows && (!vec || float_bits || p.K < 16)) blocks = 0;
  else if (p.M <= 32 && p.K > 2048) blocks = 2;
  else if ((p.M + 15) / 16 * strips <= cus) blocks = 1;
  else if (p.M <= 32) blocks = strips > cus && strips <= 2 * cus && p.K <= (vec ? 1536 : 768) ? 0 : 2;
  else if ((p.M + 31) / 32 * strips <= cus && p.K <= 1536) blocks = 2;
  if (windows && blocks != 0) {
    const FewRowsCut cut = few_rows_cut(p, blocks, 1);
    if (strips > 1 && cut.tiles * 3 > cus && cut.groups_per_split > (vec ? 192 : 288)) blocks = 0;
  }
  return blocks;
}

// The same where there are more tiles than compute units, which then share them: two row blocks with a strip of 16 columns, or one
// with a strip of 64, where the estimate for either is below that for the kernel that would have it otherwise (`split`: what
// the bf16 parts would take, if they are chosen; else gemm_kernel). An estimate is a launch, what a workgroup does round by round (16 k
// per wavefront, 32 for gemm_kernel), and per compute unit its tiles' share of fetches and matrix work and their ends; tiles count in
// part as they are and in part as full rounds over the chip. Least squares on 25000 products and 18000 convolutions of random extents in
// the ranges below, root mean square error 4 to 9% here and 5 to 7% for gemm_kernel. Of what the lines above leave to gemm_kernel,
// 85% of the convolutions are taken, on average at 0.79 of its time (0.71 where its loader has units to mend); of the products
// two thirds at 0.91 and 0.87 (ragged), with up to 700 rows nearly all at 0.84 and 0.75. 1 to 4% of what is taken is 3% slower and more.
// Of what the bf16 parts would have, 7500 that were taken: 0.90 of their time (products) and 0.76 (windows) at the median.
// us, before and here: 48 x 2304 x 2304 15.8 and 10.0, 64 x 768 x 3072 8.0 and 6.3, [3,113,75,21] 5x5/2 -> 38 14.4 and 10.5,
// [1,56,56,64] 3x3 -> 64 8.7 and 6.6. What is not taken at all: K below 384 (windows: 192), as with fewer tiles, where at most a fifth of 5 us is left; K above
// 3000 (2048), where gemm_kernel cuts k into slices; more than 10000 rows, whose A comes from memory, and 40000 windows,
// for which gemm_kernel has tiles of 256 rows (both in 0.85 of the time).
struct FewRowsForm {
  int row_blocks, col_blocks;   // 0, 0: not with this kernel
};
inline FewRowsForm few_rows_form(const GemmParams &p, int kind, bool vec, const SplitChoice &split) {
  const bool windows = kind != kLoadKAny;
  const long long cus = num_cus(), row_pairs = (p.M + 31) / 32, rows = (p.M + 15) / 16, strips = (p.N + 15) / 16;
  if (!few_rows_can(p, windows) || p.M <= 32 || p.N < 4 || row_pairs * strips > 3000) return {0, 0};
  if (windows ? rows * strips <= cus || p.M > 40000 || p.K < 192 || p.K > 2048 : row_pairs * strips <= cus || p.M > 10000 || p.K < 384 || p.K > 3000)
    return {0, 0};
  const auto us = [&](const RoundsEstimate &e, long long tiles) { return rounds_us(e, tiles, (p.K + 15) / 16, kFewRowsWaves); };
  // products; windows; windows whose units need mending
  static constexpr RoundsEstimate kTwoRows[3] = {{2.83, 0.143, 0.0435, 0.40, 0.75}, {3.16, 0.146, 0.0492, 0.71, 0.75}, {2.95, 0.279, 0.0578, 0.83, 0.75}};
  static constexpr RoundsEstimate kWide[3] = {{3.13, 0.055, 0.0610, 0.67, 0.75}, {3.22, 0.171, 0.0656, 0.77, 0.75}, {3.19, 0.216, 0.0721, 0.80, 0.75}};
  const int which = kind == kLoadKAny ? 0 : (kind == kLoadWindows ? 1 : 2);
  const double two_rows = us(kTwoRows[which], row_pairs * strips);
  const double wide = us(kWide[which], rows * ((p.N + 63) / 64));
  // (The bf16 parts have up to 32 columns only where K is long: with these rows and K they take 0.85 to 1.12 of this kernel's time.)
  const double other = split.shape >= 0 && p.N > 32 ? split.us : tiles_of_32_us(p, windows, vec);
  if (fmin(two_rows, wide) > 0.93 * other) return {0, 0};
  return two_rows < wide ? FewRowsForm{2, 1} : FewRowsForm{1, 4};
}

// `kind`: kLoadKAny (row-major A), kLoadWindows or kLoadWindowsAny. Strips of 16 `col_blocks` columns; 0: by few_rows_wide.
int launch_few_rows(const GemmParams &p, int row_blocks, int kind, int col_blocks = 0);

}  // namespace tfhip
