// Tiled product of float32 operands on the bf16 matrix cores, for products large enough to be bound by arithmetic.
//
// A float32 is the sum of three bf16 (8 + 8 + 8 bits of its 24): x = h + m + l, exactly. Six of the nine products of the
// parts of a and b are summed in float32, h h', h m', m h', m m', h l', l h'; the three left out are below 2^-26 of the
// product. v_mfma_f32_32x32x16_bf16 does 16 times the multiply-adds of v_mfma_f32_16x16x4_f32 in a cycle, so six of them
// take 3/8 of the time. Rounding: the bf16 instruction adds its 16 products to the accumulator with one rounding, the
// float32 one rounds after each of its four; the five small products have an accumulator of their own. Error against 64
// bits, 2-norm relative, K = 64, 256, 768, 3072, operands N(0, 1) and N(0, 0.02): float32 matrix instructions 1.4e-7, 2.9e-7,
// 5.0e-7, 9.8e-7, this kernel 0.5e-7, 0.9e-7, 1.6e-7, 3.4e-7; all-positive operands 1.2e-7 ... 8.3e-7 and 0.5e-7 ... 3.0e-7.
//
// us, gemm_kernel and here (rate of the product itself; extents are rows x columns x inner): 1024 x 2304 x 768 33.4 and 24.0 (151 TFLOP/s), 1024 x 3072 x 768 40.8
// and 27.9, 3072 x 3072 x 1024 153 and 106 - 112 by machine (180), 3072 x 4096 x 1024 189 and 134 - 139 (189), [8,56,56,64] 3x3 -> 64 26.7 and 16.4.
// Of a transposed B, 128 x (384 x 384 x 64) 32.5 and 26.8, 128 x (512 x 512 x 64) 56 and 44, 1024 x 3072 x 768 38.8 and 28.7.
// What bounds it: the loop, and in it the matrix cores for 67% of its cycles (128 x 128 tiles 70%), fetches and barriers for
// the rest. A k tile of a 128 x 96 tile takes 0.69 us on 64 of the 256 units and 0.99 on all of them, where the chip's clock
// falls from 2.30 to 1.70 GHz (busy and active cycles of launches of 1 ms, by counter). Over a launch of 3072 x 3072 x 1024 the
// matrix cores are busy for 43% of 2.4 GHz: that clock, the waits, and 5 to 6 us of prologue and results in each of three
// rounds are the rest. (64 rows per wavefront in tiles of 256 x 128 on four wavefronts, half of the reads of B's fragments and half of its
// splitting, change nothing: 4096^3 takes 660 us with 128 x 128 and 650, 3072 x 4096 x 1024 136 to 141 and 160. Nor do idle units: 192 tiles of
// 3072 x 1024 x 4096 take as long as 768 of 3072 x 4096 x 1024. So the power is a part of it, not all: on eight wavefronts that tile took
// 612 us, and the 16x16x32 instruction 2 to 4% less in large 128 x 128 tiles; both lose on smaller products.) On 1024 rows, 6 us of launch, prologue (2.5: arguments, the first fetch, the first tile's splitting) and
// results (2.7), and with 2304 or 768 columns a quarter of the units idle. (Slices of k that the last workgroup of a tile adds, instead of a
// launch over the whole chip: 1024 x 768 x 3072 33.2 and 37.1.)
//
// The last bit of a float32 may be 2^-149, that of a bf16 2^-133: both operands are multiplied by 2^24 before they are split
// (two vector instructions per pair of floats beside eleven), so that every part of every float is a normal bf16 or zero, and
// the sums by 2^-48 behind the loop. All of it is exact. Without, an operand below 2^-109 loses its lower parts and one below
// 2^-134 everything, whatever it is multiplied by; encoder layers of [8,128] and [8,384] took 1.4% and 2.7% less, [8,56,56,64]
// 3x3 -> 64 17.8 us (18.4 with it).
//
// An Inf or NaN in an operand, an operand from 2^104 on or a sum from 2^80 on makes every result it enters Inf or NaN, not
// always the right one of the two; the last stage sees them. It then fetches the tile's operands once more for the largest
// float of each. Where these are small enough that nothing can have overflowed, the sums of the high parts alone are right for
// such results; else the tile is done again with float32 instructions, one float per lane and fetch. us, without an Inf or NaN,
// with one, with one in every row: 1024 x 2304 x 768 28, 41, 42, 3072 x 3072 x 1024 107, 138, 159, [8,56,56,64] 3x3 -> 64 18.4, 30, 31
// (gemm_kernel 34 to 38, 154 and 27.5, all the same); with an operand of 1e32 94, 225 and 78.
//
// One workgroup: KG groups of GW wavefronts share a tile of 32 GW x 32 TN results; every group takes every KG-th k tile of
// 32. A wavefront owns 32 rows.
//  * Fetches go to the next lanes of the same row first (8 lanes, 128 bytes): with a row per lane, in the order in which the
//    matrix instruction wants A, the fetches alone took as long as everything else together (128 x 128 tile, a k tile
//    1.3 us; 0.96 as they are).
//  * A goes through LDS as it is, to change hands within the wavefront (no barrier), and is split in registers.
//  * B is split on its way into LDS, three planes of [column][k], two buffers; one barrier per k tile, in front of the last
//    block of a tile, whose fragments are in registers by then.
//  * A few instructions of the next tile's splitting stand behind each matrix instruction (`side`): vector instructions run
//    beside the bf16 matrix instructions, unlike beside the float32 ones, as many as a wavefront pair can issue: five to
//    seven of all kinds per matrix instruction of 32 cycles, and 7 to 10 are there. So none goes into the addresses of products.
//  * The results meet in LDS and leave it row by row. (Stored from the registers they were in, a row per lane, they took
//    10 us of a launch of 40.)
#pragma once

#include <hip/hip_runtime.h>

#include "common.h"
#include "gemm_kernel.h"

namespace tfhip {

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float float2_t __attribute__((ext_vector_type(2)));
typedef float float16_t __attribute__((ext_vector_type(16)));
typedef unsigned int uint2_t __attribute__((ext_vector_type(2)));
typedef unsigned int uint3_t __attribute__((ext_vector_type(3)));

// An operand's scale, and what takes both from a sum.
constexpr float kSplitScale = 0x1p24f, kSplitUnscale = 0x1p-48f;

__device__ __forceinline__ unsigned pack_bf16(float x, float y) {
  const float2_t v = {x, y};
  return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2_t));
}

__device__ __forceinline__ float16_t mfma_bf16(uint4_t a, uint4_t b, float16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// Byte offset of the 16-byte chunk `chunk` (eight k) of row `row` in a plane of 64 bytes per row: a permutation within four
// rows and one within a row, so that eight lanes that read the same chunk of consecutive rows, and the 32 lanes that write
// half a chunk each (four k units of eight columns, four columns apart), find different banks.
__device__ __forceinline__ int plane_offset(int row, int chunk) {
  const int q = row >> 2;
  return ((row & ~3) | ((row + (q & 1) + (q >> 1 & 2)) & 3)) * 64 + ((chunk ^ q) & 3) * 16;
}

template <int GW, int TN, int KG>
struct SplitTile {
  static constexpr int BM = 32 * GW, BN = 32 * TN;
  static constexpr int kGroupThreads = 64 * GW, kThreads = kGroupThreads * KG;
  static constexpr int XW = BN / (8 * GW);   // columns of B per thread, four k each
  static_assert(XW >= 1 && XW <= 4, "one fetch per k");
  static constexpr int PLANE = BN * 64, BUF = 3 * PLANE, GROUP_BYTES = 2 * BUF + BM * 128;
  static constexpr int PITCH = BN + 4;       // floats per row of the results
  static constexpr int SUM_BYTES = KG * BM * PITCH * 4;
  static constexpr int LDS_BYTES = (KG * GROUP_BYTES > SUM_BYTES ? KG * GROUP_BYTES : SUM_BYTES + 16);
};

// What a row of B is that goes with k (kLoadFilter: k counts as ConvGeom says; -1: none).
template <int B_KIND>
__device__ __forceinline__ int filter_row(const ConvGeom &g, int k) {
  if (B_KIND != kLoadFilter) return k;
  const WindowUnit u = window_unit(g, k & ~3);
  const int in_seg = u.in_seg + (k & 3);
  return in_seg < g.seg_len ? u.seg * g.seg_len + in_seg : -1;
}

// Element k of a row of A (of a window: where it begins), or zero.
template <int A_KIND>
__device__ __forceinline__ float one_of_a(const GemmParams &p, __amdgpu_buffer_rsrc_t rsrc, int row, int k, int k_end, int ih, int iw, unsigned off) {
  bool in = k < k_end && row < p.M;
  unsigned at = 4u * ((unsigned)row * (unsigned)p.a_sx + (unsigned)k);
  if (A_KIND != kLoadKAny) {
    const WindowUnit u = window_unit(p.conv, k & ~3);
    const int lin = iw + u.dl + (k & 3);
    in = in && (unsigned)(ih + u.dh) < (unsigned)p.conv.in_h && (unsigned)lin < (unsigned)p.conv.row_len;
    at = off + u.at + 4u * (unsigned)(k & 3);
  }
  return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)(in ? at : kNoOffset), 0, 0));
}

// A_KIND: kLoadKAny (row-major), kLoadWindows or kLoadWindowsAny. B_KIND: kLoadXVec (row-major), kLoadFilter, kLoadKVec
// (transposed: a row per column, K a multiple of four; its lanes run along k, eight to a column). Any extents otherwise
// and any 4-byte alignment: what lies beyond an operand reads as zero, and what the last fetch of a row of A holds of the
// next row meets rows of B that are zero.
template <int GW, int TN, int KG, int A_KIND, int B_KIND>
__global__ __launch_bounds__(64 * GW * KG, 2) void split_gemm(GemmParams p) {
  using T = SplitTile<GW, TN, KG>;
  constexpr bool kWindows = A_KIND != kLoadKAny, kColumns = B_KIND == kLoadKVec;
  // Whether the compiler keeps what goes beside a block of matrix instructions beside that block. us, as the source has it after every
  // matrix instruction, by blocks, and with the tile's order left to the compiler: [8,56,56,64] 3x3 -> 64 17.8, 16.4, 18.2, [2,56,56,96]
  // 5x5 -> 96 29.3, 28.4, 28.8; in four groups [8,28,28,128] 3x3 -> 128 19.9, 20.2, 19.3; products 1024 x 768 x 768 13.4, 13.6, 12.9,
  // 1024 x 2304 x 768 24.3, 25.1, 24.0, 3072 x 3072 x 1024 107.0, 108.9, 105.8.
  constexpr bool kByBlock = kWindows && KG == 2;
  constexpr int kOffsets = kColumns ? T::XW : (B_KIND == kLoadFilter ? 1 : 4);   // of this thread's fetches of B: a column's, or a row's
  extern __shared__ char split_lds[];
  // (the arguments of the prologue in one piece, as in gemm_kernel)
  asm volatile("" ::"s"(p.a), "s"(p.b), "s"(p.M), "s"(p.N), "s"(p.K), "s"(p.batch), "s"(p.a_sx), "s"(p.b_sk), "s"(p.a_bytes),
               "s"(p.b_bytes), "s"(p.tiles_m), "s"(p.tiles_n), "s"(p.group_m), "s"(p.by_magic),
               "s"(p.panel_magic), "s"(p.rows_magic), "s"(p.last_rows_magic), "s"(p.splits), "s"(p.k_per_split), "s"((int)gridDim.x));
  int split, bz, tile_m, tile_n;
  tile_of(p, split, bz, tile_m, tile_n);
  const int k_begin = split * p.k_per_split;
  const int k_end = k_begin + p.k_per_split < p.K ? k_begin + p.k_per_split : p.K;
  const int m0 = tile_m * T::BM, n0 = tile_n * T::BN;

  const float *A = uniform_pointer(p.a + (long long)(p.batch == 1 ? 0 : bz % p.batch_a) * p.a_batch_stride);
  const float *B = uniform_pointer(p.b + (long long)(p.batch == 1 ? 0 : bz % p.batch_b) * p.b_batch_stride);
  const int group = KG > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x / T::kGroupThreads) : 0;
  const int tid = (int)threadIdx.x - group * T::kGroupThreads, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, r = lane & 31;   // half of a 16 k step, row of A or column of B

  // LDS of the group: two buffers of B's planes, then the rows of A, 128 bytes each, its 16-byte chunks permuted by row
  char *planes = split_lds + group * T::GROUP_BYTES;
  char *a_lds = planes + 2 * T::BUF + wave * 4096;
  // A: this lane fetches the four k from 4 (lane % 8) on of rows 8 v + lane / 8; it multiplies row r
  const int a_to = (lane >> 3) * 128 + ((lane ^ lane >> 3) & 7) * 16;
  int a_from[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) a_from[v] = r * 128 + (((4 * (v >> 1) + 2 * h + (v & 1)) ^ r) & 7) * 16;
  int row_ih[4], row_iw[4];
  unsigned a_off[4], b_off[kOffsets];
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int row = m0 + 32 * wave + 8 * v + (lane >> 3);
    if (kWindows) window_row(p.conv, row, p.M, row_ih[v], row_iw[v], a_off[v]);
    else a_off[v] = row < p.M ? 4u * ((unsigned)row * (unsigned)p.a_sx + 4u * (unsigned)(lane & 7)) : kNoOffset;
  }
  // B: this thread fetches the four k from 4 kb on of columns XW xb .. XW xb + XW - 1
  const int kb = kColumns ? tid & 7 : tid >> 3 & 7, xb = (kColumns ? tid >> 3 & 7 : tid & 7) + (tid >> 6) * 8;
  int b_to[T::XW], b_from[2];
#pragma unroll
  for (int c = 0; c < T::XW; ++c) b_to[c] = plane_offset(T::XW * xb + c, kb >> 1) + (kb & 1) * 8;
#pragma unroll
  for (int s = 0; s < 2; ++s) b_from[s] = plane_offset(r, 2 * s + h);
#pragma unroll
  for (int c = 0; c < kOffsets; ++c) {
    const int x = n0 + T::XW * xb + (kColumns ? c : 0);
    const unsigned at = kColumns ? (unsigned)x * (unsigned)p.b_sx + 4u * (unsigned)kb
                                 : (B_KIND == kLoadFilter ? 0u : (unsigned)(4 * kb + c) * (unsigned)p.b_sk) + (unsigned)x;
    b_off[c] = x < p.N ? 4u * at : kNoOffset;
  }

  uint4_t ra[4];   // fetched, not yet in LDS
  int fix[4];      // (what fix_up is to do with them)
  float4_t rv[2];  // back from LDS
  float rb[4][T::XW];
  auto tile_k = [&](int tile) __attribute__((always_inline)) { return k_begin + (KG * tile + group) * 32; };
  // What lies behind the first `bytes` of an operand. The descriptor moves from k tile to k tile and the lanes' offsets stay: no
  // vector instruction goes into addresses. (A tile beyond the range: a descriptor of no bytes, zeros.)
  auto rest_of = [&](const float *base, unsigned size, unsigned bytes, bool in) __attribute__((always_inline)) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)(reinterpret_cast<const char *>(base) + bytes), 0, in && bytes < size ? (int)(size - bytes) : 0, 0x00020000);
  };
  auto load_a = [&](int tile) __attribute__((always_inline)) {
    const int k0 = tile_k(tile);
    if (kWindows) {
      const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)A, 0, k0 < k_end ? (int)p.a_bytes : 0, 0x00020000);
      const int k = k0 + 4 * (lane & 7);
      const WindowUnit u = window_unit(p.conv, k);
#pragma unroll
      for (int v = 0; v < 4; ++v) ra[v] = load_window_unit<A_KIND>(p.conv, u, k < k_end, row_ih[v], row_iw[v], a_off[v], rsrc, fix[v]);
    } else {
      const __amdgpu_buffer_rsrc_t rsrc = rest_of(A, p.a_bytes, 4u * (unsigned)k0, k0 < k_end);
#pragma unroll
      for (int v = 0; v < 4; ++v) ra[v] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)a_off[v], 0, 0);
    }
  };
  auto load_b = [&](int tile) __attribute__((always_inline)) {
    const int k0 = tile_k(tile);
    const __amdgpu_buffer_rsrc_t rsrc =
        rest_of(B, p.b_bytes, B_KIND == kLoadFilter ? 0u : 4u * (unsigned)k0 * (unsigned)(kColumns ? 1 : p.b_sk), k0 < k_end);
    if constexpr (kColumns) {   // (of k beyond the end nothing, whatever A holds there)
#pragma unroll
      for (int c = 0; c < T::XW; ++c) {
        const unsigned off = k0 + 4 * kb < k_end ? b_off[c] : kNoOffset;
        const uint4_t v = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)off, 0, 0);
#pragma unroll
        for (int j = 0; j < 4; ++j) rb[j][c] = __uint_as_float(v[j]);
      }
      return;
    }
    unsigned unit = 0;
    int live = 4;
    if (B_KIND == kLoadFilter) {
      const WindowUnit u = window_unit(p.conv, k0 + 4 * kb);
      unit = 4u * (unsigned)(u.seg * p.conv.seg_len + u.in_seg) * (unsigned)p.b_sk;
      live = k0 + 4 * kb < k_end ? p.conv.seg_len - u.in_seg : 0;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      unsigned off = B_KIND == kLoadFilter ? __builtin_elementwise_add_sat(b_off[0], unit + 4u * (unsigned)j * (unsigned)p.b_sk) : b_off[j];
      if (B_KIND == kLoadFilter) off = j < live ? off : kNoOffset;
      if constexpr (T::XW == 4) {
        const uint4_t v = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)off, 0, 0);
#pragma unroll
        for (int q = 0; q < 4; ++q) rb[j][q] = __uint_as_float(v[q]);
      } else if constexpr (T::XW == 3) {
        const uint3_t v = __builtin_amdgcn_raw_buffer_load_b96(rsrc, (int)off, 0, 0);
#pragma unroll
        for (int q = 0; q < 3; ++q) rb[j][q] = __uint_as_float(v[q]);
      } else if constexpr (T::XW == 2) {
        const uint2_t v = __builtin_amdgcn_raw_buffer_load_b64(rsrc, (int)off, 0, 0);
#pragma unroll
        for (int q = 0; q < 2; ++q) rb[j][q] = __uint_as_float(v[q]);
      } else {
        rb[j][0] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)off, 0, 0));
      }
    }
  };
  auto write_a = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      if (A_KIND == kLoadWindowsAny) *reinterpret_cast<float4 *>(a_lds + a_to + v * 1024) = fix_up<A_KIND>(as_float4(ra[v]), fix[v]);
      else *reinterpret_cast<uint4_t *>(a_lds + a_to + v * 1024) = ra[v];
    }
  };
  auto read_a = [&](int half) __attribute__((always_inline)) {
#pragma unroll
    for (int v = 0; v < 2; ++v) rv[v] = *reinterpret_cast<const float4_t *>(a_lds + a_from[2 * half + v]);
  };

  // Four floats are split in four steps, a pair's high part and its rest, then the other pair's.
  uint4_t fa[2][3], fb[2][3];   // fragments: [half][part] of A, [ring][part] of a block of B
  float rx, ry;
  uint2_t out[3];
  auto split_hi = [&](float x, float y, int at) __attribute__((always_inline)) {
    x *= kSplitScale;
    y *= kSplitScale;
    const unsigned hi = pack_bf16(x, y);
    rx = x - __uint_as_float(hi << 16);
    ry = y - __uint_as_float(hi & 0xffff0000u);
    out[0][at] = hi;
  };
  auto split_lo = [&](int at) __attribute__((always_inline)) {
    const unsigned mid = pack_bf16(rx, ry);
    out[1][at] = mid;
    out[2][at] = pack_bf16(rx - __uint_as_float(mid << 16), ry - __uint_as_float(mid & 0xffff0000u));
  };
  int from = 0, to = 0;   // byte offsets of the buffers of B that are read and filled
  auto b_step = [&](auto q_tag) __attribute__((always_inline)) {
    constexpr int c = decltype(q_tag)::value / 4, q = decltype(q_tag)::value % 4;
    if constexpr (q == 0) split_hi(rb[0][c], rb[1][c], 0);
    if constexpr (q == 2) split_hi(rb[2][c], rb[3][c], 1);
    if constexpr (q % 2 == 1) split_lo(q / 2);
    if constexpr (q == 3)
#pragma unroll
      for (int s = 0; s < 3; ++s) *reinterpret_cast<uint2_t *>(planes + to + s * T::PLANE + b_to[c]) = out[s];
  };
  auto a_step = [&](auto q_tag) __attribute__((always_inline)) {
    constexpr int v = decltype(q_tag)::value / 4, q = decltype(q_tag)::value % 4;
    if constexpr (q == 0) split_hi(rv[v & 1][0], rv[v & 1][1], 0);
    if constexpr (q == 2) split_hi(rv[v & 1][2], rv[v & 1][3], 1);
    if constexpr (q % 2 == 1) split_lo(q / 2);
    if constexpr (q == 3)
#pragma unroll
      for (int s = 0; s < 3; ++s) {
        fa[v >> 1][s][2 * (v & 1)] = out[s].x;
        fa[v >> 1][s][2 * (v & 1) + 1] = out[s].y;
      }
  };
  auto read_b = [&](int ring, int buf, int half, int j) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 2; s >= 0; --s)
      fb[ring][s] = *reinterpret_cast<const uint4_t *>(planes + buf + s * T::PLANE + b_from[half] + j * 2048);
  };

  float16_t acc[TN], low[TN];   // h h', and the small products
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int q = 0; q < 16; ++q) acc[j][q] = low[j][q] = 0.f;

  // every group goes through the same number of tiles and barriers
  const int tiles = ((k_end - k_begin + 31) / 32 + KG - 1) / KG;
  load_b(0);
  load_a(0);
  static_for(std::make_integer_sequence<int, 4 * T::XW>(), b_step);
  load_b(1);
  write_a();
  load_a(1);
  read_a(0);
  static_for(std::make_integer_sequence<int, 8>(), a_step);
  read_a(1);
  lds_barrier();
  read_b(0, 0, 0, 0);

  // What is done beside the 6 TN matrix instructions of half H of a tile, in this order:
  //  H = 0: A's second half is split; the next tile's B is split into the other buffer; the fetch of the B after it
  //  H = 1: the next tile's A goes to LDS, the fetch of the one after it; its first half is split, its second one read
  auto side = [&](int tile, auto h_tag, auto q_tag) __attribute__((always_inline)) {
    constexpr int H = decltype(h_tag)::value, q = decltype(q_tag)::value;
    if constexpr (H == 0) {
      if constexpr (q < 8) a_step(std::integral_constant<int, 8 + q>());
      else if constexpr (q < 8 + 4 * T::XW) b_step(std::integral_constant<int, q - 8>());
      else load_b(tile + 2);
    } else {
      if constexpr (q == 0) { write_a(); read_a(0); }
      else if constexpr (q == 1) load_a(tile + 2);
      else if constexpr (q < 10) a_step(std::integral_constant<int, q - 2>());
      else read_a(1);
    }
  };
  for (int tile = 0; tile < tiles; ++tile) {
    to = from ^ T::BUF;
    static_for(std::make_integer_sequence<int, 2 * TN>(), [&](auto b_tag) __attribute__((always_inline)) {
      constexpr int b = decltype(b_tag)::value, H = b / TN, j = b % TN, ring = b & 1;
      constexpr int NM = 6 * TN, NS = H == 0 ? 9 + 4 * T::XW : 11;
      if constexpr (b == 2 * TN - 1) {
        // every fragment of this tile is in registers, every part of the next one in LDS
        __builtin_amdgcn_sched_barrier(0);
        lds_barrier();
        __builtin_amdgcn_sched_barrier(0);
        read_b(ring ^ 1, to, 0, 0);
      } else {
        read_b(ring ^ 1, from, (b + 1) / TN, (b + 1) % TN);
      }
      static_for(std::make_integer_sequence<int, 6>(), [&](auto q_tag) __attribute__((always_inline)) {
        constexpr int q = decltype(q_tag)::value, m = 6 * j + q;
        constexpr int bp = q == 0 ? 2 : (q < 3 ? 1 : 0), ap = q == 2 || q == 4 ? 1 : (q == 5 ? 2 : 0);
        if constexpr (q == 3) acc[j] = mfma_bf16(fb[ring][bp], fa[H][ap], acc[j]);
        else low[j] = mfma_bf16(fb[ring][bp], fa[H][ap], low[j]);
        constexpr int first = m * NS / NM, last = (m + 1) * NS / NM;
        static_for(std::make_integer_sequence<int, last - first>(), [&](auto z) __attribute__((always_inline)) {
          side(tile, std::integral_constant<int, H>(), std::integral_constant<int, first + decltype(z)::value>());
        });
      });
      if constexpr (kByBlock) __builtin_amdgcn_sched_barrier(0);
    });
    from = to;
  }

  // ---- the groups' sums, through LDS (lane (h, r) holds row r, columns 32 j + 8 q + 4 h .. + 3) and out row by row
  constexpr int kQuads = T::BN / 4, kRowsAtOnce = T::kThreads / kQuads, kPasses = (T::BM + kRowsAtOnce - 1) / kRowsAtOnce;
  static_assert(kPasses <= 32, "a bit per pass");
  const Epilogue &e = p.epi;
  const bool fused = p.inline_epilogue != 0;
  const int quad = (int)threadIdx.x % kQuads, row0 = (int)threadIdx.x / kQuads, col = n0 + 4 * quad;
  // (no bias: a descriptor of no bytes; the strides are 0 or 1)
  float bias[4], alpha[4];
  {
    const bool with_bias = fused && e.bias != nullptr, with_alpha = fused && e.activation == TFHIP_PRELU;
    const __amdgpu_buffer_rsrc_t rsrc_bias = __builtin_amdgcn_make_buffer_rsrc((void *)e.bias, 0, with_bias ? p.N * 4 : 0, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrc_alpha = __builtin_amdgcn_make_buffer_rsrc((void *)e.prelu, 0, with_alpha ? p.N * 4 : 0, 0x00020000);
    const int bias_step = (int)e.bias_s[3] * 4, alpha_step = (int)e.prelu_s[3] * 4;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      bias[q] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsrc_bias, (col + q) * bias_step, 0, 0));
      alpha[q] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsrc_alpha, (col + q) * alpha_step, 0, 0));
    }
  }
  lds_barrier();
  float *sums = reinterpret_cast<float *>(split_lds);   // [KG][BM][PITCH]
  unsigned *seen = reinterpret_cast<unsigned *>(split_lds + T::SUM_BYTES);   // an Inf or NaN; the largest float of A's rows, of B's columns
  auto write_sums = [&](auto sum_of) __attribute__((always_inline)) {
    float *mine = sums + (group * T::BM + 32 * wave + r) * T::PITCH + 4 * h;
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int q = 0; q < 16; q += 4)
        *reinterpret_cast<float4_t *>(mine + 32 * j + 2 * q) =
            (float4_t){sum_of(acc[j][q], low[j][q]), sum_of(acc[j][q + 1], low[j][q + 1]), sum_of(acc[j][q + 2], low[j][q + 2]), sum_of(acc[j][q + 3], low[j][q + 3])};
  };
  if (threadIdx.x < 3) seen[threadIdx.x] = 0;
  write_sums([](float high, float small) { return high + small; });
  lds_barrier();
  const bool to_ws = p.splits > 1;
  const int ldc = to_ws ? p.N : (int)p.ldc;
  const __amdgpu_buffer_rsrc_t rsrc_c = __builtin_amdgcn_make_buffer_rsrc(
      (void *)uniform_pointer(to_ws ? p.ws + ((long long)split * p.batch + bz) * p.M * p.N : p.c + (long long)bz * p.c_batch_stride), 0,
      (int)p.c_bytes, 0x00020000);
  const bool residual = fused && e.residual != nullptr;   // (it lies where the result does)
  const __amdgpu_buffer_rsrc_t rsrc_r = __builtin_amdgcn_make_buffer_rsrc(
      (void *)uniform_pointer(e.residual + (long long)bz * p.c_batch_stride), 0, residual ? (int)p.c_bytes : 0, 0x00020000);
  const int rows = row0 >= kRowsAtOnce || col >= p.N ? 0 : (p.M - m0 < T::BM ? p.M - m0 : T::BM);
  const unsigned first = 4u * ((unsigned)(m0 + row0) * (unsigned)ldc + (unsigned)col), stride = 4u * (unsigned)(kRowsAtOnce * ldc);
  float unscale = kSplitUnscale;
  auto finish = [&](auto act) __attribute__((always_inline)) {   // (an integral_constant or an int)
#pragma unroll 2
    for (int i = 0; i < kPasses; ++i) {
      const int row = row0 + i * kRowsAtOnce;
      if (row >= rows) break;
      float4_t v = *reinterpret_cast<const float4_t *>(sums + row * T::PITCH + 4 * quad);
#pragma unroll
      for (int k = 1; k < KG; ++k) v += *reinterpret_cast<const float4_t *>(sums + (k * T::BM + row) * T::PITCH + 4 * quad);
      const float infinite = fmaf(v[0], 0.f, fmaf(v[1], 0.f, fmaf(v[2], 0.f, v[3] * 0.f)));   // NaN, or zero
      if (infinite != infinite) {
        bool bad = false;   // (what lies beyond the last column does not matter)
#pragma unroll
        for (int q = 0; q < 4; ++q) bad |= col + q < p.N && !(fabsf(v[q]) < INFINITY);
        if (bad) seen[0] = 1;
      }
      float res[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float x = v[q] * unscale + bias[q];
        res[q] = act == TFHIP_LINEAR ? x : activate(x, act, alpha[q], e.leaky_alpha);
      }
      const unsigned at = first + (unsigned)i * stride;
      if (residual) {
        const float4 r4 = as_float4(__builtin_amdgcn_raw_buffer_load_b128(rsrc_r, (int)at, 0, 0));
        res[0] += r4.x; res[1] += r4.y; res[2] += r4.z; res[3] += r4.w;
      }
      if (col + 4 <= p.N) {   // (a buffer store needs 4-byte alignment only)
        store_result4_through(rsrc_c, at, make_float4(res[0], res[1], res[2], res[3]));
      } else {
#pragma unroll
        for (int q = 0; q < 3; ++q)
          if (col + q < p.N) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(res[q]), rsrc_c, (int)at + 4 * q, 0, 0);
      }
    }
  };
  const int activation = fused ? e.activation : TFHIP_LINEAR;
  switch (activation) {
    case TFHIP_RELU: finish(std::integral_constant<int, TFHIP_RELU>()); break;
    case TFHIP_RELU6: finish(std::integral_constant<int, TFHIP_RELU6>()); break;
    case TFHIP_PRELU: finish(std::integral_constant<int, TFHIP_PRELU>()); break;
    case TFHIP_LEAKYRELU: finish(std::integral_constant<int, TFHIP_LEAKYRELU>()); break;
    default: finish(std::integral_constant<int, TFHIP_LINEAR>()); break;
  }
  lds_barrier();
  if (seen[0] == 0) return;   // (the same for the whole workgroup)

  // The sums of the high parts are right where an Inf or NaN enters them (a high part is zero for a zero only, so Inf times
  // anything else is Inf), and where none does the small products are finite, unless an operand or a sum is too large.
  __builtin_assume(tiles > 0);   // (a slice without any sums up zeros)
  unsigned most_a = 0, most_b = 0;
#pragma unroll 1
  for (int tile = 0; tile < tiles; ++tile) {
    load_a(tile);
    load_b(tile);
    // (behind a row of A lies the next one: an Inf there meets zeros of B, and counts as too large)
    const int live = kWindows ? 4 : k_end - tile_k(tile) - 4 * (lane & 7);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const uint4_t x = A_KIND == kLoadWindowsAny ? __builtin_bit_cast(uint4_t, fix_up<A_KIND>(as_float4(ra[v]), fix[v])) : ra[v];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const unsigned size = x[j] & 0x7fffffffu;
        if (size < 0x7f800000u || j >= live) most_a = max(most_a, size);
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int c = 0; c < T::XW; ++c) {
        const unsigned size = __float_as_uint(rb[j][c]) & 0x7fffffffu;
        if (size < 0x7f800000u) most_b = max(most_b, size);
      }
  }
  atomicMax(seen + 1, most_a);
  atomicMax(seen + 2, most_b);
  lds_barrier();
  // below 2^(exponent - 126) each, of fewer than 2^bits products: scaled and rounded up, a part and the sums stay below 2^128
  const int exponent_a = (int)(seen[1] >> 23), exponent_b = (int)(seen[2] >> 23), bits = 32 - __builtin_clz((unsigned)(k_end - k_begin));
  if (exponent_a <= 229 && exponent_b <= 229 && exponent_a + exponent_b + bits <= 331) {
    write_sums([](float high, float small) { return fabsf(high) < INFINITY ? high + small : high; });
  } else {
    // The tile once more, with float32 matrix instructions: lane (h, r) multiplies k + h of row r and of column 32 j + r.
    unscale = 1.f;
    const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc((void *)A, 0, (int)p.a_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc((void *)B, 0, (int)p.b_bytes, 0x00020000);
    const int row = m0 + 32 * wave + r;
    int ih = 0, iw = 0;
    unsigned off = 0;
    if (kWindows) window_row(p.conv, row, p.M, ih, iw, off);
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int q = 0; q < 16; ++q) acc[j][q] = 0.f;
#pragma unroll 1
    for (int tile = 0; tile < tiles; ++tile)
#pragma unroll 4
      for (int step = 0; step < 16; ++step) {
        const int k = tile_k(tile) + 2 * step + h;
        const int b_row = k < k_end ? filter_row<B_KIND>(p.conv, k) : -1;
        const float a = one_of_a<A_KIND>(p, rsrc_a, row, b_row < 0 ? k_end : k, k_end, ih, iw, off);
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const int x = n0 + 32 * j + r;
          const float b = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
              rsrc_b, (int)(b_row >= 0 && x < p.N ? 4u * ((unsigned)b_row * (unsigned)p.b_sk + (unsigned)x * (unsigned)(kColumns ? p.b_sx : 1)) : kNoOffset), 0, 0));
          acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(b, a, acc[j], 0, 0, 0);
        }
      }
    write_sums([](float sum, float) { return sum; });
  }
  lds_barrier();
  finish(activation);
}

}  // namespace tfhip
