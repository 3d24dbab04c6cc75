// Products of few rows: C[M x N] = A[M x K] * B[K x N] with M up to 64, row-major, any extents and any 4-byte
// alignment (a dense layer on a handful of examples, the layers of an encoder on a short sentence).
//
// Such a product is bound by fetching B once, and at the sizes that occur (a few megabytes) by latency: the launch,
// one trip to memory, the sum. So there is no LDS stage and no k loop to speak of. A workgroup of eight wavefronts
// takes a strip of 16 CB columns, its wavefronts take k groups of 16 in turn, and each has the fetches of U groups
// out before it waits for the first.
//  * lane (g, r) (g = lane / 16, r = lane % 16) feeds k = 16 T + 4 g + j in the j-th of the four matrix instructions
//    (v_mfma_f32_16x16x4_f32) of group T: of A a float4 of row r, of B columns CB r .. CB r + CB - 1 of row k, 16
//    lanes side by side. Buffer loads need 4-byte alignment only, and what lies beyond an operand reads as zero, dword
//    by dword.
//  * the wavefronts' sums meet in LDS and are added in order.
//  * where the strips leave compute units idle, `splits` workgroups share one and cut its k: each leaves its sums in
//    scratch, the last to arrive (a counter per strip) adds them in the order of k and finishes. One launch instead of
//    two, and the bits do not depend on who is last.
#pragma once

#include <hip/hip_runtime.h>

#include "common.h"
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
  int splits, groups_per_split;
  int finish_apart;         // another launch adds the slices
  int activation;
};

constexpr int kFewRowsWaves = 8;
// Offsets no descriptor here covers, also when a smaller one is added (operands are at most 1 GiB).
constexpr unsigned kOutside = 0x80000000u, kOutsideRow = 0x40000000u;
constexpr long long kFewRowsMaxBytes = 0x40000000LL;

// Sums over wavefronts are written through to memory and read past the reader's L2, which does not see other XCDs'
// lines (a fence at device scope would write back and drop whole caches instead).
constexpr int kThrough = 16;   // sc1

// Sum over the slices (or, of one, over the wavefronts' sums in `lds`), bias, activation, residual and store of the
// outputs of a strip; `bias` and `alpha` belong to the thread's column.
template <int MB, int CB>
__device__ __forceinline__ void finish_strip(const FewRowsArgs &p, int strip, float bias, float alpha, const float *lds) {
  constexpr int W = kFewRowsWaves, kCols = 16 * CB, kOut = 256 * MB * CB;
  static_assert((64 * W) % kCols == 0, "a thread keeps its column");
  const __amdgpu_buffer_rsrc_t rsrc_ws = __builtin_amdgcn_make_buffer_rsrc(
      (void *)uniform_pointer(p.ws + (long long)strip * p.splits * kOut), 0, p.splits * kOut * 4, 0x00020000);
  const int col = strip * kCols + (int)threadIdx.x % kCols;
  const int live = min(kOut, p.M * kCols);   // elements of the strip that exist (its rows come first)
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
    const long long at = (long long)(i / kCols) * p.N + col;
    p.c[at] = p.residual ? v + p.residual[at] : v;
  }
}

template <int MB, int CB>
__global__ __launch_bounds__(64 * kFewRowsWaves) void few_rows(FewRowsArgs p) {
  constexpr int W = kFewRowsWaves;
  constexpr int U = MB + CB <= 2 ? 8 : (MB + CB <= 4 ? 4 : 2);
  constexpr int kCols = 16 * CB, kRows = 16 * MB, kOut = kCols * kRows;
  __shared__ float lds[W * kOut];
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, r = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int id = blockIdx.x;   // neighbouring strips share cache lines: each XCD (ids i, i + 8, ..) gets a contiguous band
  {
    const int per_xcd = gridDim.x / 8;
    if (per_xcd > 0 && id < per_xcd * 8) id = (id % 8) * per_xcd + id / 8;
  }
  const int strip = id / p.splits, split = id - strip * p.splits;
  const int n0 = strip * kCols;
  const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc((void *)p.a, 0, (int)p.a_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc((void *)p.b, 0, (int)p.b_bytes, 0x00020000);
  const int begin = split * p.groups_per_split + wave;
  const int end = min(p.groups, (split + 1) * p.groups_per_split);

  unsigned a_row[MB];
#pragma unroll
  for (int m = 0; m < MB; ++m) a_row[m] = 16 * m + r < p.M ? 4u * (unsigned)(16 * m + r) * (unsigned)p.K : kOutsideRow;
  const int col = n0 + CB * r;
  const unsigned b_col = col < p.N ? 4u * (unsigned)col : kOutsideRow;
  const unsigned pitch = 4u * (unsigned)p.N;

  struct Chunk {
    uint4_t a[U][MB];
    unsigned b[U][4][CB];
  };
  auto issue = [&](Chunk &c, int first) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int t = first + u * W, k = 16 * t + 4 * g;
      const unsigned ka = t < end && k < p.K ? 4u * (unsigned)k : kOutside;
#pragma unroll
      for (int m = 0; m < MB; ++m) c.a[u][m] = __builtin_amdgcn_raw_buffer_load_b128(rsrc_a, (int)(a_row[m] + ka), 0, 0);
      const unsigned kb = t < end ? (unsigned)k * pitch + b_col : kOutside;
#pragma unroll
      for (int j = 0; j < 4; ++j) {   // (rows beyond K lie beyond the descriptor)
        const int at = (int)(kb + (unsigned)j * pitch);
        if constexpr (CB == 4) {
          const uint4_t v = __builtin_amdgcn_raw_buffer_load_b128(rsrc_b, at, 0, 0);
#pragma unroll
          for (int q = 0; q < 4; ++q) c.b[u][j][q % CB] = v[q];
        } else if constexpr (CB == 2) {
          const auto v = __builtin_amdgcn_raw_buffer_load_b64(rsrc_b, at, 0, 0);
          c.b[u][j][0] = v[0];
          c.b[u][j][CB - 1] = v[1];
        } else {
          c.b[u][j][0] = __builtin_amdgcn_raw_buffer_load_b32(rsrc_b, at, 0, 0);
        }
      }
    }
  };
  float4_t acc[MB][CB];
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int q = 0; q < CB; ++q) acc[m][q] = (float4_t){0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](const Chunk &c, int first) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = 16 * (first + u * W) + 4 * g;
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int m = 0; m < MB; ++m) {
          // (the last float4 of a row may reach into the next one)
          const float av = k + j < p.K ? __uint_as_float(c.a[u][m][j]) : 0.f;
#pragma unroll
          for (int q = 0; q < CB; ++q)
            acc[m][q] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, __uint_as_float(c.b[u][j][q]), acc[m][q], 0, 0, 0);
        }
    }
  };

  Chunk cur, nxt;
  issue(cur, begin);
  // what the column this thread finishes needs
  const int my_col = n0 + tid % kCols;
  const bool col_ok = my_col < p.N;
  const float bias = p.bias && col_ok ? p.bias[(long long)my_col * p.bias_stride] : 0.f;
  const float alpha = p.activation == TFHIP_PRELU && col_ok ? p.prelu[(long long)my_col * p.prelu_stride] : 0.f;
#pragma unroll 1
  for (int t = begin; t < end; t += U * W) {
    issue(nxt, t + U * W);   // (past the end: outside, nothing is read)
    multiply(cur, t);
    cur = nxt;
  }

  // ---- the wavefronts' sums: lane holds rows 16 m + 4 g .. +3 of columns CB r + q
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int q = 0; q < CB; ++q) lds[wave * kOut + (16 * m + 4 * g + e) * kCols + CB * r + q] = acc[m][q][e];
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
        (void *)uniform_pointer(p.ws + (long long)strip * p.splits * kOut), 0, p.splits * kOut * 4, 0x00020000);
#pragma unroll 1
    for (int i = tid; i < min(kOut, p.M * kCols); i += 64 * W)
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(wave_sum(i)), rsrc_ws, 4 * (split * kOut + i), 0, kThrough);
    if (p.finish_apart) return;
    __builtin_amdgcn_s_waitcnt(0);   // the stores are in memory
    __syncthreads();
    int *last = reinterpret_cast<int *>(lds);
    if (tid == 0) {
      const int before = __hip_atomic_fetch_add(p.counters + strip, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (before == p.splits - 1) __hip_atomic_store(p.counters + strip, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *last = before == p.splits - 1;
    }
    __syncthreads();
    if (!*last) return;
  }
  finish_strip<MB, CB>(p, strip, bias, alpha, lds);
}

// The sums of the slices of one strip each, where few_rows leaves them (FewRowsArgs::finish_apart).
template <int MB, int CB>
__global__ __launch_bounds__(64 * kFewRowsWaves) void few_rows_finish(FewRowsArgs p) {
  const int col = blockIdx.x * (16 * CB) + (int)threadIdx.x % (16 * CB);
  const float bias = p.bias && col < p.N ? p.bias[(long long)col * p.bias_stride] : 0.f;
  const float alpha = p.activation == TFHIP_PRELU && col < p.N ? p.prelu[(long long)col * p.prelu_stride] : 0.f;
  finish_strip<MB, CB>(p, blockIdx.x, bias, alpha, nullptr);
}

// Whether this kernel takes the product of two row-major operands; `vec`: the tiled kernel could fetch both as float4.
// Up to 32 rows it always wins over the tiled kernel (us, 1 x 1280 x 1000: 8.0 with its finishing launch, here 6.1;
// 23 x 768 x 768: 8.0 and 6.1; 1 x 513 x 77, on its element loads: 10.7 and 4.8). With four row blocks the
// matrix instructions take as long as the fetches and every strip reads all of A: it wins where no float4 fits
// (64 x 4095 x 64: 26.0 and 8.8) or the columns are few (64 x 1280 x 1000: 11.1 and 8.8; but 64 x 768 x 3072: 8.1
// and 10.0).
inline bool few_rows_applies(const GemmParams &p, bool vec) {
  return p.batch == 1 && p.M <= 64 && p.K > 0 && p.epi.channel_operands && p.epi.addressing != kConv &&
         (p.M <= 32 || p.N <= 1024 || !vec) && (long long)p.M * p.K * 4 <= kFewRowsMaxBytes &&
         (long long)p.K * p.N * 4 <= kFewRowsMaxBytes && tuning(kTuneTile) < 0 && tuning(kTuneSplitK) < 0;
}

int launch_few_rows(const GemmParams &p);

}  // namespace tfhip
