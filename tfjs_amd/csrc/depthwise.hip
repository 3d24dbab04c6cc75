// FusedDepthwiseConv2D, NHWC float32.
//
// Bandwidth-bound (about 2 flops per byte), so no matrix cores. Four kernels:
//  * depthwise_3x3_cols: 3x3, stride 1 or 2, channel multiplier 1 (every
//    MobileNet layer). Lanes lie along an output row in memory order, one float4
//    of one column each, and walk down a chunk of rows with the input rows in a
//    register ring; no LDS, no barriers.
//  * depthwise_3x3_halo: the same shapes when a tensor is too large for 32-bit
//    buffer offsets; stages an input halo tile of 32 channels in LDS.
//  * depthwise_cols_sums: the same walk for 5x5 filters and for channel counts
//    that are no multiple of four, with running sums instead of a row ring.
//  * depthwise_generic: any filter, stride, dilation, channel multiplier.
// Each output accumulates its taps in the reference's own order (filter row,
// then filter column: tfjs-backend-cpu/src/kernels/DepthwiseConv2dNative.ts:62-95)
// with one fused multiply-add per tap, which is the reference's
// "fround(y + x*w)" per tap up to double rounding.
#include <stdlib.h>

#include "common.h"
#include "epilogue.h"

namespace tfhip {
namespace {

struct DwParams {
  const float *x;
  const float *w;
  float *y;
  int batch, in_h, in_w, in_c;
  int f_h, f_w, ch_mul;
  int stride_h, stride_w, dil_h, dil_w;
  int pad_top, pad_left, out_h, out_w;
};

// ---- general kernel: any filter, stride, dilation, channel multiplier -------
__global__ __launch_bounds__(256) void depthwise_generic(DwParams p, Epilogue e, long long total) {
  const long long out_c = (long long)p.in_c * p.ch_mul;
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += stride) {
    const long long oc = idx % out_c;
    long long t = idx / out_c;
    const int ow = (int)(t % p.out_w);
    t /= p.out_w;
    const int oh = (int)(t % p.out_h);
    const int n = (int)(t / p.out_h);
    const int d1 = (int)(oc / p.ch_mul), q = (int)(oc % p.ch_mul);
    const float *xb = p.x + (long long)n * p.in_h * p.in_w * p.in_c;
    float acc = 0.f;
    for (int r = 0; r < p.f_h; ++r) {
      const int ih = oh * p.stride_h - p.pad_top + r * p.dil_h;
      if (ih < 0 || ih >= p.in_h) continue;
      for (int s = 0; s < p.f_w; ++s) {
        const int iw = ow * p.stride_w - p.pad_left + s * p.dil_w;
        if (iw < 0 || iw >= p.in_w) continue;
        const float xv = xb[((long long)ih * p.in_w + iw) * p.in_c + d1];
        const float wv = p.w[(((long long)r * p.f_w + s) * p.in_c + d1) * p.ch_mul + q];
        acc = fmaf(xv, wv, acc);
      }
    }
    p.y[idx] = finish(e, acc, 0, 0, oc, n, oh, ow);
  }
}

// ---- 3x3, channel multiplier 1, dilation 1, stride S in both directions -----
constexpr int kCQ = 8;              // float4 channel groups per workgroup: 32 channels
constexpr int kSlots = 256 / kCQ;   // output pixels computed per pass

template <int S>
__global__ __launch_bounds__(256) void depthwise_3x3_halo(DwParams p, Epilogue e, int tile_h, int tile_w,
                                                          int tiles_w, int c4_total) {
  extern __shared__ float4 halo[];  // [in_tile_h][in_tile_w][kCQ]
  const int in_tile_h = (tile_h - 1) * S + 3;
  const int in_tile_w = (tile_w - 1) * S + 3;
  const int tile_y = blockIdx.x / tiles_w, tile_x = blockIdx.x % tiles_w;
  const int cq0 = blockIdx.y * kCQ;
  const int n = blockIdx.z;
  const int oh0 = tile_y * tile_h, ow0 = tile_x * tile_w;
  const int ih0 = oh0 * S - p.pad_top, iw0 = ow0 * S - p.pad_left;
  const float4 *x4 = reinterpret_cast<const float4 *>(p.x) + (long long)n * p.in_h * p.in_w * c4_total;
  const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);

  const int halo_items = in_tile_h * in_tile_w * kCQ;
  for (int i = threadIdx.x; i < halo_items; i += 256) {
    const int c4 = i % kCQ;
    const int pos = i / kCQ;
    const int iy = pos / in_tile_w, ix = pos % in_tile_w;
    const int ih = ih0 + iy, iw = iw0 + ix;
    float4 v = zero;
    if (ih >= 0 && ih < p.in_h && iw >= 0 && iw < p.in_w && cq0 + c4 < c4_total) {
      v = x4[((long long)ih * p.in_w + iw) * c4_total + cq0 + c4];
    }
    halo[i] = v;
  }

  const int c4 = threadIdx.x % kCQ;
  const int slot = threadIdx.x / kCQ;
  const bool c_ok = cq0 + c4 < c4_total;
  float4 w[9];
  const float4 *w4 = reinterpret_cast<const float4 *>(p.w);
#pragma unroll
  for (int t = 0; t < 9; ++t) w[t] = c_ok ? w4[(long long)t * c4_total + cq0 + c4] : zero;
  __syncthreads();
  if (!c_ok) return;

  const int c = (cq0 + c4) * 4;
  float4 *y4 = reinterpret_cast<float4 *>(p.y);
  const int pixels = tile_h * tile_w;
  for (int pix = slot; pix < pixels; pix += kSlots) {
    const int oy = pix / tile_w, ox = pix % tile_w;
    const int oh = oh0 + oy, ow = ow0 + ox;
    if (oh >= p.out_h || ow >= p.out_w) continue;
    float4 acc = zero;
#pragma unroll
    for (int r = 0; r < 3; ++r) {
#pragma unroll
      for (int s = 0; s < 3; ++s) {
        const float4 xv = halo[((oy * S + r) * in_tile_w + ox * S + s) * kCQ + c4];
        const float4 wv = w[r * 3 + s];
        acc.x = fmaf(xv.x, wv.x, acc.x);
        acc.y = fmaf(xv.y, wv.y, acc.y);
        acc.z = fmaf(xv.z, wv.z, acc.z);
        acc.w = fmaf(xv.w, wv.w, acc.w);
      }
    }
    float4 o;
    o.x = finish(e, acc.x, 0, 0, c + 0, n, oh, ow);
    o.y = finish(e, acc.y, 0, 0, c + 1, n, oh, ow);
    o.z = finish(e, acc.z, 0, 0, c + 2, n, oh, ow);
    o.w = finish(e, acc.w, 0, 0, c + 3, n, oh, ow);
    store_result4(reinterpret_cast<float *>(y4 + (((long long)n * p.out_h + oh) * p.out_w + ow) * c4_total + cq0 + c4), o);
  }
}


// ---- shared by the 3x3 kernels ------------------------------------------------------
// All accesses are buffer loads / stores over the whole tensor with 32-bit byte offsets: padding
// taps and ragged edges use an offset outside the descriptor, which reads as zero and drops
// stores, so the row loops have no branches.
constexpr unsigned kDwNoOffset = 0xffffffffu;
// Results of at least this many bytes are stored non-temporally: an L2 holds 4 MB,
// so such a result cannot wait there for its reader (measured with operands from
// memory: 51 MB 21.3 -> 20.3 us, 12 MB at stride 2 13.7 -> 12.7 us; written through
// instead, 21.6 and 13.6 us).
constexpr long long kDwStreamBytes = 8LL << 20;
typedef unsigned int dw_uint4 __attribute__((ext_vector_type(4)));
typedef unsigned int dw_uint2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float4 dw_load4(__amdgpu_buffer_rsrc_t r, unsigned off) {
#ifndef TFHIP_DW_LOAD_AUX
#define TFHIP_DW_LOAD_AUX 0
#endif
  const dw_uint4 v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, TFHIP_DW_LOAD_AUX);
  return make_float4(__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z), __uint_as_float(v.w));
}

// STREAM: a non-temporal store, for a result too large to still be in the cache
// when its reader starts (it would only push out what the reader does find there).
template <bool STREAM>
__device__ __forceinline__ void dw_store4(__amdgpu_buffer_rsrc_t r, unsigned off, float4 v) {
  dw_uint4 u;
  u.x = __float_as_uint(v.x); u.y = __float_as_uint(v.y); u.z = __float_as_uint(v.z); u.w = __float_as_uint(v.w);
  __builtin_amdgcn_raw_buffer_store_b128(u, r, (int)off, 0, (STREAM || TFHIP_NT_OUT) ? 2 : 0);
}

// Bias + activation of four channels. The common case (per-channel operands,
// relu-family activation) is a handful of instructions inline; anything else
// takes one out-of-line call so that the row pipeline stays small.
__device__ __noinline__ float4 dw_finish4_general(const Epilogue &e, float4 a, int c, int n, int oh, int ow) {
  float4 r;
  r.x = finish(e, a.x, 0, 0, c + 0, n, oh, ow);
  r.y = finish(e, a.y, 0, 0, c + 1, n, oh, ow);
  r.z = finish(e, a.z, 0, 0, c + 2, n, oh, ow);
  r.w = finish(e, a.w, 0, 0, c + 3, n, oh, ow);
  return r;
}

__device__ __forceinline__ float relu_family(float v, int act) {
  if (act == TFHIP_LINEAR) return v;
  const float t = (v > 0.f || v != v) ? v : 0.f;     // Math.max(0, x): NaN stays, -0 becomes +0
  return (act == TFHIP_RELU6 && t > 6.f) ? 6.f : t;
}

template <bool GENERAL>
__device__ __forceinline__ float4 dw_finish4(const Epilogue &e, float4 a, float4 bias4, int c, int n, int oh, int ow) {
  if (!GENERAL) {
    float4 r;
    r.x = relu_family(a.x + bias4.x, e.activation);
    r.y = relu_family(a.y + bias4.y, e.activation);
    r.z = relu_family(a.z + bias4.z, e.activation);
    r.w = relu_family(a.w + bias4.w, e.activation);
    return r;
  }
  return dw_finish4_general(e, a, c, n, oh, ow);
}

// ---- 3x3, channel multiplier 1, dilation 1, stride S: one output column per lane ----
// The lanes of a launch lie along an output row in MEMORY order: lane f of a row chunk owns
// float4 f of the row ([column][channel quad], the NHWC order), so a wavefront's store covers
// one contiguous kilobyte and its three loads per input row (the columns left of, at and right
// of its own) cover contiguous kilobytes too, each element asked for by three lanes and served
// to two of them by the vector cache. A lane walks down `rows` output rows with the input rows
// in a register ring (the three a window needs plus S fetched ahead), so a row is fetched once
// per lane; with three float4 per input row a lane is light on registers, and a launch has
// thousands of wavefronts: the bytes in flight that a memory-bound kernel needs come from
// occupancy. Taps accumulate from zero by filter row, then column, one fused multiply-add each
// (the reference's order: DepthwiseConv2dNative.ts:62-95).
// Measured on [8,112,112,96] with operands from memory, against a kernel that gave a lane a strip of
// four columns (six loads per input row, 252 workgroups, one wavefront per SIMD): 20.3 -> 18.7 us at
// stride 1, 12.7 -> 11.6 at stride 2; a plain copy of the same bytes takes 16.1 us there. What is
// left is not latency (two to four rows fetched ahead change nothing), not the rows two chunks
// both read (chunks walking towards each other, so that those rows are read at the same time:
// no change) and not arithmetic (a third of the multiply-adds: no change): reads alone take
// 9.7 us (12.7 with the two neighbour loads), stores the rest, and the two do not overlap better
// than in the copy. Staging a workgroup's row segment through LDS, so that every element is fetched
// once instead of by three lanes, gave 18.1 us; non-temporal stores are the best of the six cache
// policies a store can carry (plain and write-through: +1 us).
constexpr int kColsThreads = 64;
struct DwColsArgs {
  int c4_total;        // channel quads per pixel
  int row_quads;       // out_w * c4_total: float4 per output row
  int blocks_per_row;  // workgroups along a row
  int chunks_h, rows;  // row chunks per image, output rows per chunk
  int xcd_run;         // workgroup ids are dealt to the XCDs in contiguous runs of this many
  int by_magic;        // the next three are exact for every workgroup and lane
  unsigned block_magic, chunk_magic, c4_magic;   // magic_of blocks_per_row, chunks_h, c4_total
  unsigned x_bytes, y_bytes;
  int streamed;        // the result is stored non-temporally (kDwStreamBytes)
};

// A lane's place: float4 f (column ow, channel quad q) of a row of image n, and the chunk of rows. The divisions as
// multiplications by the host's reciprocals, the arguments in one trip: us, before and so, [8,57,43,120] 5x5/2 5.4 and 5.2,
// [8,112,112,96] 3x3 13.7 and 13.4.
__device__ __forceinline__ void cols_place(const DwParams &p, const DwColsArgs &g, int &chunk, int &n, int &f, int &ow, int &q) {
  asm volatile("" ::"s"(p.x), "s"(p.w), "s"(p.y), "s"(p.in_h), "s"(p.in_w), "s"(p.pad_top), "s"(p.pad_left), "s"(p.out_h), "s"(p.out_w),
               "s"(g.c4_total), "s"(g.row_quads), "s"(g.blocks_per_row), "s"(g.chunks_h), "s"(g.rows), "s"(g.xcd_run), "s"(g.by_magic),
               "s"(g.block_magic), "s"(g.chunk_magic), "s"(g.c4_magic), "s"(g.x_bytes), "s"(g.y_bytes));
  // workgroup ids i, i + 8, ... share an XCD: each XCD takes a contiguous run (what eight runs leave over, as it comes), so that the
  // columns and rows that neighbouring workgroups both read come from one L2 (with no runs where the count is no multiple of
  // eight, us, without and with: [14,21,75,856] 3x3 48.0 and 26.1, [6,42,95,896] 3x3 51.5 and 27.7, [14,91,22,256] 5x5/2 14.8 and 12.1,
  // [1,28,28,240] 5x5 4.5 and 3.8)
  const int id = (int)blockIdx.x, wg = id < 8 * g.xcd_run ? (id & 7) * g.xcd_run + (id >> 3) : id;
  int t;
  if (__builtin_expect(g.by_magic, 1)) {
    t = by_magic(wg, g.block_magic);
    n = by_magic(t, g.chunk_magic);
  } else {
    t = wg / g.blocks_per_row;
    n = t / g.chunks_h;
  }
  chunk = t - n * g.chunks_h;
  f = (wg - t * g.blocks_per_row) * kColsThreads + (int)threadIdx.x;
  ow = __builtin_expect(g.by_magic, 1) ? by_magic(f, g.c4_magic) : f / g.c4_total;
  q = f - ow * g.c4_total;
}

template <int S, bool GENERAL, bool STREAM>
__global__ __launch_bounds__(kColsThreads) void depthwise_3x3_cols(DwParams p, Epilogue e, DwColsArgs g) {
  constexpr int A = S;        // input rows in flight beyond the window in use: one output row ahead (two, three and
                              // four rows ahead measured the same: the launch is not short of loads in flight)
  constexpr int NB = 3 + A;   // ring of input rows
  int chunk, n, f, ow, q;
  cols_place(p, g, chunk, n, f, ow, q);
  if (f >= g.row_quads) return;
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void *)p.x, 0, (int)g.x_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t ry = __builtin_amdgcn_make_buffer_rsrc((void *)p.y, 0, (int)g.y_bytes, 0x00020000);
  const unsigned pix = (unsigned)g.c4_total * 16u;   // bytes per pixel
  const unsigned x_row = (unsigned)p.in_w * pix, y_row = (unsigned)p.out_w * pix;
  const unsigned x_img = (unsigned)n * (unsigned)p.in_h * x_row, y_img = (unsigned)n * (unsigned)p.out_h * y_row;
  const int oh0 = chunk * g.rows;
  const int rows = oh0 + g.rows <= p.out_h ? g.rows : p.out_h - oh0;
  const int rows_in = (rows - 1) * S + 3;
  const int ih0 = oh0 * S - p.pad_top;
  unsigned x_col[3];
#pragma unroll
  for (int wc = 0; wc < 3; ++wc) {
    const int iw = ow * S - p.pad_left + wc;
    x_col[wc] = (iw >= 0 && iw < p.in_w) ? (unsigned)iw * pix + (unsigned)q * 16u : kDwNoOffset;
  }
  const unsigned y_col = (unsigned)f * 16u;
  float4 ring[NB][3];
  auto fetch = [&](float4 (&row)[3], int i) __attribute__((always_inline)) {
    const int ih = ih0 + i;
    const bool row_ok = ih >= 0 && ih < p.in_h && i < rows_in;
    const unsigned row_off = x_img + (unsigned)ih * x_row;
#pragma unroll
    for (int wc = 0; wc < 3; ++wc) row[wc] = dw_load4(rx, (row_ok && x_col[wc] != kDwNoOffset) ? row_off + x_col[wc] : kDwNoOffset);
  };
  // the first window's rows, then this lane's filter taps and bias: one round trip for all of them
#pragma unroll
  for (int i = 0; i < 3 + A - S; ++i) fetch(ring[i], i);
  float4 w[9];
  const float4 *w4 = reinterpret_cast<const float4 *>(p.w) + q;
#pragma unroll
  for (int k = 0; k < 9; ++k) w[k] = w4[(long long)k * g.c4_total];
  float4 bias4 = make_float4(0.f, 0.f, 0.f, 0.f);
  const int c = q * 4;
  if (!GENERAL && e.bias) {
    const long long bs = e.bias_s[3];
    bias4 = make_float4(e.bias[(c + 0) * bs], e.bias[(c + 1) * bs], e.bias[(c + 2) * bs], e.bias[(c + 3) * bs]);
  }
  for (int o0 = 0; o0 < rows; o0 += NB) {
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      const int o = o0 + k;
      if (o < rows) {
        // input row r of the chunk lives in ring[r % NB]; o0 is a multiple of NB
#pragma unroll
        for (int j = 0; j < S; ++j) fetch(ring[(S * k + 3 + A - S + j) % NB], S * o + 3 + A - S + j);
        float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int wr = 0; wr < 3; ++wr) {
#pragma unroll
          for (int wc = 0; wc < 3; ++wc) {
            const float4 xv = ring[(S * k + wr) % NB][wc];
            const float4 wv = w[wr * 3 + wc];
            a.x = fmaf(xv.x, wv.x, a.x);
            a.y = fmaf(xv.y, wv.y, a.y);
            a.z = fmaf(xv.z, wv.z, a.z);
            a.w = fmaf(xv.w, wv.w, a.w);
          }
        }
        const int oh = oh0 + o;
        dw_store4<STREAM>(ry, y_img + (unsigned)oh * y_row + y_col, dw_finish4<GENERAL>(e, a, bias4, c, n, oh, ow));
      }
    }
  }
}

// ---- F x F, channel multiplier 1, dilation 1, stride S: the same walk with running sums ------
// The 5x5 filters, and channel counts that are no multiple of four (a lane owns VEC = 2 or 1 channels of
// one column instead of four). Keeping the five input rows of a window in registers, as the kernel above
// keeps three, would take 120 of them beside the 100 of the filter; here an input row is used the moment it
// has arrived - it adds filter row i - S o to every output row o of the lane's column that it belongs
// to - and dropped, so the lane keeps ceil(F / S) sums instead of F rows. Each sum still takes its taps
// from zero by filter row, then column, one fused multiply-add each: the bits of the general kernel.
// That one fetches every tap's input and filter value per output element (50 loads, four 64-bit divisions):
// [8,57,43,120] 5x5 stride 2, 12 MB, 22.9 us there and 5.6 here (2 us of bytes: the launch is bound by the latency
// of its few loads per lane); [3,99,74,570] 3x3, 100 MB, 147 -> 20 us.
template <int VEC>
struct DwVec {
  float v[VEC];
};

template <int VEC>
__device__ __forceinline__ DwVec<VEC> dw_load(__amdgpu_buffer_rsrc_t r, unsigned off) {
  DwVec<VEC> t;
  if (VEC == 4) {
    const float4 q = dw_load4(r, off);
    t.v[0] = q.x; t.v[1 % VEC] = q.y; t.v[2 % VEC] = q.z; t.v[3 % VEC] = q.w;
  } else if (VEC == 2) {
    const auto q = __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0);
    t.v[0] = __uint_as_float(q[0]); t.v[1 % VEC] = __uint_as_float(q[1]);
  } else {
    t.v[0] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0));
  }
  return t;
}

template <int VEC, bool STREAM>
__device__ __forceinline__ void dw_store(__amdgpu_buffer_rsrc_t r, unsigned off, const DwVec<VEC> &t) {
  constexpr int kAux = STREAM ? 2 : 0;
  if (VEC == 4) dw_store4<STREAM>(r, off, make_float4(t.v[0], t.v[1 % VEC], t.v[2 % VEC], t.v[3 % VEC]));
  else if (VEC == 2) __builtin_amdgcn_raw_buffer_store_b64((dw_uint2){__float_as_uint(t.v[0]), __float_as_uint(t.v[1 % VEC])}, r, (int)off, 0, kAux);
  else __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(t.v[0]), r, (int)off, 0, kAux);
}

// c4_total and row_quads of the arguments count units of VEC channels.
template <int F, int S, int VEC, bool GENERAL, bool STREAM>
__global__ __launch_bounds__(kColsThreads) __attribute__((amdgpu_waves_per_eu(2)))
void depthwise_cols_sums(DwParams p, Epilogue e, DwColsArgs g) {
  constexpr int NACC = (F + S - 1) / S;   // output rows in progress
  int chunk, n, f, ow, q;
  cols_place(p, g, chunk, n, f, ow, q);
  if (f >= g.row_quads) return;
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void *)p.x, 0, (int)g.x_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t ry = __builtin_amdgcn_make_buffer_rsrc((void *)p.y, 0, (int)g.y_bytes, 0x00020000);
  constexpr unsigned kUnit = 4u * VEC;
  const unsigned pix = (unsigned)g.c4_total * kUnit;   // bytes per pixel
  const unsigned x_row = (unsigned)p.in_w * pix, y_row = (unsigned)p.out_w * pix;
  const unsigned x_img = (unsigned)n * (unsigned)p.in_h * x_row, y_img = (unsigned)n * (unsigned)p.out_h * y_row;
  const int oh0 = chunk * g.rows;
  const int rows = oh0 + g.rows <= p.out_h ? g.rows : p.out_h - oh0;
  const int rows_in = (rows - 1) * S + F;
  const int ih0 = oh0 * S - p.pad_top;
  unsigned x_col[F];
#pragma unroll
  for (int wc = 0; wc < F; ++wc) {
    const int iw = ow * S - p.pad_left + wc;
    x_col[wc] = (iw >= 0 && iw < p.in_w) ? (unsigned)iw * pix + (unsigned)q * kUnit : kDwNoOffset;
  }
  const unsigned y_col = (unsigned)f * kUnit;
  auto fetch = [&](DwVec<VEC> (&row)[F], int i) __attribute__((always_inline)) {
    const int ih = ih0 + i;
    const bool row_ok = ih >= 0 && ih < p.in_h && i < rows_in;
    const unsigned row_off = x_img + (unsigned)ih * x_row;
#pragma unroll
    for (int wc = 0; wc < F; ++wc)
      row[wc] = dw_load<VEC>(rx, (row_ok && x_col[wc] != kDwNoOffset) ? row_off + x_col[wc] : kDwNoOffset);
  };
  // the first window's rows, the filter and the bias: one round trip for all of them
  DwVec<VEC> first[F - S][F], cur[S][F], nxt[S][F], w[F * F], bias = {};
#pragma unroll
  for (int i = 0; i < F - S; ++i) fetch(first[i], i);
#pragma unroll
  for (int j = 0; j < S; ++j) fetch(cur[j], F - S + j);
#pragma unroll
  for (int k = 0; k < F * F; ++k)
#pragma unroll
    for (int v = 0; v < VEC; ++v) w[k].v[v] = p.w[((long long)k * g.c4_total + q) * VEC + v];
  const int c = q * VEC;
  if (!GENERAL && e.bias) {
#pragma unroll
    for (int v = 0; v < VEC; ++v) bias.v[v] = e.bias[(long long)(c + v) * e.bias_s[3]];
  }
  DwVec<VEC> acc[NACC] = {};
  // filter row wr of an output row in progress
  auto add = [&](DwVec<VEC> &a, const DwVec<VEC> (&row)[F], int wr) __attribute__((always_inline)) {
#pragma unroll
    for (int wc = 0; wc < F; ++wc)
#pragma unroll
      for (int v = 0; v < VEC; ++v)
        a.v[v] = fmaf(row[wc].v[v], w[wr * F + wc].v[v], (wr == 0 && wc == 0) ? 0.f : a.v[v]);
  };
#pragma unroll
  for (int i = 0; i < F - S; ++i)
#pragma unroll
    for (int d = 0; d * S <= i; ++d) add(acc[d % NACC], first[i], i - d * S);
  for (int o0 = 0; o0 < rows; o0 += NACC) {
#pragma unroll
    for (int k = 0; k < NACC; ++k) {
      const int o = o0 + k;
      if (o < rows) {
        // rows S o + F - S .. S o + F - 1 complete output row o and go into the ones after it
#pragma unroll
        for (int j = 0; j < S; ++j) fetch(nxt[j], S * (o + 1) + F - S + j);
#pragma unroll
        for (int j = 0; j < S; ++j)
#pragma unroll
          for (int d = 0; d * S <= F - S + j; ++d) add(acc[(k + d) % NACC], cur[j], F - S + j - d * S);
        const int oh = oh0 + o;
        DwVec<VEC> &a = acc[k % NACC];
#pragma unroll
        for (int v = 0; v < VEC; ++v)
          a.v[v] = GENERAL ? finish(e, a.v[v], 0, 0, c + v, n, oh, ow) : relu_family(a.v[v] + bias.v[v], e.activation);
        const unsigned off = y_img + (unsigned)oh * y_row + y_col;
        dw_store<VEC, STREAM>(ry, off, a);
#pragma unroll
        for (int j = 0; j < S; ++j)
#pragma unroll
          for (int wc = 0; wc < F; ++wc) cur[j][wc] = nxt[j][wc];
      }
    }
  }
}

int balanced_tile(int extent, int max_tile) {
  const int tiles = (extent + max_tile - 1) / max_tile;
  return (extent + tiles - 1) / tiles;
}

// What a launch of the column kernels takes beside what does not depend on the rows per lane: a lane's way down its rows (`first`,
// and `step` per output row), and a compute unit's share of the wavefronts (`wave` each, `row` per input row); the root of the
// cubes' sum. Only which rows have the least of it matters: some entries are least squares in microseconds, the others (those with a
// `first` and a `step` near 1 among them) were fitted to the choice itself, to the time of the rows they choose over that of the best.
// Measured on 4378 random maps of [1-256,7-112,7-112,16-960], up to 15 row counts each, operands from memory: the rows chosen take
// 1.006 of the time of the best of them; chunks of 14 (stride 2: 8) rows, halved until there are 8 wavefronts per compute unit (5x5 of
// float4s: 2), 1.06. 43 maps are more than 3% slower than with those, 12 more than 6%. us, with those and so: [2,31,8,910] 5x5 8.4
// and 4.9, [4,7,38,744] 3x3 5.4 and 4.1, [1,49,107,119] 5x5/2 4.6 and 3.9, [6,16,49,784] 3x3 8.3 and 6.9, [3,79,32,357] 3x3 9.3 and 8.7.
// The streamed results of 3x3 at stride 2 are on a par up to 8 rows and fall behind beyond, which the estimate does not know
// ([128,112,112,96] 4 rows 143, 8 144, 12 148, 28 156).
constexpr int kMostRows = 28;
struct ColsEstimate {
  double first, step, wave, row;
  int most = kMostRows;   // rows per lane
};
// [filter 3, 5][stride 1, 2][channels per lane 1, 2, 4][result streamed]
constexpr ColsEstimate kColsEstimates[2][2][3][2] = {
    {{{{0.98, 0.907, 0.196, 0.040}, {0.36, 0.769, 0.346, 0.038}}, {{0.01, 0.973, 0.245, 0.104}, {0.06, 0.274, 0.096, 0.024}},
      {{0.20, 0.972, 0.834, 0.003}, {0.00, 0.262, 0.141, 0.027}}},
     {{{0.94, 0.025, 0.051, 0.001}, {0.94, 0.488, 0.727, 0.008}}, {{0.85, 0.896, 0.262, 0.057}, {0.29, 0.915, 0.279, 0.076}},
      {{0.98, 0.826, 0.367, 0.107}, {0.97, 0.029, 0.790, 0.020, 8}}}},
    {{{{0.42, 0.934, 0.102, 0.078}, {0.00, 0.328, 0.058, 0.023}}, {{0.00, 0.277, 0.196, 0.045}, {0.00, 0.319, 0.205, 0.039}},
      {{0.95, 0.028, 0.194, 0.000}, {0.73, 0.469, 0.516, 0.059}}},
     {{{0.46, 0.858, 0.213, 0.082}, {0.00, 0.347, 0.124, 0.028}}, {{0.87, 0.236, 0.374, 0.016}, {0.09, 0.367, 0.275, 0.046}},
      {{0.84, 0.354, 0.090, 0.078}, {0.97, 0.453, 0.373, 0.064}}}}};
struct Inverses {
  double of[kMostRows + 1] = {};
  constexpr Inverses() {
    for (int i = 1; i <= kMostRows; ++i) of[i] = 1.0 / i;
  }
};
constexpr Inverses kInverses;

// Output rows per lane: the fewest whose estimate is within 2% of the least. (Counts that do not divide a map evenly stand here as they
// are: the even count with as many chunks is smaller, so its estimate is less and it is met first. Every call goes through this: with
// integer divisions for the chunks of 28 counts it took the host 0.2 us, so 0.06.)
int rows_per_lane(const DwParams &p, int vec, bool streamed, long long blocks_per_row) {
  const ColsEstimate &e = kColsEstimates[p.f_h == 5][p.stride_h - 1][vec >> 1][streamed];
  const int most = p.out_h < e.most ? p.out_h : e.most;
  const double share = (double)blocks_per_row * p.batch / num_cus();
  const double wave = share * (e.wave + e.row * (p.f_h - p.stride_h)), row = share * e.row * p.stride_h;
  double cubes[kMostRows + 1];
  for (int rows = 1; rows <= most; ++rows) {
    const double chunks = (double)((int)((p.out_h - 0.5) * kInverses.of[rows]) + 1);   // (exact: the quotient is no nearer to a whole number than half of 1 / rows)
    const double way = e.first + e.step * rows, work = chunks * (wave + row * rows);
    cubes[rows] = way * way * way + work * work * work;
  }
  double least = cubes[1];
  for (int rows = 2; rows <= most; ++rows) least = cubes[rows] < least ? cubes[rows] : least;
  int rows = 1;
  while (cubes[rows] > 1.06 * least) ++rows;
  return rows;
}

// Fills the launch geometry of the column kernels; false when it does not fit a grid.
bool plan_cols(DwColsArgs &g, const DwParams &p, int vec) {
  g.c4_total = p.in_c / vec;
  g.row_quads = p.out_w * g.c4_total;
  g.blocks_per_row = (g.row_quads + kColsThreads - 1) / kColsThreads;
  g.x_bytes = (unsigned)((long long)p.batch * p.in_h * p.in_w * p.in_c * 4);
  g.y_bytes = (unsigned)((long long)p.batch * p.out_h * p.out_w * p.in_c * 4);
  g.streamed = g.y_bytes >= kDwStreamBytes;
  int rows = tuning(kTuneDwRows) > 0 ? tuning(kTuneDwRows) : rows_per_lane(p, vec, g.streamed, g.blocks_per_row);
  rows = rows > p.out_h ? p.out_h : rows;
  g.rows = balanced_tile(p.out_h, rows);
  g.chunks_h = (p.out_h + g.rows - 1) / g.rows;
  const long long wgs = (long long)g.blocks_per_row * g.chunks_h * p.batch;
  g.xcd_run = (int)(wgs / 8);
  const int most = g.blocks_per_row > g.chunks_h ? g.blocks_per_row : g.chunks_h;
  g.by_magic = (double)wgs * most < 4294967296.0 && ((double)g.row_quads + kColsThreads) * g.c4_total < 4294967296.0 ? 1 : 0;
  g.block_magic = magic_of(g.blocks_per_row);
  g.chunk_magic = magic_of(g.chunks_h);
  g.c4_magic = magic_of(g.c4_total);
  return wgs <= 0x7fffffffLL;
}

template <int F, int S, int VEC>
int launch_cols_sums(const DwParams &p, const Epilogue &e, const DwColsArgs &g, bool general) {
  const dim3 grid((unsigned)((long long)g.blocks_per_row * g.chunks_h * p.batch)), block(kColsThreads);
  const bool streamed = !general && g.streamed;
  note_kernel("depthwise_cols_sums<%d, %d, %d, %s, %s>", F, S, VEC, general ? "true" : "false", streamed ? "true" : "false");
  if (general) TFHIP_LAUNCH((depthwise_cols_sums<F, S, VEC, true, false><<<grid, block, 0, stream()>>>(p, e, g)));
  else if (streamed) TFHIP_LAUNCH((depthwise_cols_sums<F, S, VEC, false, true><<<grid, block, 0, stream()>>>(p, e, g)));
  else TFHIP_LAUNCH((depthwise_cols_sums<F, S, VEC, false, false><<<grid, block, 0, stream()>>>(p, e, g)));
  return kOk;
}

}  // namespace
}  // namespace tfhip

using namespace tfhip;

extern "C" int tfhip_fused_depthwise_conv2d(
    const float *x, const float *filter, float *y, int64_t batch, int64_t in_h, int64_t in_w,
    int64_t in_c, int64_t f_h, int64_t f_w, int64_t ch_mul, int64_t stride_h, int64_t stride_w,
    int64_t dilation_h, int64_t dilation_w, int64_t pad_top, int64_t pad_left, int64_t out_h,
    int64_t out_w, const float *bias, const int64_t bias_strides[4], int activation,
    const float *prelu_weights, const int64_t prelu_strides[4], double leakyrelu_alpha) {
  TFHIP_REQUIRE_INIT();
  TFHIP_CHECK_ARG(batch >= 0 && in_h > 0 && in_w > 0 && in_c > 0 && f_h > 0 && f_w > 0 && ch_mul > 0 &&
                      stride_h > 0 && stride_w > 0 && dilation_h > 0 && dilation_w > 0 && out_h >= 0 &&
                      out_w >= 0,
                  "tfhip_fused_depthwise_conv2d: non-positive dimension");
  TFHIP_CHECK_ARG(activation >= TFHIP_LINEAR && activation <= TFHIP_ELU,
                  "tfhip_fused_depthwise_conv2d: unknown activation %d", activation);
  TFHIP_CHECK_ARG(activation != TFHIP_PRELU || prelu_weights != nullptr,
                  "tfhip_fused_depthwise_conv2d: prelu activation without weights");
  const int64_t lim = 0x7fffffff;
  TFHIP_CHECK_ARG(batch < lim && in_h < lim && in_w < lim && product_below(lim, {in_c, ch_mul}) && out_h < lim && out_w < lim,
                  "tfhip_fused_depthwise_conv2d: dimension exceeds 2^31-1");
  TFHIP_CHECK_ARG(pad_top >= 0 && pad_left >= 0, "tfhip_fused_depthwise_conv2d: negative padding");
  TFHIP_CHECK_ARG(product_below(kMaxElems, {batch, in_h, in_w, in_c}) && product_below(kMaxElems, {batch, out_h, out_w, in_c, ch_mul}) &&
                      product_below(lim, {f_h, f_w, in_c, ch_mul}),
                  "tfhip_fused_depthwise_conv2d: tensor exceeds the supported range");
  const int64_t out_c = in_c * ch_mul;
  const int64_t total = batch * out_h * out_w * out_c;
  if (total == 0) return kOk;
  TFHIP_CHECK_RANGE(x, batch * in_h * in_w * in_c, 4, "x");
  TFHIP_CHECK_RANGE(filter, f_h * f_w * in_c * ch_mul, 4, "filter");
  TFHIP_CHECK_OUTPUT(y, total, 4, "y");
  const int64_t dims[4] = {batch, out_h, out_w, out_c};

  Epilogue e = {};
  e.activation = activation;
  e.leaky_alpha = leakyrelu_alpha;
  e.addressing = kConv;
  e.out_h = (int)out_h;
  e.out_w = (int)out_w;
  bool channel_only = true;
  if (bias) {
    TFHIP_CHECK_ARG(bias_strides != nullptr, "tfhip_fused_depthwise_conv2d: bias without strides");
    for (int i = 0; i < 4; ++i) {
      TFHIP_CHECK_ARG(bias_strides[i] >= 0, "tfhip_fused_depthwise_conv2d: negative bias stride");
      e.bias_s[i] = bias_strides[i];
      if (i < 3 && bias_strides[i] != 0) channel_only = false;
    }
    TFHIP_CHECK_RANGE(bias, strided_extent(dims, bias_strides, 4), 4, "bias");
    e.bias = bias;
  }
  if (activation == TFHIP_PRELU) {
    TFHIP_CHECK_ARG(prelu_strides != nullptr, "tfhip_fused_depthwise_conv2d: prelu weights without strides");
    for (int i = 0; i < 4; ++i) {
      TFHIP_CHECK_ARG(prelu_strides[i] >= 0, "tfhip_fused_depthwise_conv2d: negative prelu stride");
      e.prelu_s[i] = prelu_strides[i];
      if (i < 3 && prelu_strides[i] != 0) channel_only = false;
    }
    TFHIP_CHECK_RANGE(prelu_weights, strided_extent(dims, prelu_strides, 4), 4, "prelu_weights");
    e.prelu = prelu_weights;
  }
  if (channel_only) e.addressing = kChannel;

  DwParams p;
  p.x = x; p.w = filter; p.y = y;
  p.batch = (int)batch; p.in_h = (int)in_h; p.in_w = (int)in_w; p.in_c = (int)in_c;
  p.f_h = (int)f_h; p.f_w = (int)f_w; p.ch_mul = (int)ch_mul;
  p.stride_h = (int)stride_h; p.stride_w = (int)stride_w; p.dil_h = (int)dilation_h; p.dil_w = (int)dilation_w;
  p.pad_top = (int)pad_top; p.pad_left = (int)pad_left; p.out_h = (int)out_h; p.out_w = (int)out_w;

  const bool aligned16 = reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(filter) % 16 == 0 &&
                         reinterpret_cast<uintptr_t>(y) % 16 == 0;
  const bool aligned8 = (reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(y)) % 8 == 0;
  // The 3x3 kernels read a zero for a tap outside the image and multiply it by the filter value; the
  // reference skips the tap (DepthwiseConv2dNative.ts:72-86), which differs under a value that is not
  // finite: such a filter, where a window can reach outside, takes the general kernel, which skips.
  const bool taps_can_miss = pad_top > 0 || pad_left > 0 ||
                             (out_h - 1) * stride_h - pad_top + (f_h - 1) * dilation_h >= in_h ||
                             (out_w - 1) * stride_w - pad_left + (f_w - 1) * dilation_w >= in_w;
  bool nonfinite = false;
  if (taps_can_miss) {
    const int rc = scan_filter(filter, f_h * f_w * in_c * ch_mul, "tfhip_fused_depthwise_conv2d", &nonfinite);
    if (rc != kOk) return rc;
  }
  // square 3x3 and 5x5 filters whose windows move by one or two pixels
  const bool walk = f_h == f_w && (f_h == 3 || f_h == 5) && ch_mul == 1 && dilation_h == 1 && dilation_w == 1 &&
                    stride_h == stride_w && (stride_h == 1 || stride_h == 2) && !nonfinite;
  const bool quads = in_c % 4 == 0 && aligned16;
  const bool fast = walk && f_h == 3 && quads && batch <= 65535;
  // the row pipeline addresses both tensors with 32-bit byte offsets
  const bool fits32 = batch * in_h * in_w * in_c * 4 <= 0xfffffff0LL && total * 4 <= 0xfffffff0LL;
  if (fast && fits32 && tuning(kTuneDwHalo) <= 0) {
    const int S = (int)stride_h;
    DwColsArgs g;
    if (plan_cols(g, p, 4)) {
      const long long wgs = (long long)g.blocks_per_row * g.chunks_h * batch;
      const bool general = !(e.addressing == kChannel && activation <= TFHIP_RELU6);
      const bool streamed = !general && g.streamed;
      note_kernel("depthwise_3x3_cols<%d, %s, %s>", S, general ? "true" : "false", streamed ? "true" : "false");
      const dim3 grid((unsigned)wgs), block(kColsThreads);
      if (S == 1 && streamed)
        TFHIP_LAUNCH((depthwise_3x3_cols<1, false, true><<<grid, block, 0, stream()>>>(p, e, g)));
      else if (S == 1 && !general)
        TFHIP_LAUNCH((depthwise_3x3_cols<1, false, false><<<grid, block, 0, stream()>>>(p, e, g)));
      else if (S == 1)
        TFHIP_LAUNCH((depthwise_3x3_cols<1, true, false><<<grid, block, 0, stream()>>>(p, e, g)));
      else if (streamed)
        TFHIP_LAUNCH((depthwise_3x3_cols<2, false, true><<<grid, block, 0, stream()>>>(p, e, g)));
      else if (!general)
        TFHIP_LAUNCH((depthwise_3x3_cols<2, false, false><<<grid, block, 0, stream()>>>(p, e, g)));
      else
        TFHIP_LAUNCH((depthwise_3x3_cols<2, true, false><<<grid, block, 0, stream()>>>(p, e, g)));
      return kOk;
    }
  }
  if (walk && !fast && fits32) {
    DwColsArgs g;
    const int vec = quads ? 4 : (in_c % 2 == 0 && aligned8 ? 2 : 1);
    if (plan_cols(g, p, vec)) {
      const bool general = !(e.addressing == kChannel && activation <= TFHIP_RELU6);
      const bool one = stride_h == 1;
      if (f_h == 5) {
        if (vec == 4) return one ? launch_cols_sums<5, 1, 4>(p, e, g, general) : launch_cols_sums<5, 2, 4>(p, e, g, general);
        if (vec == 2) return one ? launch_cols_sums<5, 1, 2>(p, e, g, general) : launch_cols_sums<5, 2, 2>(p, e, g, general);
        return one ? launch_cols_sums<5, 1, 1>(p, e, g, general) : launch_cols_sums<5, 2, 1>(p, e, g, general);
      }
      if (vec == 2) return one ? launch_cols_sums<3, 1, 2>(p, e, g, general) : launch_cols_sums<3, 2, 2>(p, e, g, general);
      if (vec == 1) return one ? launch_cols_sums<3, 1, 1>(p, e, g, general) : launch_cols_sums<3, 2, 1>(p, e, g, general);
    }
  }
  if (fast) {
    const int S = (int)stride_h;
    const int c4_total = (int)(in_c / 4);
    const int tile_w = balanced_tile((int)out_w, 16);
    // about 128 output pixels per workgroup, shrunk until the halo fits 48 KiB of LDS
    int cap_h = 128 / tile_w;
    cap_h = cap_h < 1 ? 1 : (cap_h > 16 ? 16 : cap_h);
    int tile_h = balanced_tile((int)out_h, cap_h);
    size_t lds = 0;
    for (;;) {
      const int in_tile_h = (tile_h - 1) * S + 3, in_tile_w = (tile_w - 1) * S + 3;
      lds = (size_t)in_tile_h * in_tile_w * kCQ * sizeof(float4);
      if (lds <= 48 * 1024 || tile_h == 1) break;
      tile_h = balanced_tile((int)out_h, tile_h - 1);
    }
    const int tiles_h = ((int)out_h + tile_h - 1) / tile_h, tiles_w = ((int)out_w + tile_w - 1) / tile_w;
    if (lds <= 64 * 1024) {
      dim3 grid(tiles_h * tiles_w, (c4_total + kCQ - 1) / kCQ, (unsigned)batch);
      note_kernel("depthwise_3x3_halo<%d>", S);
      if (S == 1)
        TFHIP_LAUNCH((depthwise_3x3_halo<1><<<grid, 256, lds, stream()>>>(p, e, tile_h, tile_w, tiles_w, c4_total)));
      else
        TFHIP_LAUNCH((depthwise_3x3_halo<2><<<grid, 256, lds, stream()>>>(p, e, tile_h, tile_w, tiles_w, c4_total)));
      return kOk;
    }
  }
  long long blocks = (total + 255) / 256;
  const long long cap = (long long)num_cus() * 64;
  if (blocks > cap) blocks = cap;
  note_kernel("depthwise_generic");
  TFHIP_LAUNCH((depthwise_generic<<<(int)blocks, 256, 0, stream()>>>(p, e, total)));
  return kOk;
}
