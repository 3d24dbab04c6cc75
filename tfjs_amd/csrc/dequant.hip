// Weight dequantisation on load: uint8 / uint16 affine and float16 -> float32.
//
// Bandwidth-bound: 1 or 2 bytes in, 4 bytes out per weight. The aligned kernel
// reads 16 bytes of codes per lane and writes four (uint8) or two (uint16 /
// float16) float4s per lane, arranged so that every wavefront load and store
// instruction covers one contiguous 1 KB span. The byte-wise kernel takes
// quantized data at any byte offset, which is how tensors sit inside a weight
// shard (tfjs-core/src/io/io_utils.ts:137-158).
//
// Arithmetic follows the reference's JavaScript exactly
// (tfjs-core/src/io/io_utils.ts:223-227): integer -> double, one double
// multiply, one double add (never fused), one round-to-nearest-even to float32.
//
// A whole weight buffer is decoded by one launch (decode_batch, behind tfhip_decode_weights);
// tfhip_dequant_* decode one tensor that is on the device already.
#include <string.h>

#include <new>
#include <vector>

#include "common.h"

namespace tfhip {
namespace {

constexpr int kThreads = 256;

__device__ __forceinline__ float affine_f32(unsigned v, double scale, double min) {
  return __double2float_rn(__dadd_rn(__dmul_rn((double)v, scale), min));
}

// Math.round (ties toward +infinity) followed by the Int32Array store's ToInt32
// (io_utils.ts:243-247).
__device__ __forceinline__ int affine_i32(unsigned v, double scale, double min) {
  const double x = __dadd_rn(__dmul_rn((double)v, scale), min);
  if (x != x || isinf(x)) return 0;
  const double f = floor(x);
  const double r = (x - f >= 0.5) ? f + 1.0 : f;
  if (fabs(r) < 9.0e15) {
    return (int)(unsigned)(unsigned long long)(long long)r;
  }
  double m = fmod(r, 4294967296.0);
  if (m < 0) m += 4294967296.0;
  return (int)(unsigned)(unsigned long long)m;
}

// float16 bit pattern -> float32 bit pattern, the value the reference's three
// lookup tables produce (io_utils.ts:645-741): exact for normals, subnormals,
// zeros and infinities; a NaN keeps its payload (m << 13) and its quiet bit is
// not forced.
__device__ __forceinline__ unsigned half_bits_to_float_bits(unsigned h) {
  const unsigned sign = (h & 0x8000u) << 16;
  const unsigned exp = (h >> 10) & 0x1fu;
  const unsigned man = h & 0x3ffu;
  if (exp == 0) {
    if (man == 0) return sign;
    // subnormal: value = man * 2^-24, normalise
    const int shift = __clz(man) - 21;  // leading zeros above bit 10
    const unsigned m = (man << shift) & 0x3ffu;
    return sign | ((unsigned)(113 - shift) << 23) | (m << 13);
  }
  if (exp == 31) return sign | 0x7f800000u | (man << 13);
  return sign | ((exp + 112u) << 23) | (man << 13);
}

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// mode 0: affine -> float32, 1: affine -> int32, 2: float16 (two-byte codes only)
template <int MODE>
__device__ __forceinline__ float decode_one(unsigned code, double scale, double min) {
  if (MODE == 2) return __uint_as_float(half_bits_to_float_bits(code));
  if (MODE == 1) return __int_as_float(affine_i32(code, scale, min));
  return affine_f32(code, scale, min);
}

// The aligned kernel. A lane reads 16 bytes of codes (16 one-byte or 8 two-byte codes), so a
// wavefront's load instruction covers 1 KB in one piece. Written out directly, lane l's results
// would be the float4s 4l..4l+3 (2l, 2l+1), a 64-byte (32-byte) stride between lanes in every store
// instruction; instead the wavefront passes its 1 KB of codes through LDS and lane l decodes the
// float4s l, 64+l, 128+l, 192+l (l, 64+l) of the span, so every store instruction also covers 1 KB
// in one piece. The LDS span belongs to one wavefront, whose LDS instructions complete in order:
// no workgroup barrier, and a wavefront's lanes all run the same number of rounds. The results are
// read and written with streaming (non-temporal) loads and stores: nothing here touches either
// twice.
template <int BYTES_PER, int MODE>
__global__ __launch_bounds__(kThreads) void dequant_vec16(const u32x4 *__restrict__ q, f32x4 *__restrict__ out,
                                                          long long groups, double scale, double min) {
  __shared__ u32x4 stage[kThreads];
  const int lane = threadIdx.x & 63, wave_first = threadIdx.x & ~63;
  u32x4 *span = stage + wave_first;
  constexpr int kOutPerGroup = BYTES_PER == 1 ? 4 : 2;   // float4s decoded from one 16-byte group
  const long long out_count = groups * kOutPerGroup;
  const long long stride = (long long)gridDim.x * kThreads;
  for (long long base = (long long)blockIdx.x * kThreads + wave_first; base < groups; base += stride) {
    const long long g = base + lane;
    u32x4 w = {0u, 0u, 0u, 0u};
    if (g < groups) w = __builtin_nontemporal_load(q + g);
    span[lane] = w;
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int k = 0; k < kOutPerGroup; ++k) {
      const long long o = base * kOutPerGroup + k * 64 + lane;
      f32x4 r;
      if (BYTES_PER == 1) {
        const unsigned c = reinterpret_cast<const unsigned *>(span)[k * 64 + lane];
        r.x = decode_one<MODE>(c & 0xffu, scale, min);
        r.y = decode_one<MODE>((c >> 8) & 0xffu, scale, min);
        r.z = decode_one<MODE>((c >> 16) & 0xffu, scale, min);
        r.w = decode_one<MODE>(c >> 24, scale, min);
      } else {
        const u32x2 c = reinterpret_cast<const u32x2 *>(span)[k * 64 + lane];
        r.x = decode_one<MODE>(c.x & 0xffffu, scale, min);
        r.y = decode_one<MODE>(c.x >> 16, scale, min);
        r.z = decode_one<MODE>(c.y & 0xffffu, scale, min);
        r.w = decode_one<MODE>(c.y >> 16, scale, min);
      }
      if (o < out_count) __builtin_nontemporal_store(r, out + o);
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// One element per lane, source read byte by byte: any source alignment, and the
// tail of the aligned kernels. MODE 0: affine f32, 1: affine i32, 2: float16.
template <int MODE>
__global__ __launch_bounds__(kThreads) void dequant_bytes(const unsigned char *__restrict__ q,
                                                          unsigned *__restrict__ out, long long first,
                                                          long long n, int bytes_per, double scale,
                                                          double min) {
  const long long stride = (long long)gridDim.x * kThreads;
  for (long long i = first + (long long)blockIdx.x * kThreads + threadIdx.x; i < n; i += stride) {
    unsigned v = q[i * bytes_per];
    if (bytes_per == 2) v |= (unsigned)q[i * 2 + 1] << 8;
    unsigned r;
    if (MODE == 2) {
      r = half_bits_to_float_bits(v);
    } else if (MODE == 1) {
      r = (unsigned)affine_i32(v, scale, min);
    } else {
      r = __float_as_uint(affine_f32(v, scale, min));
    }
    out[i] = r;
  }
}

// ---- all the tensors of a weight buffer in one launch ------------------------------------------
// The buffer sits on the device as it came from the shards, every tensor at some byte offset. What
// loading cost was not the decoding but the launches: up to three per tensor (an unaligned head, the
// 16-byte stretch, a tail), 633 us for 52 tensors of 3.4 million weights. Here a table entry describes a
// tensor, a map names the entry of every workgroup (kSpan outputs of one tensor), and any alignment of
// the codes is read by the same kernel: lane l of a wavefront decodes the four codes behind element
// 4 (64 k + l) of its span for k = 0 .. 3, a 4- or 8-byte load that the hardware takes at any byte
// address, so that loads and stores of a wavefront are contiguous without a trip through LDS. The
// codes have just been uploaded and come from the memory-side cache; the launch is bound by
// writing the results.
enum EntryKind { kPlainWords = 0, kPlainBytes = 1, kU8F32 = 2, kU8I32 = 3, kU16F32 = 4, kU16I32 = 5, kF16 = 6, kEntryKinds = 7 };
constexpr int kSpan = kThreads * 16;

struct BatchEntry {
  const unsigned char *q;
  void *out;
  long long n;            // elements (kPlainWords: 4-byte words, kPlainBytes: bytes)
  double scale, min;
  unsigned first_block;   // workgroup of the grid that takes the entry's first span
  int kind;
};

// The bytes of a code behind four of which a lane loads at once.
__host__ __device__ constexpr int code_bytes(int kind) { return kind == kPlainWords ? 4 : (kind <= kU8I32 ? 1 : 2); }

template <typename V>
__device__ __forceinline__ V load_anywhere(const unsigned char *p) {
  V v;
  __builtin_memcpy(&v, p, sizeof v);
  return v;
}

template <int KIND>
__device__ __forceinline__ float decode_code(unsigned code, double scale, double min) {
  if (KIND == kF16) return decode_one<2>(code, scale, min);
  if (KIND == kU8I32 || KIND == kU16I32) return decode_one<1>(code, scale, min);
  return decode_one<0>(code, scale, min);
}

template <int KIND>
__device__ __forceinline__ void decode_span(const BatchEntry &e, long long first) {
  constexpr int B = code_bytes(KIND);
  const int lane = threadIdx.x & 63;
  const long long base = first + (threadIdx.x >> 6) * (kSpan / 4);
  const unsigned char *q = e.q;
  if (KIND == kPlainBytes) {
    unsigned char *out = static_cast<unsigned char *>(e.out);
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const long long i = base + k * 64 + lane;
      if (i < e.n) out[i] = q[i];
    }
    return;
  }
  typedef unsigned words_t __attribute__((ext_vector_type(B)));   // four codes
  f32x4 *out4 = static_cast<f32x4 *>(e.out);   // (a block of the pool: aligned)
  words_t w[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const long long i = base + k * 256 + lane * 4;
    if (i + 4 <= e.n) w[k] = load_anywhere<words_t>(q + i * B);
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const long long i = base + k * 256 + lane * 4;
    if (i + 4 <= e.n) {
      f32x4 r;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (B == 4) r[j] = __uint_as_float(w[k][j % B]);
        else if (B == 1) r[j] = decode_code<KIND>((w[k][0] >> (8 * j)) & 0xffu, e.scale, e.min);
        else r[j] = decode_code<KIND>((w[k][(j / 2) % B] >> (16 * (j % 2))) & 0xffffu, e.scale, e.min);
      }
      __builtin_nontemporal_store(r, out4 + i / 4);
    } else {
      // the last elements of a tensor whose size is no multiple of four
      for (long long t = i; t < e.n; ++t) {
        unsigned c = 0;
        for (int b = 0; b < B; ++b) c |= (unsigned)q[t * B + b] << (8 * b);
        static_cast<float *>(e.out)[t] = B == 4 ? __uint_as_float(c) : decode_code<KIND>(c, e.scale, e.min);
      }
    }
  }
}

__global__ __launch_bounds__(kThreads) void decode_batch(const BatchEntry *__restrict__ entries,
                                                         const unsigned *__restrict__ entry_of_block) {
  const BatchEntry e = entries[entry_of_block[blockIdx.x]];
  const long long first = (long long)(blockIdx.x - e.first_block) * kSpan;
  switch (e.kind) {
    case kPlainWords: return decode_span<kPlainWords>(e, first);
    case kPlainBytes: return decode_span<kPlainBytes>(e, first);
    case kU8F32: return decode_span<kU8F32>(e, first);
    case kU8I32: return decode_span<kU8I32>(e, first);
    case kU16F32: return decode_span<kU16F32>(e, first);
    case kU16I32: return decode_span<kU16I32>(e, first);
    default: return decode_span<kF16>(e, first);
  }
}

// Plain tensors of at least this much are uploaded into their own blocks. Smaller ones pass through the temporary block of
// the codes, since each DMA costs some 8 us of its own (64 MB of plain tensors of 4 MB, 1 MB, 256 KB: 1585, 2019, 3927 us
// into their blocks, 1618, 1638, 1727 through the temporary one).
constexpr size_t kOwnUploadBytes = size_t(4) << 20;
// What passes through the temporary block at once (a larger tensor alone): it stays in the pool afterwards.
constexpr size_t kTemporaryBytes = size_t(256) << 20;
bool uploads_alone(const BatchEntry &e) { return e.kind <= kPlainBytes && (size_t)e.n * code_bytes(e.kind) >= kOwnUploadBytes; }

constexpr size_t kGap = 4096;   // bytes between two tensors of the buffer that are not worth a DMA of their own

// Tensors that pass through the temporary block together, and those among them that do not need it.
struct DecodeGroup {
  std::vector<BatchEntry> entries;             // what the launch decodes
  std::vector<size_t> code_at;                 // where an entry's codes lie in the temporary block
  std::vector<UploadSegment> codes, own;
  size_t code_bytes = 0, blocks = 0;

  size_t table_at() const { return (code_bytes + 255) & ~size_t(255); }
  size_t table_bytes() const { return entries.size() * sizeof(BatchEntry) + blocks * sizeof(unsigned); }

  void take(BatchEntry e, const char *h) {
    const size_t bytes = (size_t)e.n * tfhip::code_bytes(e.kind);
    if (bytes == 0) return;
    if (uploads_alone(e)) {
      own.push_back({static_cast<char *>(e.out), h, bytes});
      return;
    }
    e.first_block = (unsigned)blocks;
    blocks += (size_t)((e.n + kSpan - 1) / kSpan);
    // side by side (or nearly) in the buffer: one segment
    const char *end = codes.empty() ? nullptr : codes.back().h + codes.back().bytes;
    if (end == nullptr || h < end || h > end + kGap) codes.push_back({nullptr, h, 0});
    const size_t gap = (size_t)(h - codes.back().h) - codes.back().bytes;
    code_at.push_back(code_bytes + gap);
    codes.back().bytes += gap + bytes;
    code_bytes += gap + bytes;
    entries.push_back(e);
  }
};

// Uploads what the tensors of a group hold, and the table, and enqueues the launch that decodes.
int decode_group(DecodeGroup &group, char *temporary) {
  if (group.entries.empty()) return stage_upload(group.own.data(), group.own.size());
  std::vector<char> table(group.table_bytes());
  unsigned *map = reinterpret_cast<unsigned *>(table.data() + group.entries.size() * sizeof(BatchEntry));
  for (size_t i = 0; i < group.entries.size(); ++i) {
    BatchEntry &e = group.entries[i];
    e.q = reinterpret_cast<const unsigned char *>(temporary) + group.code_at[i];
    const size_t n = (size_t)((e.n + kSpan - 1) / kSpan);
    for (size_t b = 0; b < n; ++b) *map++ = (unsigned)i;
  }
  memcpy(table.data(), group.entries.data(), group.entries.size() * sizeof(BatchEntry));
  std::vector<UploadSegment> segments = group.codes;
  char *d = temporary;
  for (UploadSegment &s : segments) {
    s.d = d;
    d += s.bytes;
  }
  segments.insert(segments.end(), group.own.begin(), group.own.end());
  // the table first: its DMA runs while the first piece of the buffer is being staged
  const UploadSegment table_segment = {temporary + group.table_at(), table.data(), table.size()};
  int rc = stage_upload(&table_segment, 1);
  if (rc == kOk) rc = stage_upload(segments.data(), segments.size());
  if (rc != kOk) return rc;
  note_kernel("decode_batch");
  const BatchEntry *d_entries = reinterpret_cast<const BatchEntry *>(temporary + group.table_at());
  const unsigned *d_map = reinterpret_cast<const unsigned *>(d_entries + group.entries.size());
  decode_batch<<<dim3((unsigned)group.blocks), dim3(kThreads), 0, stream()>>>(d_entries, d_map);
  const hipError_t err = hipGetLastError();
  return err == hipSuccess ? kOk : fail(kHipError, "tfhip_decode_weights: launch failed: %s", hipGetErrorString(err));
}

// `tensors` with their blocks (`out`) allocated, at `offsets` of `host`.
int decode_all(const char *host, const std::vector<BatchEntry> &tensors, const int64_t *offsets) {
  std::vector<DecodeGroup> groups(1);
  groups[0].entries.reserve(tensors.size());   // (nearly always the only one)
  groups[0].code_at.reserve(tensors.size());
  for (size_t i = 0; i < tensors.size(); ++i) {
    const BatchEntry &e = tensors[i];
    const size_t bytes = uploads_alone(e) ? 0 : (size_t)e.n * code_bytes(e.kind);
    if (groups.back().code_bytes > 0 && groups.back().code_bytes + bytes > kTemporaryBytes) groups.emplace_back();
    groups.back().take(e, host + offsets[i]);
  }
  size_t need = 0;
  for (const DecodeGroup &group : groups) {
    if (group.blocks > 0x7fffffffu)
      return fail(kBadArgument, "tfhip_decode_weights: %zu spans exceed the grid limit", group.blocks);
    if (!group.entries.empty() && group.table_at() + group.table_bytes() > need) need = group.table_at() + group.table_bytes();
  }
  struct Block {
    void *ptr = nullptr;
    ~Block() {
      if (ptr) (void)tfhip_free(ptr);
    }
  } temporary;
  int rc = need > 0 ? tfhip_alloc(need, &temporary.ptr) : kOk;
  // (the stream is done with a group before the next one's codes arrive, and with the block before anybody is handed it)
  for (size_t i = 0; i < groups.size() && rc == kOk; ++i) rc = decode_group(groups[i], static_cast<char *>(temporary.ptr));
  return rc;
}

int grid_for(long long items, int blocks_per_cu) {
  long long blocks = (items + kThreads - 1) / kThreads;
  const long long cap = (long long)num_cus() * blocks_per_cu;
  if (blocks > cap) blocks = cap;
  return blocks < 1 ? 1 : (int)blocks;
}

template <int MODE>
int launch_bytes(const void *q, void *out, long long first, long long end, int bytes_per, double scale, double min) {
  TFHIP_LAUNCH((dequant_bytes<MODE><<<grid_for(end - first, 32), kThreads, 0, stream()>>>(
      (const unsigned char *)q, (unsigned *)out, first, end, bytes_per, scale, min)));
  return kOk;
}

int bytes_kernel(const void *q, void *out, long long first, long long end, int bytes_per, double scale, double min,
                  int mode) {
  if (first >= end) return kOk;
  if (mode == 2) return launch_bytes<2>(q, out, first, end, bytes_per, scale, min);
  if (mode == 1) return launch_bytes<1>(q, out, first, end, bytes_per, scale, min);
  return launch_bytes<0>(q, out, first, end, bytes_per, scale, min);
}

template <int BYTES_PER, int MODE>
int launch_vec16(const void *q, void *out, long long groups, double scale, double min) {
  // One round per lane: workgroups start in address order and drift apart, which spreads the
  // requests in flight over the memory channels. A grid capped at a few workgroups per compute unit,
  // every lane striding through the tensor in step with all others, measured 68% of the memory
  // bandwidth at 1.3 GB where this grid reaches 77%. (The loop in the kernel serves tensors beyond
  // 2^31 lanes.)
  const long long blocks = (groups + kThreads - 1) / kThreads;
  TFHIP_LAUNCH((dequant_vec16<BYTES_PER, MODE><<<(unsigned)(blocks > 0x3fffffLL ? 0x3fffffLL : blocks), kThreads, 0, stream()>>>(
      (const u32x4 *)q, (f32x4 *)out, groups, scale, min)));
  return kOk;
}

// mode: 0 affine f32, 1 affine i32, 2 float16.
// The 16-byte kernel takes the stretch of the tensor whose codes start on a 16-byte boundary and
// whose results do too; that needs the source on a 4-byte (one-byte codes) or 8-byte (two-byte
// codes) boundary and the output on a 16-byte one. Elements before and after that stretch, and
// tensors at any other alignment (they sit at arbitrary byte offsets inside a weight shard), go
// through the byte-wise kernel.
int launch(const void *q, int bytes_per, long long n, double scale, double min, void *out, int mode) {
  const uintptr_t qa = reinterpret_cast<uintptr_t>(q);
  const uintptr_t oa = reinterpret_cast<uintptr_t>(out);
  const int codes_per_group = 16 / bytes_per;
  long long head = 0, groups = 0;
  if (qa % (bytes_per == 1 ? 4 : 8) == 0 && oa % 16 == 0) {
    head = (long long)((16 - qa % 16) % 16) / bytes_per;   // a multiple of four elements
    if (head > n) head = n;
    groups = (n - head) / codes_per_group;
  }
  if (groups == 0) {
    note_kernel("dequant_bytes<%d>", mode);
    return bytes_kernel(q, out, 0, n, bytes_per, scale, min, mode);
  }
  note_kernel("dequant_vec16<%d, %d>", bytes_per, mode);
  int rc = bytes_kernel(q, out, 0, head, bytes_per, scale, min, mode);
  if (rc != kOk) return rc;
  const void *qv = (const unsigned char *)q + head * bytes_per;
  void *ov = (unsigned char *)out + head * 4;
  if (bytes_per == 1) {
    rc = mode == 1 ? launch_vec16<1, 1>(qv, ov, groups, scale, min) : launch_vec16<1, 0>(qv, ov, groups, scale, min);
  } else {
    rc = mode == 2 ? launch_vec16<2, 2>(qv, ov, groups, scale, min) :
         mode == 1 ? launch_vec16<2, 1>(qv, ov, groups, scale, min) : launch_vec16<2, 0>(qv, ov, groups, scale, min);
  }
  if (rc != kOk) return rc;
  return bytes_kernel(q, out, head + groups * codes_per_group, n, bytes_per, scale, min, mode);
}

}  // namespace
}  // namespace tfhip

using namespace tfhip;

extern "C" {

int tfhip_dequant_affine(const void *q, int bits, int64_t n, double scale, double min, void *out,
                         int to_int32) {
  TFHIP_REQUIRE_INIT();
  TFHIP_CHECK_ARG(bits == 8 || bits == 16, "tfhip_dequant_affine: bits must be 8 or 16, got %d", bits);
  TFHIP_CHECK_ARG(n >= 0, "tfhip_dequant_affine: negative element count");
  if (n == 0) return kOk;
  TFHIP_CHECK_RANGE(q, n, bits / 8, "q");
  TFHIP_CHECK_OUTPUT(out, n, 4, "out");
  TFHIP_CHECK_ARG(reinterpret_cast<uintptr_t>(out) % 4 == 0, "tfhip_dequant_affine: out is not 4-byte aligned");
  return launch(q, bits / 8, n, scale, min, out, to_int32 ? 1 : 0);
}

int tfhip_dequant_f16(const void *q, int64_t n, float *out) {
  TFHIP_REQUIRE_INIT();
  TFHIP_CHECK_ARG(n >= 0, "tfhip_dequant_f16: negative element count");
  if (n == 0) return kOk;
  TFHIP_CHECK_RANGE(q, n, 2, "q");
  TFHIP_CHECK_OUTPUT(out, n, 4, "out");
  TFHIP_CHECK_ARG(reinterpret_cast<uintptr_t>(out) % 4 == 0, "tfhip_dequant_f16: out is not 4-byte aligned");
  return launch(q, 2, n, 0.0, 0.0, out, 2);
}

int tfhip_decode_weights(const void *host, size_t bytes, int64_t count, const int64_t *offsets, const int64_t *elems,
                         const int *kinds, const double *scale_min, void **outs) {
  TFHIP_REQUIRE_INIT();
  TFHIP_REFUSE_WHILE_RECORDING();
  TFHIP_CHECK_ARG(count >= 0 && count < 0x7fffffff, "tfhip_decode_weights: bad tensor count");
  if (count == 0) return kOk;
  TFHIP_CHECK_ARG(offsets && elems && kinds && scale_min && outs && (host || bytes == 0), "tfhip_decode_weights: missing argument");
  std::vector<BatchEntry> entries;
  try {
    entries.resize((size_t)count);
  } catch (const std::bad_alloc &) {
    return fail(kOutOfMemory, "tfhip_decode_weights: no host memory for a table of %lld tensors", (long long)count);
  }
  for (int64_t i = 0; i < count; ++i) {
    TFHIP_CHECK_ARG(kinds[i] >= 0 && kinds[i] < kEntryKinds, "tfhip_decode_weights: tensor %lld has unknown kind %d",
                    (long long)i, kinds[i]);
    TFHIP_CHECK_ARG(offsets[i] >= 0 && elems[i] >= 0 && elems[i] <= kMaxElems && (size_t)offsets[i] <= bytes &&
                        (size_t)elems[i] * code_bytes(kinds[i]) <= bytes - (size_t)offsets[i],
                    "tfhip_decode_weights: tensor %lld reaches outside the buffer of %zu bytes", (long long)i, bytes);
    entries[i] = {nullptr, nullptr, elems[i], scale_min[2 * i], scale_min[2 * i + 1], 0, kinds[i]};
    outs[i] = nullptr;
  }
  int rc = kOk;
  for (int64_t i = 0; i < count && rc == kOk; ++i) {
    const size_t out_bytes = (size_t)elems[i] * (kinds[i] == kPlainBytes ? 1 : 4);
    rc = tfhip_alloc(out_bytes < 1 ? 1 : out_bytes, &outs[i]);
    entries[i].out = outs[i];
  }
  try {
    if (rc == kOk) rc = decode_all(static_cast<const char *>(host), entries, offsets);
  } catch (const std::bad_alloc &) {
    rc = fail(kOutOfMemory, "tfhip_decode_weights: no host memory for a table of %lld tensors", (long long)count);
  }
  for (int64_t i = 0; i < count && rc != kOk; ++i) {
    if (outs[i]) {
      (void)hipStreamSynchronize(stream());
      (void)tfhip_free(outs[i]);
    }
    outs[i] = nullptr;
  }
  return rc;
}

}  // extern "C"
