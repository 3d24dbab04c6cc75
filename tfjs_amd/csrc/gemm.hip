// _FusedMatMul / BatchMatMul entry point: validates the operands, picks the
// loaders the memory layout allows and a tile shape, and launches gemm_kernel.
#include "gemm_host.h"
#include "few_rows.h"
#include "skinny_gemm.h"

using namespace tfhip;

int tfhip::launch_plain_gemm(GemmParams &p, bool transpose_a, bool transpose_b, bool vec, bool float_bits) {
  if (skinny_applies(p, transpose_a, transpose_b, vec) && tuning(kTuneNoSkinny) <= 0) return launch_skinny(p);
  if (!transpose_a && !transpose_b) {
    const int row_blocks = few_rows_blocks(p, false, vec, float_bits);
    if (row_blocks) return launch_few_rows(p, row_blocks, kLoadKAny);
    if (!float_bits) {
      const SplitChoice split = split_gemm_choice(p, kLoadKAny);
      const FewRowsForm few = few_rows_form(p, kLoadKAny, vec, split);
      if (few.row_blocks) return launch_few_rows(p, few.row_blocks, kLoadKAny, few.col_blocks);
      if (split.shape >= 0) return launch_split_gemm(split, p, kLoadKAny);
    }
  }
  if (!transpose_a && transpose_b && vec && !float_bits) {
    const SplitChoice split = split_gemm_choice(p, kLoadKAny, true);
    if (split.shape >= 0) return launch_split_gemm(split, p, kLoadKAny, true);
  }
  if (vec) {
    const int shape = choose_tile_shape(p.M, p.N, p.K, p.batch, num_cus());
    if (!transpose_a && !transpose_b) return launch_gemm_shape<kLoadKVec, kLoadXVec>(shape, p);
    if (!transpose_a && transpose_b) return launch_gemm_shape<kLoadKVec, kLoadKVec>(shape, p);
    if (transpose_a && !transpose_b) return launch_gemm_shape<kLoadXVec, kLoadXVec>(shape, p);
    return launch_gemm_shape<kLoadXVec, kLoadKVec>(shape, p);
  }
  if (!transpose_a && p.a_bytes != 0 && p.b_bytes != 0 && tuning(kTuneTile) < 0) return launch_ragged_gemm(p, transpose_b);
  return launch_gemm<64, 64, 16, 2, 2, kLoadScalar, kLoadScalar>(p);
}

namespace tfhip {
namespace {

// Device memory that belongs to the library for as long as the process lasts. Every GPU the library runs on holds a
// copy of each array, at an address of its own; in host code the names are only stand-ins for the symbols. The
// addresses are resolved once per device by setup_static_scratch (with that device current), and a launch takes those of
// the device that tfhip_init was last given.
static __device__ int few_rows_counters[kFewRowsCounters];   // one per tile that is cut, zero between launches
// The split-K partial sums of tfhip_fused_matmul_noalloc, which tfhip_fused_matmul keeps in the library's growing workspace.
static __device__ __align__(256) float scratch[TFHIP_NOALLOC_SCRATCH_BYTES / sizeof(float)];

constexpr int kMaxDevices = 64;
struct DeviceArrays {
  float *scratch;
  int *few_rows_counters;
};
DeviceArrays g_device_arrays[kMaxDevices] = {};

int resolve(const void *symbol, const char *name, int device, void **ptr) {
  const hipError_t e = hipGetSymbolAddress(ptr, symbol);
  if (e == hipSuccess && *ptr != nullptr) return kOk;
  (void)hipGetLastError();
  return fail(kHipError, "tfhip_init: hipGetSymbolAddress(%s) on device %d failed: %s", name, device, hipGetErrorString(e));
}

template <int MB, int CB, int KIND, bool ROW = false>
int launch_few_rows_shape(FewRowsArgs &q, const FewRowsCut &cut) {
  q.inner = q.M <= q.N ? cut.row_tiles : -cut.strips;
  q.splits = 1;
  q.groups_per_split = q.groups;
  std::unique_lock<std::mutex> held;
  if (cut.splits > 1) {
    held = lock_workspace();
    q.ws = static_cast<float *>(workspace((size_t)cut.tiles * cut.splits * 256 * MB * CB * sizeof(float)));
    if (q.ws) {
      q.splits = cut.splits;
      q.groups_per_split = cut.groups_per_split;
    }
  }
  // (exact: a number below 2^32 / d; d is at most about the square root of the tiles, or 256 where there are 256 workgroups)
  q.inner_magic = magic_of(abs(q.inner));
  q.splits_magic = magic_of(q.splits);
  note_splits(q.splits);
  // In a recording the slices are added by a launch of their own: a node of a graph costs a fraction of a launch, and a
  // replay then shares no counter with whatever else the program runs. The sums and their order are the same.
  q.finish_apart = q.splits > 1 && capturing();
  note_kernel("few_rows<%d, %d, %d, %s>", MB, CB, KIND, ROW ? "true" : "false");
  const dim3 grid((unsigned)(cut.tiles * q.splits)), block(64 * kFewRowsWaves);
  if (q.finish_apart) {
    TFHIP_LAUNCH((few_rows<MB, CB, KIND, ROW><<<grid, block, 0, stream()>>>(q),
                  few_rows_finish<MB, CB><<<dim3((unsigned)cut.tiles), block, 0, stream()>>>(q)));
  } else {
    TFHIP_LAUNCH((few_rows<MB, CB, KIND, ROW><<<grid, block, 0, stream()>>>(q)));
  }
  return kOk;
}

}  // namespace

int launch_few_rows(const GemmParams &p, int row_blocks, int kind, int col_blocks) {
  FewRowsArgs q = {};
  q.a = p.a; q.b = p.b; q.c = p.c;
  q.bias = p.epi.bias; q.bias_stride = p.epi.bias ? p.epi.bias_s[3] : 0;
  q.prelu = p.epi.prelu; q.prelu_stride = p.epi.prelu ? p.epi.prelu_s[3] : 0;
  q.residual = p.epi.residual;
  q.leaky_alpha = p.epi.leaky_alpha;
  q.activation = p.epi.activation;
  q.M = p.M; q.N = p.N; q.K = p.K;
  q.conv = p.conv;
  q.a_bytes = kind == kLoadKAny ? (unsigned)((long long)p.M * p.K * 4) : p.a_bytes;
  q.b_bytes = kind == kLoadKAny ? (unsigned)((long long)p.K * p.N * 4) : p.b_bytes;
  q.groups = (p.K + 15) / 16;
  q.counters = g_device_arrays[device_index()].few_rows_counters;
  const FewRowsCut narrow = few_rows_cut(p, row_blocks, 1);
  const bool one = row_blocks == 1;
  if (kind != kLoadKAny && col_blocks == 4) {
    const FewRowsCut wide = few_rows_cut(p, row_blocks, 4);
    return kind == kLoadWindows ? launch_few_rows_shape<1, 4, kLoadWindows>(q, wide) : launch_few_rows_shape<1, 4, kLoadWindowsAny>(q, wide);
  }
  if (kind == kLoadWindows) return one ? launch_few_rows_shape<1, 1, kLoadWindows>(q, narrow) : launch_few_rows_shape<2, 1, kLoadWindows>(q, narrow);
  if (kind == kLoadWindowsAny) return one ? launch_few_rows_shape<1, 1, kLoadWindowsAny>(q, narrow) : launch_few_rows_shape<2, 1, kLoadWindowsAny>(q, narrow);
  if (col_blocks ? col_blocks == 4 : few_rows_wide(narrow, row_blocks)) {
    const FewRowsCut wide = few_rows_cut(p, row_blocks, 4);
    if (p.M == 1) return launch_few_rows_shape<1, 4, kLoadKAny, true>(q, wide);
    return one ? launch_few_rows_shape<1, 4, kLoadKAny>(q, wide) : launch_few_rows_shape<2, 4, kLoadKAny>(q, wide);
  }
  if (p.M == 1) return launch_few_rows_shape<1, 1, kLoadKAny, true>(q, narrow);
  return one ? launch_few_rows_shape<1, 1, kLoadKAny>(q, narrow) : launch_few_rows_shape<2, 1, kLoadKAny>(q, narrow);
}

int setup_static_scratch(int device) {
  if (device < 0 || device >= kMaxDevices)
    return fail(kBadArgument, "tfhip_init: device %d is beyond the %d devices the table of device arrays covers", device,
                kMaxDevices);
  DeviceArrays &d = g_device_arrays[device];
  int rc = kOk;
  if (d.scratch == nullptr) rc = resolve(HIP_SYMBOL(scratch), "scratch", device, reinterpret_cast<void **>(&d.scratch));
  if (rc == kOk && d.few_rows_counters == nullptr)
    rc = resolve(HIP_SYMBOL(few_rows_counters), "few_rows_counters", device, reinterpret_cast<void **>(&d.few_rows_counters));
  return rc;
}

}  // namespace tfhip

static int fused_matmul_impl(const char *who, const float *a, const float *b, float *out, int64_t batch_a,
                             int64_t batch_b, int64_t M, int64_t N, int64_t K, int transpose_a, int transpose_b,
                             const float *bias, const int64_t bias_strides[3], int activation,
                             const float *prelu_weights, const int64_t prelu_strides[3], double leakyrelu_alpha);

extern "C" int tfhip_fused_matmul(const float *a, const float *b, float *out, int64_t batch_a, int64_t batch_b,
                                  int64_t M, int64_t N, int64_t K, int transpose_a, int transpose_b,
                                  const float *bias, const int64_t bias_strides[3], int activation,
                                  const float *prelu_weights, const int64_t prelu_strides[3],
                                  double leakyrelu_alpha) {
  return fused_matmul_impl("tfhip_fused_matmul", a, b, out, batch_a, batch_b, M, N, K, transpose_a, transpose_b, bias,
                           bias_strides, activation, prelu_weights, prelu_strides, leakyrelu_alpha);
}

extern "C" int tfhip_fused_matmul_noalloc(const float *a, const float *b, float *out, int64_t batch_a,
                                          int64_t batch_b, int64_t M, int64_t N, int64_t K, int transpose_a,
                                          int transpose_b, const float *bias, const int64_t bias_strides[3],
                                          int activation, const float *prelu_weights,
                                          const int64_t prelu_strides[3], double leakyrelu_alpha) {
  TFHIP_REQUIRE_INIT();
  float *ptr = g_device_arrays[device_index()].scratch;
  if (ptr == nullptr)
    return fail(kHipError, "tfhip_fused_matmul_noalloc: the static scratch array was not resolved on device %d",
                device_index());
  // Same kernels and the same choice of K slices as tfhip_fused_matmul (fewer where they do not fit); only the home of
  // the partial sums differs. Nothing needs clearing between calls: every element that gemm_finish or the last
  // workgroup of a few_rows tile reads was written by this call's own kernel, and the counters of few_rows are zero
  // between launches. Its slices never take more than 2 MiB (256 tiles x slices of at most 32 x 64).
  FixedWorkspace fixed(ptr, TFHIP_NOALLOC_SCRATCH_BYTES);
  return fused_matmul_impl("tfhip_fused_matmul_noalloc", a, b, out, batch_a, batch_b, M, N, K, transpose_a,
                           transpose_b, bias, bias_strides, activation, prelu_weights, prelu_strides,
                           leakyrelu_alpha);
}

static int fused_matmul_impl(const char *who, const float *a, const float *b, float *out, int64_t batch_a,
                             int64_t batch_b, int64_t M, int64_t N, int64_t K, int transpose_a, int transpose_b,
                             const float *bias, const int64_t bias_strides[3], int activation,
                             const float *prelu_weights, const int64_t prelu_strides[3], double leakyrelu_alpha) {
  TFHIP_REQUIRE_INIT();
  TFHIP_CHECK_ARG(batch_a >= 0 && batch_b >= 0 && M >= 0 && N >= 0 && K >= 0, "%s: negative dimension", who);
  const int64_t lim = 0x7fffffff;
  TFHIP_CHECK_ARG(M < lim && N < lim && K < lim && batch_a < lim && batch_b < lim,
                  "%s: dimension exceeds 2^31-1", who);
  const int64_t batch = batch_a > batch_b ? batch_a : batch_b;
  int rc = kOk;
  if (batch_a == 0 || batch_b == 0 || M == 0 || N == 0) return kOk;
  // three factors below 2^31 each can pass 2^63: bound every operand's element count before forming it
  const int64_t max_elems = int64_t(1) << 40;
  TFHIP_CHECK_ARG(product_below(max_elems, {batch_a, M, K > 0 ? K : 1}) && product_below(max_elems, {batch_b, K > 0 ? K : 1, N}) &&
                      product_below(max_elems, {batch, M, N}),
                  "%s: an operand exceeds 2^40 elements", who);
  auto live = [&](const void *ptr, int64_t elems, const char *name) {
    if (ptr != nullptr && range_is_live(ptr, (size_t)elems * 4)) return (int)kOk;
    return fail(kOutOfRange, "%s: operand '%s' (%lld elements of 4 bytes at %p) is not inside a live device buffer",
                who, name, (long long)elems, ptr);
  };
  if (K > 0) {
    if ((rc = live(a, batch_a * M * K, "a")) != kOk) return rc;
    if ((rc = live(b, batch_b * K * N, "b")) != kOk) return rc;
  }
  if ((rc = live(out, batch * M * N, "out")) != kOk) return rc;
  forget_filter_scans(out);

  GemmParams p = {};
  p.a = a; p.b = b; p.c = out;
  p.M = (int)M; p.N = (int)N; p.K = (int)K;
  p.batch = (int)batch; p.batch_a = (int)batch_a; p.batch_b = (int)batch_b;
  p.a_batch_stride = M * K; p.b_batch_stride = K * N; p.c_batch_stride = M * N;
  // strides folded as in tfjs-backend-cpu/src/kernels/BatchMatMul.ts:82-87
  p.a_sx = transpose_a ? 1 : K; p.a_sk = transpose_a ? M : 1;
  p.b_sx = transpose_b ? K : 1; p.b_sk = transpose_b ? 1 : N;
  p.ldc = N;
  const int64_t dims[3] = {batch, M, N};
  rc = fill_epilogue(p.epi, who, dims, 3, bias, bias_strides, activation, prelu_weights,
                         prelu_strides, leakyrelu_alpha, kMatmul);
  if (rc) return rc;

  const int64_t kMaxBufferBytes = 0xfffffffeLL;   // one buffer descriptor addresses at most this much
  p.a_bytes = (unsigned)(M * K * 4 <= kMaxBufferBytes ? M * K * 4 : 0);
  p.b_bytes = (unsigned)(K * N * 4 <= kMaxBufferBytes ? K * N * 4 : 0);
  p.c_bytes = (unsigned)(M * N * 4 <= kMaxBufferBytes ? M * N * 4 : 0);
  p.vec_store = N % 4 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0;
  const bool a16 = reinterpret_cast<uintptr_t>(a) % 16 == 0 && p.a_bytes != 0,
             b16 = reinterpret_cast<uintptr_t>(b) % 16 == 0 && p.b_bytes != 0;
  // float4 loads need the contiguous extent (and with it every row start and
  // batch start) to be a multiple of four elements
  const bool a_vec = a16 && K > 0 && (transpose_a ? M % 4 == 0 : K % 4 == 0) && (M * K) % 4 == 0;
  const bool b_vec = b16 && K > 0 && (transpose_b ? K % 4 == 0 : N % 4 == 0) && (K * N) % 4 == 0;
  return launch_plain_gemm(p, transpose_a != 0, transpose_b != 0, a_vec && b_vec);
}
