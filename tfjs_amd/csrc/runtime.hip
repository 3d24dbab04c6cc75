// Library lifetime, the single stream, the pooled device allocator with its
// live-block registry, host<->device copies through pinned staging, event
// timing, and recording of a sequence of launches into a HIP graph.
#include <ctype.h>
#include <pthread.h>
#include <sched.h>
#include <string.h>
#include <unistd.h>
#if defined(__x86_64__)
#include <emmintrin.h>
#endif

#include <atomic>
#include <condition_variable>
#include <map>
#include <mutex>
#include <set>
#include <thread>
#include <unordered_map>
#include <vector>

#include "common.h"

namespace tfhip {
namespace {

// Pinned staging: a ring of slots. A transfer goes through it in pieces (an upload's of up to four slots), so that
// copying a piece between the caller's memory and its slot overlaps the DMA of the pieces before it.
constexpr size_t kSlotBytes = size_t(4) << 20;
constexpr int kSlots = 16;

// What a search of a filter for Inf / NaN found.
struct FilterScan {
  uintptr_t ptr;
  size_t elems;
  uint64_t generation;
  bool nonfinite;
};

struct RecordedGraph {
  hipGraphExec_t exec = nullptr;
  size_t nodes = 0;
  std::vector<std::pair<void *, size_t>> owned;         // block, class size
  struct Ref {
    uintptr_t base;
    size_t size;
    uint64_t generation;
  };
  std::vector<Ref> refs;   // blocks a recorded kernel names and that were live when the recording ended
  std::vector<uintptr_t> writes;   // of those, the blocks a recorded call writes: a replay changes their contents
  std::vector<FilterScan> scans;   // filters found finite, on which the choice of a recorded kernel rests
  uint64_t scans_forgotten = 0;    // Runtime::scans_forgotten when they were last found to hold
};

struct Runtime {
  bool ready = false;
  int device = 0;
  hipStream_t stream = nullptr;
  hipDeviceProp_t prop;
  // live blocks: base address -> usable size. `owned` blocks came from the pool.
  std::map<uintptr_t, size_t> live;
  std::map<uintptr_t, bool> owned;
  // Every hand-out of an address (tfhip_alloc, tfhip_register_external) gets a new
  // number: an address that was freed and handed out again is a different block.
  std::map<uintptr_t, uint64_t> generation;
  uint64_t next_generation = 1;
  std::unordered_map<size_t, std::vector<void *>> free_lists;  // by class size
  size_t live_bytes = 0, pooled_bytes = 0;
  char *staging = nullptr;              // [kSlots][kSlotBytes]
  hipEvent_t slot_done[kSlots] = {};    // the DMA that reads or writes the slot
  bool slot_busy[kSlots] = {};
  int next_slot = 0;
  void *workspace = nullptr;
  size_t workspace_bytes = 0;
  hipEvent_t events[TFHIP_MAX_EVENTS] = {};
  bool event_recorded[TFHIP_MAX_EVENTS] = {};
  // Recording (tfhip_capture_begin .. tfhip_capture_end). A recorded graph
  // replays kernels with the addresses they were given, so it keeps what it
  // needs: blocks freed while recording go to `capture_free` (reused by later
  // allocations of the same recording, then owned by the graph), and every
  // block an operand check saw is noted in `capture_refs` (checked again at
  // each replay).
  // The launches of the thread that records go to a stream of their own, which runs nothing, so that other
  // threads go on launching and copying meanwhile.
  hipStream_t capture_stream = nullptr;
  uint64_t capture_forgotten = 0;   // scans_forgotten when the recording was opened
  std::unordered_map<size_t, std::vector<void *>> capture_free;
  std::set<uintptr_t> capture_refs;
  std::set<uintptr_t> capture_writes;   // of those, the blocks some recorded call writes
  std::map<int, RecordedGraph> graphs;
  int next_graph = 1;
  std::vector<void *> retired_workspaces;  // outgrown while a graph might still name them
  std::vector<FilterScan> capture_scans;   // filters that scan_filter called finite while recording
  // Filters that were searched for Inf / NaN: block base -> scans of ranges inside that block.
  // An entry holds the generation of the block it was made for, and leaves when the block is
  // written through this library (uploads, kernel results) or freed.
  std::unordered_map<uintptr_t, std::vector<FilterScan>> filter_scans;
  uint64_t scans_forgotten = 0;   // how many times entries have left
  int *scan_flag = nullptr;   // pinned host word the scan kernel's verdict is copied to
  int *scan_flag_dev = nullptr;
};


Runtime g;
std::mutex g_mutex;
std::atomic<pthread_t> g_recorder{0};   // the thread whose launches are recorded, 0: none
bool recording() { return g_recorder.load(std::memory_order_relaxed) != 0; }
bool recording_here() {
  const pthread_t r = g_recorder.load(std::memory_order_relaxed);
  return r != 0 && r == pthread_self();
}
std::mutex g_scan_mutex;      // a search of a filter for Inf / NaN (taken before g_mutex)
std::mutex g_staging_mutex;   // the staging ring: one transfer at a time (taken before g_mutex where both are)
thread_local char g_error[1024] = "";
int g_repeat = 1;

// Size classes: eight per power of two, at least 256 bytes.
size_t class_size(size_t bytes) {
  if (bytes <= 256) return 256;
  size_t p = 256;
  while (p < bytes) p <<= 1;
  const size_t step = p >> 4;  // p/2 .. p in eight steps of p/16
  const size_t lo = p >> 1;
  size_t c = lo + ((bytes - lo + step - 1) / step) * step;
  return c < 256 ? 256 : c;
}

void give_back_locked(void *p, size_t cls) {
  g.free_lists[cls].push_back(p);
  g.pooled_bytes += cls;
}

// What was remembered about the filters of the block at `base` no longer holds.
void forget_scans_locked(uintptr_t base) {
  if (g.filter_scans.erase(base) > 0) ++g.scans_forgotten;
}

void release_pool_locked() {
  for (auto &kv : g.free_lists) {
    for (void *p : kv.second) (void)hipFree(p);
    kv.second.clear();
  }
  g.pooled_bytes = 0;
}

}  // namespace

int fail(int code, const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_error, sizeof g_error, fmt, ap);
  va_end(ap);
  return code;
}

__thread KernelLabel g_kernel_label = {};

int launch_repeat() { return g_repeat; }

int g_init_count = 0;
const char *const kTuningNames[kTuneCount] = {
#define TFHIP_TUNING_NAME(id, name) name,
    TFHIP_TUNING_KNOBS(TFHIP_TUNING_NAME)
#undef TFHIP_TUNING_NAME
};
// Every knob starts unset, whatever their number.
struct TuningTable {
  int value[kTuneCount];
  TuningTable() {
    for (int &v : value) v = -1;
  }
};
TuningTable g_tuning;
int g_tuning_changes = 0;   // (a recording keeps the kernels that the knobs chose then)
int tuning(int key) { return g_tuning.value[key]; }

void read_tuning_from_environment() {
  for (int i = 0; i < kTuneCount; ++i) {
    char env_name[64] = "TFHIP_";
    size_t at = strlen(env_name);
    for (const char *c = kTuningNames[i]; *c && at + 1 < sizeof env_name; ++c) env_name[at++] = (char)toupper((unsigned char)*c);
    env_name[at] = 0;
    const char *e = getenv(env_name);
    g_tuning.value[i] = e ? atoi(e) : -1;
  }
}

bool initialised() { return g.ready; }
int init_count() { return g_init_count; }
int device_index() { return g.device; }
hipStream_t stream() { return recording_here() ? g.capture_stream : g.stream; }
int num_cus() { return g.prop.multiProcessorCount; }

// Scratch for kernels that need device memory beyond their operands (split-K
// partial sums). One block that only grows; work on the single stream is
// ordered, so consecutive launches may share it.
// The fixed block belongs to the calling thread (the entry point that allocates
// nothing sets it for the length of its call): another thread's launches keep
// the library's own block.
thread_local void *g_fixed_ws = nullptr;
thread_local size_t g_fixed_ws_bytes = 0;
thread_local bool g_ws_fixed = false;
size_t g_workspace_allocations = 0;   // hipMalloc calls made by workspace() since tfhip_init
int g_last_splits = 0;                // K slices of the last GEMM launch

FixedWorkspace::FixedWorkspace(void *ptr, size_t bytes) {
  g_fixed_ws = ptr;
  g_fixed_ws_bytes = bytes;
  g_ws_fixed = true;
}
FixedWorkspace::~FixedWorkspace() {
  g_ws_fixed = false;
  g_fixed_ws = nullptr;
  g_fixed_ws_bytes = 0;
}
bool workspace_is_fixed() { return g_ws_fixed; }
size_t fixed_workspace_bytes() { return g_fixed_ws_bytes; }

std::mutex g_workspace_mutex;
std::unique_lock<std::mutex> lock_workspace() { return std::unique_lock<std::mutex>(g_workspace_mutex); }

void *workspace(size_t bytes) {
  if (g_ws_fixed) return bytes <= g_fixed_ws_bytes ? g_fixed_ws : nullptr;
  if (bytes <= g.workspace_bytes) return g.workspace;
  if (recording() || !g.graphs.empty()) {
    // a recorded graph may name the old block: it stays allocated until shutdown
    if (g.workspace) g.retired_workspaces.push_back(g.workspace);
  } else {
    (void)hipStreamSynchronize(g.stream);   // a launch in flight may still use the old block
    if (g.workspace) (void)hipFree(g.workspace);
  }
  g.workspace = nullptr;
  g.workspace_bytes = 0;
  const size_t want = (bytes + (size_t(1) << 24) - 1) & ~((size_t(1) << 24) - 1);
  if (hipMalloc(&g.workspace, want) != hipSuccess) {
    (void)hipGetLastError();
    g.workspace = nullptr;
    return nullptr;
  }
  g.workspace_bytes = want;
  ++g_workspace_allocations;
  return g.workspace;
}

void note_splits(int splits) { g_last_splits = splits; }

bool range_is_live(const void *p, size_t bytes) {
  std::lock_guard<std::mutex> lock(g_mutex);
  const uintptr_t a = reinterpret_cast<uintptr_t>(p);
  auto it = g.live.upper_bound(a);
  if (it == g.live.begin()) return false;
  --it;
  const bool inside = a >= it->first && a + bytes <= it->first + it->second && a + bytes >= a;
  if (inside && recording_here()) g.capture_refs.insert(it->first);
  return inside;
}

bool capturing() { return recording_here(); }

__global__ void clear_word(int *word) { *word = 0; }

// 1 in *flag when any of the n values has an all-ones exponent (Inf or NaN)
__global__ __launch_bounds__(256) void find_nonfinite(const unsigned *__restrict__ bits, long long n, int *flag) {
  const long long stride = (long long)gridDim.x * 256;
  bool hit = false;
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) hit |= (bits[i] & 0x7f800000u) == 0x7f800000u;
  if (hit) *flag = 1;   // (every writer writes the same value)
}

void forget_filter_scans(const void *p) {
  std::lock_guard<std::mutex> lock(g_mutex);
  if (g.filter_scans.empty() && !recording_here()) return;
  const uintptr_t a = reinterpret_cast<uintptr_t>(p);
  auto it = g.live.upper_bound(a);
  if (it == g.live.begin()) return;
  --it;
  if (a >= it->first + it->second) return;
  forget_scans_locked(it->first);
  // a replay writes the block again, with whatever its inputs hold then
  if (recording_here()) g.capture_writes.insert(it->first);
}

int scan_filter(const float *w, int64_t elems, const char *who, bool *nonfinite) {
  *nonfinite = false;
  if (elems <= 0) return kOk;
  const uintptr_t a = reinterpret_cast<uintptr_t>(w);
  uintptr_t base = 0;
  uint64_t generation = 0;
  {
    std::lock_guard<std::mutex> lock(g_mutex);
    auto it = g.live.upper_bound(a);
    if (it == g.live.begin()) return fail(kOutOfRange, "%s: the filter is not inside a live device buffer", who);
    --it;
    if (a + (size_t)elems * 4 > it->first + it->second)
      return fail(kOutOfRange, "%s: the filter is not inside a live device buffer", who);
    base = it->first;
    generation = g.generation[base];
    auto found = g.filter_scans.find(base);
    if (found != g.filter_scans.end()) {
      for (const FilterScan &f : found->second) {
        if (f.ptr == a && f.elems == (size_t)elems && f.generation == generation) {
          *nonfinite = f.nonfinite;
          if (recording_here() && !f.nonfinite) g.capture_scans.push_back(f);   // a replay rests on this answer
          return kOk;
        }
      }
    }
  }
  // not known yet: one small kernel and a wait for its verdict, once per filter (and one search at a time: they share
  // the word that the verdict comes back in)
  if (recording_here())
    return fail(kBadArgument,
                "%s: this filter has not been searched for Inf / NaN yet, which needs a wait for the stream; run the "
                "call once outside the recording",
                who);
  std::lock_guard<std::mutex> searching(g_scan_mutex);
  *g.scan_flag = 0;
  clear_word<<<dim3(1), dim3(1), 0, g.stream>>>(g.scan_flag_dev);
  long long blocks = (elems + 255) / 256;
  if (blocks > 1024) blocks = 1024;
  find_nonfinite<<<dim3((unsigned)blocks), dim3(256), 0, g.stream>>>(reinterpret_cast<const unsigned *>(w), elems,
                                                                     g.scan_flag_dev);
  TFHIP_CHECK_HIP(hipGetLastError());
  TFHIP_CHECK_HIP(hipMemcpyAsync(g.scan_flag, g.scan_flag_dev, sizeof(int), hipMemcpyDeviceToHost, g.stream));
  TFHIP_CHECK_HIP(hipStreamSynchronize(g.stream));
  *nonfinite = *g.scan_flag != 0;
  std::lock_guard<std::mutex> lock(g_mutex);
  // (the block may have gone while the lock was open: the entry would then never match)
  g.filter_scans[base].push_back({a, (size_t)elems, generation, *nonfinite});
  return kOk;
}

// Copies a small result straight into pinned host memory: a kernel starts within
// a few microseconds, the copy engine needs 10-15 for a transfer of any size.
__global__ __launch_bounds__(256) void copy_to_host(const float4 *__restrict__ src, float4 *__restrict__ dst, int n4) {
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n4; i += gridDim.x * 256) dst[i] = src[i];
}

// A block of at least `bytes` from the pool (g_mutex is held).
int alloc_locked(size_t bytes, void **dptr) {
  const size_t cls = class_size(bytes);
  void *p = nullptr;
  auto &fl = g.free_lists[cls];
  if (recording_here() && !g.capture_free[cls].empty()) {
    p = g.capture_free[cls].back();
    g.capture_free[cls].pop_back();
  } else if (!fl.empty()) {
    p = fl.back();
    fl.pop_back();
    g.pooled_bytes -= cls;
  } else {
    hipError_t e = hipMalloc(&p, cls);
    if (e == hipErrorOutOfMemory) {
      (void)hipGetLastError();
      (void)hipStreamSynchronize(g.stream);
      release_pool_locked();
      e = hipMalloc(&p, cls);
    }
    if (e != hipSuccess) {
      (void)hipGetLastError();
      return fail(kOutOfMemory, "tfhip_alloc: hipMalloc(%zu) failed: %s", cls, hipGetErrorString(e));
    }
  }
  g.live[reinterpret_cast<uintptr_t>(p)] = cls;
  g.owned[reinterpret_cast<uintptr_t>(p)] = true;
  g.generation[reinterpret_cast<uintptr_t>(p)] = g.next_generation++;
  g.live_bytes += cls;
  *dptr = p;
  return kOk;
}

// One turn of a wait that is expected to end within microseconds.
inline void relax() {
#if defined(__x86_64__) || defined(__i386__)
  __builtin_ia32_pause();
#else
  std::this_thread::yield();
#endif
}

// CPUs that the process may use now (a container's or a batch system's set, not the machine's).
int usable_cpus() {
  cpu_set_t set;
  if (sched_getaffinity(0, sizeof set, &set) != 0) return 1;
  return CPU_COUNT(&set);
}

// memcpy into the staging ring past the caches: the ring is not read by the host, and an ordinary store first fetches the line it
// is to overwrite (one thread, a range that no cache holds: 31 GB/s, so 44; four 91 and 126). Small copies stay in the
// cache, where the DMA finds them.
void copy_past_caches(char *d, const char *s, size_t n) {
#if defined(__x86_64__)
  constexpr size_t kSmall = size_t(64) << 10;
  if (n >= kSmall) {
    const size_t head = (64 - reinterpret_cast<uintptr_t>(d) % 64) % 64;
    memcpy(d, s, head);
    d += head;
    s += head;
    n -= head;
    for (; n >= 64; n -= 64, d += 64, s += 64) {
      const __m128i *from = reinterpret_cast<const __m128i *>(s);
      __m128i *to = reinterpret_cast<__m128i *>(d);
      const __m128i a = _mm_loadu_si128(from), b = _mm_loadu_si128(from + 1), c = _mm_loadu_si128(from + 2), e = _mm_loadu_si128(from + 3);
      _mm_stream_si128(to, a);
      _mm_stream_si128(to + 1, b);
      _mm_stream_si128(to + 2, c);
      _mm_stream_si128(to + 3, e);
    }
    _mm_sfence();
  }
#endif
  memcpy(d, s, n);
}

// memcpy by several threads, for the pieces of a transfer between the caller's memory and the staging
// ring: one thread moves 30 GB/s of a range that no cache holds, half of what the DMA engine behind it
// does (57 GB/s); four move 99. The workers, at most one per CPU beside the caller's, are started by the
// first large transfer, sleep between transfers and last as long as the process (the object is never
// destroyed: a worker may be asleep in it when the process ends). Whoever waits looks for a while
// (kSpins turns, some 100 us) and then sleeps: where the threads outnumber the CPUs, the one that is waited
// for needs the waiter's.
struct CopyCrew {
  static constexpr int kWorkers = 3, kSpins = 4000;
  static constexpr size_t kShare = size_t(256) << 10;   // the least that is worth waking a worker for
  std::mutex m;
  std::condition_variable wake, done;
  std::atomic<unsigned> round{0};   // a new value: a copy to join
  std::atomic<int> left{0};         // workers that have not finished the present one
  char *dst = nullptr;
  const char *src = nullptr;
  size_t bytes = 0, share = 0;
  bool past_caches = false;
  int workers = 0;

  CopyCrew() {
    try {
      for (int i = 1; i <= kWorkers && i < usable_cpus(); ++i) {
        std::thread([this, i] { work(i); }).detach();
        ++workers;
      }
    } catch (...) {   // a process at its thread limit: fewer workers, or none
    }
  }
  void part(int i) {
    const size_t at = share * (size_t)i;
    if (at >= bytes) return;
    const size_t n = bytes - at < share ? bytes - at : share;
    if (past_caches) copy_past_caches(dst + at, src + at, n);
    else memcpy(dst + at, src + at, n);
  }
  void work(int i) {
    unsigned seen = 0;
    for (;;) {
      // look for the next piece of the same transfer for a while before going to sleep
      for (int spin = 0; spin < kSpins && round.load(std::memory_order_acquire) == seen; ++spin) relax();
      if (round.load(std::memory_order_acquire) == seen) {
        std::unique_lock<std::mutex> lock(m);
        wake.wait(lock, [&] { return round.load(std::memory_order_acquire) != seen; });
      }
      seen = round.load(std::memory_order_acquire);
      part(i);
      if (left.fetch_sub(1, std::memory_order_acq_rel) == 1) {
        std::lock_guard<std::mutex> lock(m);
        done.notify_one();
      }
    }
  }
  // (one caller at a time: the staging ring's mutex is held)
  void copy(char *d, const char *s, size_t n, bool streamed) {
    past_caches = streamed;
    dst = d;
    src = s;
    bytes = n;
    share = (n / (size_t)(workers + 1) + 4096) & ~size_t(4095);   // (times workers + 1: at least n)
    left.store(workers, std::memory_order_relaxed);
    {
      std::lock_guard<std::mutex> lock(m);
      round.fetch_add(1, std::memory_order_release);
    }
    wake.notify_all();
    part(0);
    for (int spin = 0; spin < kSpins && left.load(std::memory_order_acquire) > 0; ++spin) relax();
    if (left.load(std::memory_order_acquire) > 0) {
      std::unique_lock<std::mutex> lock(m);
      done.wait(lock, [&] { return left.load(std::memory_order_acquire) == 0; });
    }
  }
};

// `together`: the transfer this piece belongs to is long enough for the crew to be awake anyway; `to_ring`: the host does
// not read d (a shorter transfer through the caches all the same, where the DMA finds it: 256 KB that a cache holds take 25 us,
// past the caches 28, 600 KB 37 and 43)
void host_copy(char *d, const char *s, size_t n, bool together, bool to_ring) {
  if (!together || n < 2 * CopyCrew::kShare) {
    if (together && to_ring) copy_past_caches(d, s, n);
    else memcpy(d, s, n);
    return;
  }
  static CopyCrew *crew = nullptr;   // (the staging ring's mutex is held)
  static pid_t owner = 0;            // a forked child has no such threads and starts its own
  if (owner != getpid()) {
    crew = new CopyCrew();
    owner = getpid();
  }
  crew->copy(d, s, n, to_ring);
}

// A transfer of at least this much is copied by the crew: waking it costs 10 - 15 us, and one thread takes 78 us for the
// 3.4 MB of a mobile network, four 27. (Downloads, us, one thread and four: 2 MB 126 and 92, 3.5 206 and 143, 6 316 and 186.)
constexpr size_t kCrewBytes = size_t(2) << 20;

// How much of a transfer goes into one piece: each as much as all before it (the threads fill the ring at more than twice the
// DMA's rate, so the DMA never waits for the next one), from 1 MB, which nothing overlaps, to 16 MB: between two DMAs pass
// some 9 us (85 MB in pieces of 1, 4 and 16 MB: 2225, 1690, 1533 us). What one thread copies begins with half as much
// (1 MB that no cache holds: 67 us, in one piece 71; 1.7 MB 93 and 99).
constexpr size_t kMostPiece = size_t(16) << 20;
size_t piece_bytes(size_t done, size_t left, bool together) {
  const size_t least = size_t(together ? 1024 : 512) << 10;
  const size_t want = done < least ? least : (done < kMostPiece ? done : kMostPiece);
  return left < want + want / 2 && left <= kMostPiece ? left : (left < want ? left : want);
}

// `count` free slots side by side in the ring (waits for the transfers that last used them). A transfer through several is
// noted at the first one: the ring goes round in order, so nobody takes the others before it.
int take_slots(int count, int *slot) {
  if (g.next_slot + count > kSlots) g.next_slot = 0;
  const int s = g.next_slot;
  g.next_slot = (s + count) % kSlots;
  for (int i = s; i < s + count; ++i) {
    if (g.slot_busy[i]) TFHIP_CHECK_HIP(hipEventSynchronize(g.slot_done[i]));
    g.slot_busy[i] = false;
  }
  *slot = s;
  return kOk;
}
int take_slot(int *slot) { return take_slots(1, slot); }

// Behind the wait for the ring: the library may have been shut down, and set up again, since the caller
// checked the range.
int still_live(const char *d, size_t bytes) {
  if (g.ready && range_is_live(d, bytes)) return kOk;
  return fail(kNotInitialised, "a transfer of %zu bytes: the library was shut down while it waited", bytes);
}

// A place in a list of segments to be uploaded one behind the other.
struct UploadPlace {
  const UploadSegment *seg;
  size_t off;   // in *seg
};

// Calls each(at, segment, offset in it, length) for what the next n bytes take of each segment; `at` counts from 0.
// Returns the place behind them.
template <typename F>
UploadPlace for_segments(UploadPlace p, size_t n, F each) {
  for (size_t at = 0; at < n;) {
    if (p.off == p.seg->bytes) {
      p = {p.seg + 1, 0};
      continue;
    }
    const size_t part = p.seg->bytes - p.off < n - at ? p.seg->bytes - p.off : n - at;
    each(at, *p.seg, p.off, part);
    p.off += part;
    at += part;
  }
  return p;
}

// Host memory -> device memory (checked by the caller), on the library's stream. 89 MB that no cache holds: 1.74 ms, 89% of
// the DMA's rate; 3.4 MB 121 us (in pieces of 1 and 4 MB, with ordinary stores into the ring, 2.04 ms and 144 us).
int stage_upload(const UploadSegment *segments, size_t count) {
  std::lock_guard<std::mutex> lock(g_staging_mutex);
  size_t total = 0;
  for (size_t i = 0; i < count; ++i) {
    const int alive = still_live(segments[i].d, segments[i].bytes);
    if (alive != kOk) return alive;
    total += segments[i].bytes;
  }
  const bool together = total >= kCrewBytes;
  UploadPlace place = {segments, 0};
  for (size_t done = 0; done < total;) {
    const size_t n = piece_bytes(done, total - done, together);
    int s = 0;
    const int rc = take_slots((int)((n + kSlotBytes - 1) / kSlotBytes), &s);
    if (rc != kOk) return rc;
    char *slot = g.staging + s * kSlotBytes;
    // (segments that lie side by side in host memory, as the tensors of a shard do, are copied together)
    const char *h = nullptr;
    size_t from = 0, until = 0;
    for_segments(place, n, [&](size_t at, const UploadSegment &seg, size_t off, size_t bytes) {
      if (until > from && seg.h + off != h + (at - from)) {
        host_copy(slot + from, h, until - from, together, true);
        from = at;
      }
      if (at == from) h = seg.h + off;
      until = at + bytes;
    });
    host_copy(slot + from, h, until - from, together, true);
    // (a DMA for each: two blocks side by side on the device are still two allocations)
    hipError_t e = hipSuccess;
    place = for_segments(place, n, [&](size_t at, const UploadSegment &seg, size_t off, size_t bytes) {
      if (e == hipSuccess) e = hipMemcpyAsync(seg.d + off, slot + at, bytes, hipMemcpyHostToDevice, g.stream);
    });
    if (e != hipSuccess) return fail(kHipError, "stage_upload: hipMemcpyAsync failed: %s", hipGetErrorString(e));
    TFHIP_CHECK_HIP(hipEventRecord(g.slot_done[s], g.stream));
    g.slot_busy[s] = true;
    done += n;
  }
  return kOk;
}

// Device memory -> host memory; returns when the last byte has arrived. While a piece is copied out of
// its slot the DMA fills the next ones.
int stage_download(char *h, const char *d, size_t bytes) {
  std::lock_guard<std::mutex> lock(g_staging_mutex);
  const int alive = still_live(d, bytes);
  if (alive != kOk) return alive;
  constexpr size_t kKernelCopyBytes = size_t(1) << 20;
  constexpr int kAhead = 4;
  if (bytes <= kKernelCopyBytes) {
    int s = 0;
    const int rc = take_slot(&s);
    if (rc != kOk) return rc;
    char *slot = g.staging + s * kSlotBytes;
    if (bytes % 16 == 0 && reinterpret_cast<uintptr_t>(d) % 16 == 0) {
      const int n4 = (int)(bytes / 16);
      const int blocks = (n4 + 255) / 256 < 64 ? (n4 + 255) / 256 : 64;
      copy_to_host<<<blocks, 256, 0, g.stream>>>(reinterpret_cast<const float4 *>(d), reinterpret_cast<float4 *>(slot), n4);
      TFHIP_CHECK_HIP(hipGetLastError());
    } else {
      TFHIP_CHECK_HIP(hipMemcpyAsync(slot, d, bytes, hipMemcpyDeviceToHost, g.stream));
    }
    TFHIP_CHECK_HIP(hipStreamSynchronize(g.stream));
    memcpy(h, slot, bytes);
    return kOk;
  }
  struct Piece {
    int slot;
    size_t at, n;
  } pieces[kAhead];
  int head = 0, waiting = 0;
  for (size_t issued = 0, done = 0; done < bytes;) {
    while (issued < bytes && waiting < kAhead) {
      Piece p = {0, issued, bytes - issued < kSlotBytes ? bytes - issued : kSlotBytes};
      const int rc = take_slot(&p.slot);
      if (rc != kOk) return rc;
      TFHIP_CHECK_HIP(hipMemcpyAsync(g.staging + p.slot * kSlotBytes, d + p.at, p.n, hipMemcpyDeviceToHost, g.stream));
      TFHIP_CHECK_HIP(hipEventRecord(g.slot_done[p.slot], g.stream));
      g.slot_busy[p.slot] = true;
      pieces[(head + waiting++) % kAhead] = p;
      issued += p.n;
    }
    const Piece &p = pieces[head];
    TFHIP_CHECK_HIP(hipEventSynchronize(g.slot_done[p.slot]));
    g.slot_busy[p.slot] = false;
    host_copy(h + p.at, g.staging + p.slot * kSlotBytes, p.n, bytes >= kCrewBytes, false);
    done += p.n;
    head = (head + 1) % kAhead;
    --waiting;
  }
  return kOk;
}

}  // namespace tfhip

using namespace tfhip;

extern "C" {

const char *tfhip_last_error(void) { return g_error; }

int tfhip_init(int device) {
  std::lock_guard<std::mutex> no_transfer(g_staging_mutex);
  std::lock_guard<std::mutex> lock(g_mutex);
  if (g.ready) {
    if (device == g.device) return kOk;
    return fail(kBadArgument, "tfhip_init: already initialised on device %d", g.device);
  }
  int count = 0;
  TFHIP_CHECK_HIP(hipGetDeviceCount(&count));
  TFHIP_CHECK_ARG(device >= 0 && device < count,
                  "tfhip_init: device %d not present (%d visible)", device, count);
  TFHIP_CHECK_HIP(hipSetDevice(device));
  TFHIP_CHECK_HIP(hipGetDeviceProperties(&g.prop, device));
  if (strncmp(g.prop.gcnArchName, "gfx950", 6) != 0) {
    return fail(kBadArgument,
                "tfhip_init: device %d is %s; this library carries gfx950 code only",
                device, g.prop.gcnArchName);
  }
  {
    const int rc = setup_static_scratch(device);   // this device's copy of the static scratch array
    if (rc != kOk) return rc;
  }
  TFHIP_CHECK_HIP(hipStreamCreateWithFlags(&g.stream, hipStreamNonBlocking));
  TFHIP_CHECK_HIP(hipStreamCreateWithFlags(&g.capture_stream, hipStreamNonBlocking));
  TFHIP_CHECK_HIP(hipHostMalloc(reinterpret_cast<void **>(&g.staging), kSlots * kSlotBytes, hipHostMallocDefault));
  for (int i = 0; i < kSlots; ++i) {
    TFHIP_CHECK_HIP(hipEventCreateWithFlags(&g.slot_done[i], hipEventDisableTiming));
    g.slot_busy[i] = false;
  }
  g.next_slot = 0;
  TFHIP_CHECK_HIP(hipHostMalloc(reinterpret_cast<void **>(&g.scan_flag), sizeof(int), hipHostMallocDefault));
  TFHIP_CHECK_HIP(hipMalloc(reinterpret_cast<void **>(&g.scan_flag_dev), sizeof(int)));
  g.device = device;
  ++g_init_count;
  read_tuning_from_environment();
  g.ready = true;
  return kOk;
}

int tfhip_shutdown(void) {
  std::lock_guard<std::mutex> no_transfer(g_staging_mutex);   // (one that is under way ends first)
  std::lock_guard<std::mutex> lock(g_mutex);
  if (!g.ready) return kOk;
  if (recording()) {
    hipGraph_t abandoned = nullptr;
    (void)hipStreamEndCapture(g.capture_stream, &abandoned);
    if (abandoned) (void)hipGraphDestroy(abandoned);
    (void)hipGetLastError();
    g_recorder = 0;
  }
  (void)hipStreamSynchronize(g.stream);
  for (auto &kv : g.graphs) {
    if (kv.second.exec) (void)hipGraphExecDestroy(kv.second.exec);
    for (auto &b : kv.second.owned) (void)hipFree(b.first);
  }
  g.graphs.clear();
  for (auto &kv : g.capture_free) {
    for (void *p : kv.second) (void)hipFree(p);
  }
  g.capture_free.clear();
  g.capture_refs.clear();
  g.capture_writes.clear();
  g.capture_scans.clear();
  for (void *p : g.retired_workspaces) (void)hipFree(p);
  g.retired_workspaces.clear();
  for (auto &kv : g.live) {
    if (g.owned[kv.first]) (void)hipFree(reinterpret_cast<void *>(kv.first));
  }
  g.live.clear();
  g.owned.clear();
  g.generation.clear();
  g.filter_scans.clear();
  if (g.scan_flag) (void)hipHostFree(g.scan_flag);
  if (g.scan_flag_dev) (void)hipFree(g.scan_flag_dev);
  g.scan_flag = nullptr;
  g.scan_flag_dev = nullptr;
  g.live_bytes = 0;
  release_pool_locked();
  if (g.staging) (void)hipHostFree(g.staging);
  g.staging = nullptr;
  for (int i = 0; i < kSlots; ++i) {
    if (g.slot_done[i]) (void)hipEventDestroy(g.slot_done[i]);
    g.slot_done[i] = nullptr;
    g.slot_busy[i] = false;
  }
  for (int i = 0; i < TFHIP_MAX_EVENTS; ++i) {
    if (g.events[i]) (void)hipEventDestroy(g.events[i]);
    g.events[i] = nullptr;
    g.event_recorded[i] = false;
  }
  if (g.workspace) (void)hipFree(g.workspace);
  g.workspace = nullptr;
  g.workspace_bytes = 0;
  g_workspace_allocations = 0;
  g_last_splits = 0;
  (void)hipStreamDestroy(g.stream);
  (void)hipStreamDestroy(g.capture_stream);
  g.stream = g.capture_stream = nullptr;
  g.ready = false;
  return kOk;
}

int tfhip_device_info(char *name, size_t name_len, char *arch, size_t arch_len,
                      int *cus, int *clock_khz, size_t *hbm_bytes) {
  TFHIP_REQUIRE_INIT();
  if (name && name_len) snprintf(name, name_len, "%s", g.prop.name);
  if (arch && arch_len) snprintf(arch, arch_len, "%s", g.prop.gcnArchName);
  if (cus) *cus = g.prop.multiProcessorCount;
  if (clock_khz) *clock_khz = g.prop.clockRate;
  if (hbm_bytes) *hbm_bytes = g.prop.totalGlobalMem;
  return kOk;
}

int tfhip_alloc(size_t bytes, void **dptr) {
  TFHIP_REQUIRE_INIT();
  TFHIP_CHECK_ARG(dptr != nullptr, "tfhip_alloc: dptr is NULL");
  std::lock_guard<std::mutex> lock(g_mutex);
  return alloc_locked(bytes, dptr);
}

int tfhip_free(void *dptr) {
  TFHIP_REQUIRE_INIT();
  std::lock_guard<std::mutex> lock(g_mutex);
  const uintptr_t a = reinterpret_cast<uintptr_t>(dptr);
  auto it = g.live.find(a);
  if (it == g.live.end() || !g.owned[a]) {
    return fail(kBadArgument, "tfhip_free: %p is not a live block of this library", dptr);
  }
  // Work already enqueued on the single stream runs before any later kernel
  // that is handed this block again, so the block can be reused at once.
  const size_t cls = it->second;
  g.live.erase(it);
  g.owned.erase(a);
  g.generation.erase(a);
  forget_scans_locked(a);
  g.live_bytes -= cls;
  // (another thread may free a block that the graph names as well)
  if (recording_here() || (recording() && g.capture_refs.count(a) > 0)) {
    g.capture_free[cls].push_back(dptr);   // the graph being recorded names it: the graph keeps it
  } else {
    give_back_locked(dptr, cls);
  }
  return kOk;
}

int tfhip_register_external(void *dptr, size_t bytes) {
  TFHIP_REQUIRE_INIT();
  TFHIP_CHECK_ARG(dptr != nullptr && bytes > 0, "tfhip_register_external: empty range");
  std::lock_guard<std::mutex> lock(g_mutex);
  g.live[reinterpret_cast<uintptr_t>(dptr)] = bytes;
  g.owned[reinterpret_cast<uintptr_t>(dptr)] = false;
  g.generation[reinterpret_cast<uintptr_t>(dptr)] = g.next_generation++;
  return kOk;
}

int tfhip_unregister_external(void *dptr) {
  TFHIP_REQUIRE_INIT();
  std::lock_guard<std::mutex> lock(g_mutex);
  const uintptr_t a = reinterpret_cast<uintptr_t>(dptr);
  auto it = g.live.find(a);
  if (it == g.live.end() || g.owned[a]) {
    return fail(kBadArgument, "tfhip_unregister_external: %p was not registered", dptr);
  }
  g.live.erase(it);
  g.owned.erase(a);
  g.generation.erase(a);
  forget_scans_locked(a);
  return kOk;
}

int tfhip_memory_info(size_t *live, size_t *live_bytes, size_t *pooled_bytes) {
  TFHIP_REQUIRE_INIT();
  std::lock_guard<std::mutex> lock(g_mutex);
  size_t n = 0;
  for (auto &kv : g.owned) n += kv.second ? 1 : 0;
  if (live) *live = n;
  if (live_bytes) *live_bytes = g.live_bytes;
  if (pooled_bytes) *pooled_bytes = g.pooled_bytes;
  return kOk;
}

int tfhip_workspace_info(size_t *bytes, size_t *allocations, int *last_splits) {
  TFHIP_REQUIRE_INIT();
  if (bytes) *bytes = g.workspace_bytes;
  if (allocations) *allocations = g_workspace_allocations;
  if (last_splits) *last_splits = g_last_splits;
  return kOk;
}

int tfhip_filter_is_finite(const float *filter, int64_t elems, int *finite) {
  TFHIP_REQUIRE_INIT();
  TFHIP_CHECK_ARG(finite != nullptr && elems >= 0, "tfhip_filter_is_finite: bad argument");
  bool nonfinite = false;
  const int rc = scan_filter(filter, elems, "tfhip_filter_is_finite", &nonfinite);
  if (rc != kOk) return rc;
  *finite = nonfinite ? 0 : 1;
  return kOk;
}

int tfhip_upload(void *dst, size_t dst_offset, const void *host, size_t bytes) {
  TFHIP_REQUIRE_INIT();
  TFHIP_REFUSE_WHILE_RECORDING();
  if (bytes == 0) return kOk;
  TFHIP_CHECK_ARG(host != nullptr, "tfhip_upload: host pointer is NULL");
  char *d = static_cast<char *>(dst) + dst_offset;
  TFHIP_CHECK_OUTPUT(d, bytes, 1, "dst");
  const UploadSegment whole = {d, static_cast<const char *>(host), bytes};
  return stage_upload(&whole, 1);
}

int tfhip_download(void *host, const void *src, size_t src_offset, size_t bytes) {
  TFHIP_REQUIRE_INIT();
  TFHIP_REFUSE_WHILE_RECORDING();
  if (bytes == 0) {
    TFHIP_CHECK_HIP(hipStreamSynchronize(g.stream));
    return kOk;
  }
  TFHIP_CHECK_ARG(host != nullptr, "tfhip_download: host pointer is NULL");
  const char *s = static_cast<const char *>(src) + src_offset;
  TFHIP_CHECK_RANGE(s, bytes, 1, "src");
  return stage_download(static_cast<char *>(host), s, bytes);
}

int tfhip_set_tuning(const char *name, int value) {
  for (int i = 0; name && i < kTuneCount; ++i) {
    if (strcmp(name, kTuningNames[i]) == 0) {
      if (value < 0) value = -1;
      if (g_tuning.value[i] != value) ++g_tuning_changes;
      g_tuning.value[i] = value;
      return kOk;
    }
  }
  return fail(kBadArgument, "tfhip_set_tuning: unknown knob '%s'", name ? name : "(null)");
}

int tfhip_tuning_changes(int *changes) {
  TFHIP_CHECK_ARG(changes != nullptr, "tfhip_tuning_changes: changes is NULL");
  *changes = g_tuning_changes;
  return kOk;
}

int tfhip_set_launch_repeat(int n) {
  if (n < 1 || n > 100000) return fail(kBadArgument, "tfhip_set_launch_repeat: %d not in 1..100000", n);
  g_repeat = n;
  return kOk;
}

int tfhip_last_kernel(char *name, size_t name_len) {
  if (name && name_len) {
    if (g_kernel_label.print) g_kernel_label.print(name, name_len, g_kernel_label);
    else name[0] = 0;
  }
  return kOk;
}

int tfhip_sync(void) {
  TFHIP_REQUIRE_INIT();
  TFHIP_REFUSE_WHILE_RECORDING();
  TFHIP_CHECK_HIP(hipStreamSynchronize(g.stream));
  return kOk;
}

int tfhip_event_record(int slot) {
  TFHIP_REQUIRE_INIT();
  TFHIP_REFUSE_WHILE_RECORDING();
  TFHIP_CHECK_ARG(slot >= 0 && slot < TFHIP_MAX_EVENTS, "tfhip_event_record: slot %d out of range", slot);
  if (!g.events[slot]) TFHIP_CHECK_HIP(hipEventCreate(&g.events[slot]));
  TFHIP_CHECK_HIP(hipEventRecord(g.events[slot], g.stream));
  g.event_recorded[slot] = true;
  return kOk;
}

int tfhip_event_elapsed(int start_slot, int end_slot, float *ms) {
  TFHIP_REQUIRE_INIT();
  TFHIP_REFUSE_WHILE_RECORDING();
  TFHIP_CHECK_ARG(start_slot >= 0 && start_slot < TFHIP_MAX_EVENTS && end_slot >= 0 &&
                      end_slot < TFHIP_MAX_EVENTS && ms != nullptr,
                  "tfhip_event_elapsed: bad arguments");
  TFHIP_CHECK_ARG(g.event_recorded[start_slot] && g.event_recorded[end_slot],
                  "tfhip_event_elapsed: slot %d or %d was never recorded", start_slot, end_slot);
  TFHIP_CHECK_HIP(hipEventSynchronize(g.events[end_slot]));
  TFHIP_CHECK_HIP(hipEventElapsedTime(ms, g.events[start_slot], g.events[end_slot]));
  return kOk;
}

int tfhip_capture_begin(void) {
  TFHIP_REQUIRE_INIT();
  std::lock_guard<std::mutex> lock(g_mutex);
  TFHIP_CHECK_ARG(!recording(), "tfhip_capture_begin: a recording is already open");
  // Relaxed mode: an allocation that misses the pool may still call hipMalloc.
  TFHIP_CHECK_HIP(hipStreamBeginCapture(g.capture_stream, hipStreamCaptureModeRelaxed));
  g_recorder = pthread_self();
  g.capture_forgotten = g.scans_forgotten;
  g.capture_refs.clear();
  g.capture_writes.clear();
  g.capture_scans.clear();
  return kOk;
}

int tfhip_capture_end(int *graph_id, int *nodes) {
  TFHIP_REQUIRE_INIT();
  std::lock_guard<std::mutex> lock(g_mutex);
  TFHIP_CHECK_ARG(recording(), "tfhip_capture_end: no recording is open");
  g_recorder = 0;
  hipGraph_t graph = nullptr;
  hipError_t e = hipStreamEndCapture(g.capture_stream, &graph);
  RecordedGraph rec;
  if (e == hipSuccess) {
    (void)hipGraphGetNodes(graph, nullptr, &rec.nodes);
    if (graph_id != nullptr) e = hipGraphInstantiate(&rec.exec, graph, nullptr, nullptr, 0);
  }
  if (graph) (void)hipGraphDestroy(graph);
  if (e != hipSuccess || graph_id == nullptr) {
    // nothing will replay: the blocks set aside for the graph return to the pool
    (void)hipGetLastError();
    for (auto &kv : g.capture_free) {
      for (void *p : kv.second) give_back_locked(p, kv.first);
    }
    g.capture_free.clear();
    g.capture_refs.clear();
    g.capture_writes.clear();
    g.capture_scans.clear();
    if (e != hipSuccess) return fail(kHipError, "tfhip_capture_end: %s", hipGetErrorString(e));
    if (nodes) *nodes = (int)rec.nodes;
    return kOk;
  }
  for (auto &kv : g.capture_free) {
    for (void *p : kv.second) {
      rec.owned.emplace_back(p, kv.first);
      g.capture_refs.erase(reinterpret_cast<uintptr_t>(p));
    }
  }
  g.capture_free.clear();
  for (uintptr_t base : g.capture_refs) {
    auto it = g.live.find(base);
    if (it != g.live.end()) {
      rec.refs.push_back({base, it->second, g.generation[base]});
      if (g.capture_writes.count(base)) rec.writes.push_back(base);
    }
  }
  rec.scans = std::move(g.capture_scans);
  rec.scans_forgotten = g.capture_forgotten;
  g.capture_refs.clear();
  g.capture_writes.clear();
  g.capture_scans.clear();
  const int id = g.next_graph++;
  if (nodes) *nodes = (int)rec.nodes;
  g.graphs[id] = std::move(rec);
  *graph_id = id;
  return kOk;
}

int tfhip_graph_launch(int graph_id) {
  TFHIP_REQUIRE_INIT();
  std::vector<FilterScan> scans;   // to be compared before the replay
  uint64_t forgotten = 0;
  for (;;) {
    std::unique_lock<std::mutex> lock(g_mutex);
    TFHIP_CHECK_ARG(!recording_here(), "tfhip_graph_launch: a recording is open");
    auto it = g.graphs.find(graph_id);
    TFHIP_CHECK_ARG(it != g.graphs.end(), "tfhip_graph_launch: no graph %d", graph_id);
    RecordedGraph &rec = it->second;
    for (auto &r : rec.refs) {
      // the same address, size AND hand-out: a block that was freed and handed out again
      // at the same address belongs to someone else now
      auto b = g.live.find(r.base);
      auto gen = g.generation.find(r.base);
      if (b == g.live.end() || b->second != r.size || gen == g.generation.end() || gen->second != r.generation) {
        return fail(kOutOfRange,
                    "tfhip_graph_launch: graph %d names the device buffer at %p (%zu bytes), which has been freed since it was recorded",
                    graph_id, reinterpret_cast<void *>(r.base), r.size);
      }
    }
    if (!scans.empty()) rec.scans_forgotten = forgotten;   // (compared in the round before)
    if (rec.scans.empty() || rec.scans_forgotten == g.scans_forgotten) {
      // what the library remembered about the old contents of the blocks this replay writes
      for (uintptr_t base : rec.writes) forget_scans_locked(base);
      for (int r = g_repeat; r > 0; --r) TFHIP_CHECK_HIP(hipGraphLaunch(rec.exec, g.stream));
      return kOk;
    }
    // Some filter, perhaps one of these, has been written since: a kernel that multiplies padding by its filter must not
    // be replayed with an Inf or a NaN in it. What was not written is remembered, what was costs a search.
    scans = rec.scans;
    forgotten = g.scans_forgotten;
    lock.unlock();
    for (const FilterScan &f : scans) {
      bool nonfinite = false;
      const int rc = scan_filter(reinterpret_cast<const float *>(f.ptr), (int64_t)f.elems, "tfhip_graph_launch", &nonfinite);
      if (rc != kOk) return rc;
      if (nonfinite)
        return fail(kBadArgument, "tfhip_graph_launch: the filter at %p was finite when graph %d was recorded and holds Inf or NaN now",
                    reinterpret_cast<void *>(f.ptr), graph_id);
    }
  }
}

int tfhip_graph_destroy(int graph_id) {
  TFHIP_REQUIRE_INIT();
  std::lock_guard<std::mutex> lock(g_mutex);
  auto it = g.graphs.find(graph_id);
  TFHIP_CHECK_ARG(it != g.graphs.end(), "tfhip_graph_destroy: no graph %d", graph_id);
  (void)hipStreamSynchronize(g.stream);   // no replay is in flight when the executable goes
  if (it->second.exec) (void)hipGraphExecDestroy(it->second.exec);
  for (auto &b : it->second.owned) give_back_locked(b.first, b.second);
  g.graphs.erase(it);
  return kOk;
}

}  // extern "C"
