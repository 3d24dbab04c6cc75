// The part of the HIP runtime that libtfjs_hip.so calls, on host memory, for tests of its host code without a GPU:
// several devices, devices' copies of device symbols, streams that run everything at once, recordings. Of the kernels
// only those that the host code itself depends on have an effect (see run_kernel); the others are counted.
//
// Loaded into the global scope before libtfjs_hip.so, so that the library's calls end here. Misuse that a GPU would
// answer with a fault (a copy or a kernel argument outside live memory) is counted instead (fake_hip_errors).
#include <hip/hip_runtime_api.h>
#include <string.h>
#include <unistd.h>

#include <atomic>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

namespace {

constexpr int kDevices = 2;
constexpr size_t kNotedBytes = 192;   // of a launch's first argument

struct Block {
  size_t bytes;
  int device;   // -1: host
};
struct Launch {
  std::string name;
  std::vector<char> first;   // the leading bytes of the first argument (of few_rows and decode_batch)
  int device;
  bool recorded;
  unsigned grid_x;
};
struct Recording {
  std::vector<std::string> kernels;
  std::vector<std::vector<long long>> args;
};

std::recursive_mutex m;
std::map<uintptr_t, Block> blocks;
std::map<std::pair<int, const void *>, void *> symbols;
std::map<const void *, size_t> symbol_bytes;
std::map<const void *, std::string> kernel_names;
std::map<hipStream_t, Recording *> recording_on;
std::vector<Launch> launches;
thread_local int current_device = 0;
int errors = 0;
std::string first_error;
std::atomic<int> copy_delay_us{0}, launch_delay_us{0};
std::atomic<int> copies_now{0};
std::vector<uint64_t> copy_sizes;
std::map<hipStream_t, int> stream_device;
thread_local struct {
  dim3 grid, block;
  size_t shared;
  hipStream_t stream;
} pushed;

void note_error(const std::string &what) {
  ++errors;
  if (first_error.empty()) first_error = what;
}

bool inside_locked(const void *p, size_t bytes, Block *b = nullptr) {
  auto it = blocks.upper_bound((uintptr_t)p);
  if (it == blocks.begin()) return false;
  --it;
  if (b) *b = it->second;
  return (uintptr_t)p + bytes <= it->first + it->second.bytes;
}

void *take(size_t bytes, int device) {
  void *p = aligned_alloc(256, (bytes + 255) & ~size_t(255));
  memset(p, 0, bytes);
  std::lock_guard<std::recursive_mutex> lock(m);
  blocks[(uintptr_t)p] = {bytes, device};
  return p;
}

void drop(void *p) {
  if (!p) return;
  std::lock_guard<std::recursive_mutex> lock(m);
  if (!blocks.erase((uintptr_t)p)) return note_error("a block was freed that is not live");
  if (copies_now > 0) note_error("memory was freed while a copy was under way");
  free(p);
}

// The kernels whose effect the host code reads back.
void run_kernel(const std::string &name, const std::vector<long long> &a) {
  auto is = [&](const char *s) { return name.find(s) != std::string::npos; };
  if (is("clear_word")) {
    *(int *)a[0] = 0;
  } else if (is("find_nonfinite")) {
    const unsigned *bits = (const unsigned *)a[0];
    if (!inside_locked(bits, (size_t)a[1] * 4)) return note_error("find_nonfinite reads outside live memory");
    for (long long i = 0; i < a[1]; ++i)
      if ((bits[i] & 0x7f800000u) == 0x7f800000u) *(int *)a[2] = 1;
  } else if (is("copy_to_host")) {
    if (!inside_locked((void *)a[0], (size_t)(int)a[2] * 16) || !inside_locked((void *)a[1], (size_t)(int)a[2] * 16))
      return note_error("copy_to_host outside live memory");
    memcpy((void *)a[1], (void *)a[0], (size_t)(int)a[2] * 16);
  }
}
bool has_effect(const std::string &name) {
  for (const char *s : {"clear_word", "find_nonfinite", "copy_to_host"})
    if (name.find(s) != std::string::npos) return true;
  return false;
}

}  // namespace

extern "C" {

// ---- what the tests ask ----
int fake_hip_errors(char *text, size_t len) {
  std::lock_guard<std::recursive_mutex> lock(m);
  if (text && len) snprintf(text, len, "%s", first_error.c_str());
  return errors;
}
// Of the launch `back` launches ago: name, leading bytes of its first argument, whether it was recorded.
int fake_hip_launch(int back, char *name, size_t len, void *first, size_t first_len, int *recorded) {
  std::lock_guard<std::recursive_mutex> lock(m);
  if (back >= (int)launches.size()) return -1;
  const Launch &l = launches[launches.size() - 1 - back];
  snprintf(name, len, "%s", l.name.c_str());
  memcpy(first, l.first.data(), first_len < l.first.size() ? first_len : l.first.size());
  *recorded = l.recorded;
  return l.device;
}
// Workgroups along x of the launch `back` launches ago.
int fake_hip_grid(int back) {
  std::lock_guard<std::recursive_mutex> lock(m);
  return back < (int)launches.size() ? (int)launches[launches.size() - 1 - back].grid_x : -1;
}
int fake_hip_launches(void) {
  std::lock_guard<std::recursive_mutex> lock(m);
  return (int)launches.size();
}
// The device whose memory holds p, or -1.
int fake_hip_device_of(const void *p) {
  std::lock_guard<std::recursive_mutex> lock(m);
  Block b;
  return inside_locked(p, 1, &b) ? b.device : -1;
}
void fake_hip_copy_delay(int us) { copy_delay_us = us; }
int fake_hip_copies_now(void) { return copies_now; }
// The sizes of the copies since the last call, the first `most` of them; how many there were.
int fake_hip_copy_sizes(uint64_t *sizes, int most) {
  std::lock_guard<std::recursive_mutex> lock(m);
  const int n = (int)copy_sizes.size();
  for (int i = 0; i < n && i < most; ++i) sizes[i] = copy_sizes[i];
  copy_sizes.clear();
  return n;
}
void fake_hip_launch_delay(int us) { launch_delay_us = us; }

// ---- devices, memory ----
hipError_t hipGetDeviceCount(int *n) { *n = kDevices; return hipSuccess; }
hipError_t hipSetDevice(int d) { current_device = d; return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int) {   // (the header renames it)
  memset(p, 0, sizeof *p);
  strcpy(p->name, "stand-in");
  strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  p->totalGlobalMem = size_t(288) << 30;
  return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t bytes) { *p = take(bytes, current_device); return hipSuccess; }
hipError_t hipFree(void *p) { drop(p); return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) { *p = take(bytes, -1); return hipSuccess; }
hipError_t hipHostFree(void *p) { drop(p); return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *symbol) {
  std::lock_guard<std::recursive_mutex> lock(m);
  void *&at = symbols[{current_device, symbol}];
  if (!at) at = take(symbol_bytes.count(symbol) ? symbol_bytes[symbol] : 1 << 20, current_device);
  *p = at;
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t bytes, hipMemcpyKind, hipStream_t) {
  {
    std::lock_guard<std::recursive_mutex> lock(m);
    if (!inside_locked(d, bytes) || !inside_locked(s, bytes)) {
      note_error("a copy touches memory that is not live");
      return hipSuccess;
    }
    ++copies_now;
    copy_sizes.push_back(bytes);
  }
  if (copy_delay_us) usleep(copy_delay_us);
  std::lock_guard<std::recursive_mutex> lock(m);
  if (inside_locked(d, bytes) && inside_locked(s, bytes)) memcpy(d, s, bytes);
  --copies_now;
  return hipSuccess;
}

// ---- streams, events ----
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  *s = (hipStream_t)take(256, -1);
  std::lock_guard<std::recursive_mutex> lock(m);
  stream_device[*s] = current_device;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) { drop(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {
  std::lock_guard<std::recursive_mutex> lock(m);
  return recording_on.count(s) ? hipErrorStreamCaptureUnsupported : hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { *e = (hipEvent_t)take(8, -1); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { drop(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 0.f; return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "stand-in error"; }
hipError_t hipGetLastError(void) { return hipSuccess; }

// ---- launches ----
void **__hipRegisterFatBinary(const void *) { static void *handle; return &handle; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *, int *) {
  std::lock_guard<std::recursive_mutex> lock(m);
  kernel_names[host] = name;
}
void __hipRegisterVar(void **, void *var, char *, char *, int, size_t bytes, int, int) {
  std::lock_guard<std::recursive_mutex> lock(m);
  symbol_bytes[var] = bytes;
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream) {
  pushed = {grid, block, shared, stream};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shared, hipStream_t *stream) {
  *grid = pushed.grid; *block = pushed.block; *shared = pushed.shared; *stream = pushed.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3, void **args, size_t, hipStream_t stream) {
  if (launch_delay_us) usleep(launch_delay_us);
  std::lock_guard<std::recursive_mutex> lock(m);
  const std::string name = kernel_names[f];
  std::vector<long long> words;
  if (has_effect(name)) words = {*(long long *)args[0], *(long long *)(args[name.find("clear_word") == std::string::npos ? 1 : 0]),
                                 name.find("find_nonfinite") != std::string::npos ? *(long long *)args[2] :
                                 name.find("copy_to_host") != std::string::npos ? (long long)*(int *)args[2] : 0};
  Launch l = {name, {}, stream_device[stream], recording_on.count(stream) > 0, grid.x};
  if (name.find("few_rows") != std::string::npos) l.first.assign((const char *)args[0], (const char *)args[0] + kNotedBytes);
  if (name.find("decode_batch") != std::string::npos) l.first.assign((const char *)args[0], (const char *)args[0] + sizeof(void *));
  launches.push_back(l);
  if (l.recorded) {
    recording_on[stream]->kernels.push_back(name);
    recording_on[stream]->args.push_back(words);
  } else if (!words.empty()) {
    run_kernel(name, words);
  }
  return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) { *n = 2; return hipSuccess; }

// ---- recordings ----
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) {
  std::lock_guard<std::recursive_mutex> lock(m);
  recording_on[s] = new Recording();
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t *g) {
  std::lock_guard<std::recursive_mutex> lock(m);
  *g = (hipGraph_t)recording_on[s];
  recording_on.erase(s);
  return hipSuccess;
}
hipError_t hipGraphGetNodes(hipGraph_t g, hipGraphNode_t *, size_t *n) { *n = ((Recording *)g)->kernels.size(); return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t g, hipGraphNode_t *, char *, size_t) {
  *e = (hipGraphExec_t) new Recording(*(Recording *)g);
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) { delete (Recording *)g; return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { delete (Recording *)e; return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t stream) {
  std::lock_guard<std::recursive_mutex> lock(m);
  const Recording &r = *(Recording *)e;
  for (size_t i = 0; i < r.kernels.size(); ++i) {
    launches.push_back({r.kernels[i], {}, stream_device[stream], false, 0});
    if (!r.args[i].empty()) run_kernel(r.kernels[i], r.args[i]);
  }
  return hipSuccess;
}

}  // extern "C"
