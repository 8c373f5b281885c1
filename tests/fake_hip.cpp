// A HIP runtime that launches nothing: each kernel launch is only written down (kernel,
// grid, K splits of the mid-batch and large-M kernels, host thread).  Loaded into a process
// of its own ahead of libmarlin_hip.so, it shows on the CPU which kernels a call runs and
// in which order the launches of several host threads reach a stream.  Every launch
// takes a millisecond, so that threads that may interleave do.
#include <stddef.h>
#include <string.h>
#include <time.h>

#include <atomic>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

struct dim3 {
  unsigned x, y, z;
};

namespace {
struct Launch {
  std::string kernel;
  unsigned grid, block;
  int splits;  // of the mid-batch and large-M kernels (else 0)
  int caller;  // set by fake_hip_caller on the calling thread
};
std::mutex mu;
std::map<const void*, std::string> kernels;
std::vector<Launch> launches;
thread_local int caller = 0;
thread_local struct {
  dim3 grid, block;
  size_t lds;
  void* stream;
} config;
char symbol[256];
std::atomic<size_t> next{size_t(1) << 40};
}  // namespace

extern "C" {
void fake_hip_caller(int id) { caller = id; }
int fake_hip_launches() {
  std::lock_guard<std::mutex> lock(mu);
  return (int)launches.size();
}
const char* fake_hip_launch(int i, unsigned* grid, unsigned* block, int* splits, int* id) {
  std::lock_guard<std::mutex> lock(mu);
  const Launch& l = launches[i];
  *grid = l.grid;
  *block = l.block;
  *splits = l.splits;
  *id = l.caller;
  return l.kernel.c_str();
}

void** __hipRegisterFatBinary(const void*) {
  static void* module;
  return &module;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*,
                           int*) {
  kernels[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, void* stream) {
  config = {grid, block, lds, stream};
  return 0;
}
int __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, void** stream) {
  *grid = config.grid;
  *block = config.block;
  *lds = config.lds;
  *stream = config.stream;
  return 0;
}
int hipLaunchKernel(const void* fn, dim3 grid, dim3 block, void** args, size_t, void*) {
  {
    std::lock_guard<std::mutex> lock(mu);
    Launch l{kernels[fn], grid.x * grid.y * grid.z, block.x, 0, caller};
    // their arguments: A, B, s, M, N, K, splits and B, meta, s, A, zeros, M, N, K, splits
    if (l.kernel.find("marlin_dense_mid_kernel") != std::string::npos) l.splits = *static_cast<int*>(args[6]);
    if (l.kernel.find("sm24_mid_kernel") != std::string::npos) l.splits = *static_cast<int*>(args[8]);
    // its GemmArgs: six pointers, M, N, K, splits
    if (l.kernel.find("sm24_prefill_kernel") != std::string::npos)
      l.splits = *reinterpret_cast<int*>(static_cast<char*>(args[0]) + 6 * sizeof(void*) + 3 * sizeof(int));
    launches.push_back(l);
  }
  const timespec ms{0, 1000000};
  nanosleep(&ms, nullptr);
  return 0;
}
int hipGetLastError() { return 0; }
const char* hipGetErrorString(int) { return "fake"; }
int hipGetDevice(int* d) {
  *d = 0;
  return 0;
}
int hipSetDevice(int) { return 0; }
int hipDeviceGetAttribute(int* v, int, int) {
  *v = 256;
  return 0;
}
int hipFuncGetAttributes(void*, const void*) { return 0; }
int hipGetSymbolAddress(void** p, const void*) {
  *p = symbol;
  return 0;
}
int hipStreamIsCapturing(void*, int* st) {
  *st = 0;
  return 0;
}
int hipMalloc(void** p, size_t n) {
  *p = reinterpret_cast<void*>(next.fetch_add((n + 4095) / 4096 * 4096));
  return 0;
}
int hipExtMallocWithFlags(void** p, size_t n, unsigned) { return hipMalloc(p, n); }
int hipMemset(void*, int, size_t) { return 0; }
int hipMemcpyAsync(void*, const void*, size_t, int, void*) { return 0; }
}
