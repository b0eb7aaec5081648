// Host stand-in for the HIP calls that the engine's host code makes, for tests
// of that code without a GPU. Device memory is host memory, copies are copies
// and kernels do not run; each launch looks for words of its descriptor (the
// block that the first argument points to) that name freed memory.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>

namespace {
std::map<void*, size_t> live;
std::map<void*, size_t> freed;  // kept, so that no address comes back
long mallocs_left = -1;         // hipMalloc calls until they fail (-1: none fails)
int stale = 0, launches = 0;
constexpr int kOutOfMemory = 2;

bool in_freed(uint64_t word) {
  auto it = freed.upper_bound(reinterpret_cast<void*>(word));
  if (it == freed.begin()) return false;
  --it;
  return word - reinterpret_cast<uint64_t>(it->first) < it->second;
}
}  // namespace

struct Dim3 {
  uint32_t x, y, z;
};

extern "C" {
void host_hip_fail_after(long n) { mallocs_left = n; }
int host_hip_stale() { return stale; }
int host_hip_launches() { return launches; }

int hipGetDeviceCount(int* n) { return *n = 1, 0; }
int hipGetDevice(int* d) { return *d = 0, 0; }
int hipSetDevice(int) { return 0; }
int hipGetLastError() { return 0; }
int hipMalloc(void** p, size_t n) {
  if (mallocs_left == 0) return kOutOfMemory;
  if (mallocs_left > 0) --mallocs_left;
  live[*p = std::calloc(n, 1)] = n;
  return 0;
}
int hipFree(void* p) {
  if (!p) return 0;
  freed[p] = live.at(p);
  live.erase(p);
  return 0;
}
int hipHostMalloc(void** p, size_t n, unsigned) { return *p = std::calloc(n, 1), 0; }
int hipHostFree(void* p) { return std::free(p), 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void*) { return std::memcpy(d, s, n), 0; }
int hipMemcpy(void* d, const void* s, size_t n, int) { return std::memcpy(d, s, n), 0; }
int hipMemsetAsync(void* d, int v, size_t n, void*) { return std::memset(d, v, n), 0; }
int hipStreamCreateWithFlags(void** s, unsigned) { return *s = nullptr, 0; }
int hipStreamSynchronize(void*) { return 0; }
int hipStreamDestroy(void*) { return 0; }
int hipEventCreateWithFlags(void** e, unsigned) { return *e = nullptr, 0; }
int hipEventRecord(void*, void*) { return 0; }
int hipEventSynchronize(void*) { return 0; }
int hipEventDestroy(void*) { return 0; }
int __hipPushCallConfiguration(Dim3, Dim3, size_t, void*) { return 0; }
int __hipPopCallConfiguration(Dim3* grid, Dim3* block, size_t* lds, void** stream) {
  *grid = *block = Dim3{1, 1, 1};
  return *lds = 0, *stream = nullptr, 0;
}
int hipLaunchKernel(const void*, Dim3, Dim3, void** args, size_t, void*) {
  ++launches;
  void* desc = nullptr;
  std::memcpy(&desc, args[0], sizeof(desc));
  const auto it = live.find(desc);
  for (size_t i = 0; it != live.end() && i + 8 <= it->second && it->second <= 4096; i += 8) {
    uint64_t word;
    std::memcpy(&word, static_cast<char*>(desc) + i, 8);
    stale += in_freed(word);
  }
  return 0;
}
}
