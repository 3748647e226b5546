// libvkv.so's device allocations over a host allocator of limited size: the
// HIP calls that the library makes resolve to the functions of this program.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <exception>
#include <map>

#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime_api.h>

static std::map<void*, size_t> live;
static size_t capacity = 0;
static size_t used() {
  size_t n = 0;
  for (auto& b : live) n += b.second;
  return n;
}

extern "C" {
hipError_t hipMalloc(void** p, size_t bytes) {
  if (used() + bytes > capacity) return hipErrorOutOfMemory;
  *p = std::malloc(1);
  live[*p] = bytes;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  if (!live.erase(p)) std::abort();
  std::free(p);
  return hipSuccess;
}
hipError_t hipGetDevice(int* dev) {
  *dev = 0;
  return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) {
  *s = hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipMemsetAsync(void*, int, size_t, hipStream_t) { return hipSuccess; }
}

namespace vkv {
struct DevPool {
  static void* take(size_t bytes, size_t* cap, int* dev);
  static void give(void* p, size_t cap, int dev);
};
float* attention_workspace(hipStream_t st, size_t floats);
uint32_t* attention_counters(hipStream_t st, size_t n);
size_t workspace_release(hipStream_t st);
}  // namespace vkv

#define CHECK(x)                                 \
  do {                                           \
    if (!(x)) {                                  \
      std::printf("line %d: %s\n", __LINE__, #x); \
      return 1;                                  \
    }                                            \
  } while (0)

int main() try {
  constexpr size_t kMb = size_t{1} << 20;
  capacity = 300 * kMb;
  auto keep = [&] {
    size_t cap = 0;
    int dev = 0;
    void* p = vkv::DevPool::take(128 * kMb, &cap, &dev);
    vkv::DevPool::give(p, cap, dev);
  };
  keep();
  CHECK(used() == 128 * kMb);
  // a stream's workspace and counters have the kept blocks' memory
  CHECK(vkv::attention_workspace(nullptr, 200 * kMb / 4) && used() == 200 * kMb);
  capacity = 260 * kMb;
  size_t cap = 0;
  int dev = 0;
  void* p = vkv::DevPool::take(60 * kMb - 512, &cap, &dev);
  vkv::DevPool::give(p, cap, dev);
  CHECK(vkv::attention_counters(nullptr, 50 * kMb / 4) && used() == 250 * kMb);
  // a release counts the kept blocks beside the stream's scratch, with or
  // without one
  capacity = 400 * kMb;
  keep();
  CHECK(vkv::workspace_release(nullptr) == 378 * kMb && used() == 0);
  keep();
  CHECK(vkv::workspace_release(nullptr) == 128 * kMb && used() == 0);
  CHECK(vkv::workspace_release(nullptr) == 0);
  std::printf("ok\n");
  return 0;
} catch (const std::exception& e) {
  std::printf("%s\n", e.what());
  return 1;
}
