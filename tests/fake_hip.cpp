// A HIP runtime without a GPU, for tests of what the host does: memory is host memory, a stream is always idle, the two
// copy kernels are made on the spot and every other launch is none.  fake_hip_refuse(name, n): the n-th launch from now
// of a kernel whose name holds `name` is refused, as the runtime refuses one that it cannot make ("hipHostMalloc": the n-th such call).
// fake_hip_launched(): the names of the kernels launched since the last call; fake_hip_products(): of the matrix products among them a line
// each, the name and what the kernel is told of its walk along k - slices, values to a slice, whether column tiles start at different ones -;
// fake_hip_outside(): those that are told to add values which lie outside of what was allocated; fake_hip_static_lds(n): what every kernel's
// own __shared__ variables take.
// Loaded with RTLD_GLOBAL before the library, whose references to the runtime it then answers.
#include <hip/hip_runtime.h>
#include <atomic>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#define HIP_INCLUDE_HIP_HIP_EXT_H  // (templates that only a HIP compiler takes, of which the descriptors need nothing)
#include "launch.hpp"

namespace {
std::map<const void *, std::string> &names() {
  static std::map<const void *, std::string> m;
  return m;
}
std::mutex lock;
std::string refuse, launched, products, outside;
std::map<const char *, size_t> rooms;  // what hipMalloc has given out
bool within(const void *p, size_t n) {
  auto it = rooms.upper_bound((const char *)p);
  return it != rooms.begin() && (--it, (const char *)p + n <= it->first + it->second);
}
std::atomic<int> countdown{0}, waits{0}, static_lds{0};
thread_local hipError_t last = hipSuccess;

// the argument lists of to_host_kernel and from_host_kernel (k_misc.hip)
void to_host(void **a) {
  const uint32_t *src = *(const uint32_t **)a[0], *err = *(const uint32_t **)a[3];
  uint32_t *dst = *(uint32_t **)a[1], *tail = *(uint32_t **)a[4];
  const uint64_t n = *(uint64_t *)a[2], piece = 32768, words = 16;
  if (n) std::memcpy(dst, src, n * 4);
  for (uint64_t p = 0; p == 0 || p * piece < n; ++p) {
    tail[p * words] = err[0];
    tail[p * words + 1] = err[1];
    __atomic_store_n(tail + p * words + 2, 1u, __ATOMIC_RELEASE);
  }
}
void from_host(void **a) {
  std::memcpy(*(void **)a[1], *(void **)a[0], *(uint32_t *)a[2] * (size_t)4);
  __atomic_store_n(*(uint32_t **)a[3], 1u, __ATOMIC_RELEASE);
}
hipError_t launch(const void *f, void **args) {
  const std::string &name = names()[f];
  {
    std::lock_guard<std::mutex> lk(lock);
    launched += name + "\n";
    if (name.find("NS_8GemmDescE") != std::string::npos) {
      const auto &g = *(const cgk::GemmDesc *)args[0];
      const uint32_t splits = g.splits > 1 ? g.splits : 1;
      if (g.c_add && splits == 1 && !within(g.c_add, (size_t)g.nb0 * g.nb1 * g.M * g.N * 4)) outside += name + "\n";
      products += name + " " + std::to_string(splits) + " " + std::to_string(splits > 1 ? g.k_per_split : g.K) + " " + std::to_string(g.k_rotate) + "\n";
    }
    if (name.find("NS_11MoeGemmDescE") != std::string::npos) {
      const auto &g = *(const cgk::MoeGemmDesc *)args[0];
      products += name + " 1 " + std::to_string(g.K) + " " + std::to_string(g.k_rotate) + "\n";
    }
    if (name.find("splitk_reduce_kernel") != std::string::npos) {  // (slices, sums, values of a slice, slices, what is added)
      const void *add = *(const void **)args[4];
      if (add && !within(add, *(uint64_t *)args[2] * 4)) outside += name + "\n";
    }
    if (!refuse.empty() && name.find(refuse) != std::string::npos && countdown.fetch_sub(1) == 1) {
      refuse.clear();
      return last = hipErrorInvalidConfiguration;
    }
  }
  if (name.find("to_host_kernel") != std::string::npos) to_host(args);
  if (name.find("from_host_kernel") != std::string::npos) from_host(args);
  return hipSuccess;
}
hipError_t memory(void **p, size_t n) { return (*p = aligned_alloc(4096, (n + 4095) / 4096 * 4096)) ? hipSuccess : hipErrorOutOfMemory; }
}  // namespace

extern "C" {
void fake_hip_refuse(const char *name, int n) {
  std::lock_guard<std::mutex> lk(lock);
  refuse = name;
  countdown = n;
}
int fake_hip_waits() { return waits; }  // on the stream
static const char *taken(std::string &lines) {
  static thread_local std::string since;
  std::lock_guard<std::mutex> lk(lock);
  since.clear();
  since.swap(lines);
  return since.c_str();
}
const char *fake_hip_launched() { return taken(launched); }
const char *fake_hip_products() { return taken(products); }
const char *fake_hip_outside() { return taken(outside); }
void fake_hip_static_lds(int n) { static_lds = n; }

void **__hipRegisterFatBinary(const void *) { static void *h[4]; return h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, uint3 *, uint3 *, dim3 *, dim3 *, int *) { names()[f] = name; }
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *) { return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_t *p, int) {
  std::memset(p, 0, sizeof(*p));
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) { static char room[1 << 18]; return *p = room, hipSuccess; }
hipError_t hipGetLastError() { const hipError_t e = last; return last = hipSuccess, e; }
const char *hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "launch refused"; }
hipError_t hipMalloc(void **p, size_t n) {
  const hipError_t e = memory(p, n);
  std::lock_guard<std::mutex> lk(lock);
  if (e == hipSuccess) rooms[(const char *)*p] = n;
  return e;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  std::lock_guard<std::mutex> lk(lock);
  if (refuse == "hipHostMalloc" && countdown.fetch_sub(1) == 1) {
    refuse.clear();
    return last = hipErrorOutOfMemory;
  }
  return memory(p, n);
}
hipError_t hipFree(void *p) {
  std::lock_guard<std::mutex> lk(lock);
  rooms.erase((const char *)p);
  return free(p), hipSuccess;
}
hipError_t hipHostFree(void *p) { return free(p), hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) { return std::memset(d, v, n), hipSuccess; }
hipError_t hipStreamCreate(hipStream_t *s) { return *s = nullptr, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return ++waits, hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return *e = nullptr, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 0.f, hipSuccess; }
hipError_t hipFuncGetAttributes(hipFuncAttributes *a, const void *) {
  std::memset(a, 0, sizeof(*a));
  a->sharedSizeBytes = static_lds;
  return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **args, size_t, hipStream_t) { return launch(f, args); }
hipError_t hipExtLaunchKernel(const void *f, dim3, dim3, void **args, size_t, hipStream_t, hipEvent_t, hipEvent_t, int) { return launch(f, args); }
}
