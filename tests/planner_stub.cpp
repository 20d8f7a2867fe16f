/* The HIP calls of csrc/runtime.cpp without a GPU: a device of 256 compute units,
 * addresses that nothing reads, kernels looked up by name in the images built into
 * the library, launches written down (tests/planner.py). */
#include <hip/hip_runtime.h>

#include <cstring>
#include <set>
#include <string>

#include "scratch.h"

#define EXPORT extern "C" __attribute__((visibility("default")))

struct Blob {
  const char *start, *end;
};
extern "C" const Blob tm_builtin_blob_table[];
extern "C" const int32_t tm_builtin_blob_count;

namespace {
std::string g_log;
uintptr_t g_next = (uintptr_t)1 << 44;
std::set<std::string> g_names;
void *fake(size_t size) {
  void *p = (void *)g_next;
  g_next += (size + 8191) & ~(size_t)4095;
  return p;
}
}  // namespace

/* the launches since the last call: "name gx gy gz block lds" lines */
EXPORT int planner_take_log(char *out, int size) {
  const int n = (int)g_log.size();
  if (n + 1 > size) return -1;
  memcpy(out, g_log.c_str(), n + 1);
  g_log.clear();
  return n;
}

hipError_t tm_scratch_address(void **ptr) {
  static void *scratch = fake(TM_SCRATCH_BYTES);
  *ptr = scratch;
  return hipSuccess;
}

EXPORT hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
EXPORT hipError_t hipSetDevice(int) { return hipSuccess; }
EXPORT hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int) {
  memset(p, 0, sizeof *p);
  strcpy(p->name, "no device");
  strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  return hipSuccess;
}
EXPORT hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return *s = (hipStream_t)&g_log, hipSuccess; }
EXPORT hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
EXPORT hipError_t hipMalloc(void **p, size_t size) { return *p = fake(size), hipSuccess; }
EXPORT hipError_t hipFree(void *) { return hipSuccess; }
EXPORT hipError_t hipHostMalloc(void **, size_t, unsigned) { return hipErrorOutOfMemory; }
EXPORT hipError_t hipHostFree(void *) { return hipSuccess; }
EXPORT hipError_t hipMemcpy(void *, const void *, size_t, hipMemcpyKind) { return hipSuccess; }
EXPORT hipError_t hipMemcpyAsync(void *, const void *, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
EXPORT hipError_t hipMemsetAsync(void *, int, size_t, hipStream_t) { return hipSuccess; }
EXPORT hipError_t hipGetLastError() { return hipSuccess; }
EXPORT const char *hipGetErrorName(hipError_t) { return "hipErrorNotFound"; }
EXPORT const char *hipGetErrorString(hipError_t) { return "not found"; }
EXPORT hipError_t hipEventCreate(hipEvent_t *) { return hipErrorNotSupported; }
EXPORT hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
EXPORT hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipErrorNotSupported; }
EXPORT hipError_t hipEventElapsedTime(float *, hipEvent_t, hipEvent_t) { return hipErrorNotSupported; }

EXPORT hipError_t hipModuleLoadData(hipModule_t *m, const void *image) { return *m = (hipModule_t)image, hipSuccess; }
EXPORT hipError_t hipModuleUnload(hipModule_t) { return hipSuccess; }
/* a kernel is there if the image has its descriptor's symbol name, "<name>.kd" */
EXPORT hipError_t hipModuleGetFunction(hipFunction_t *f, hipModule_t m, const char *name) {
  const std::string symbol = std::string(1, '\0') + name + ".kd" + std::string(1, '\0');
  for (int i = 0; i < tm_builtin_blob_count; ++i) {
    const Blob &b = tm_builtin_blob_table[i];
    if ((const void *)b.start == (const void *)m && memmem(b.start, b.end - b.start, symbol.data(), symbol.size())) {
      *f = (hipFunction_t)g_names.insert(name).first->c_str();
      return hipSuccess;
    }
  }
  return hipErrorNotFound;
}
EXPORT hipError_t hipFuncGetAttribute(int *v, hipFunction_attribute, hipFunction_t) { return *v = 1024, hipSuccess; }
EXPORT hipError_t hipModuleLaunchKernel(hipFunction_t f, unsigned gx, unsigned gy, unsigned gz, unsigned bx, unsigned,
                                        unsigned, unsigned lds, hipStream_t, void **, void **) {
  g_log += std::string((const char *)f) + " " + std::to_string(gx) + " " + std::to_string(gy) + " " +
           std::to_string(gz) + " " + std::to_string(bx) + " " + std::to_string(lds) + "\n";
  return hipSuccess;
}
