// A stand-in for the HIP runtime on a machine without a GPU, for tests of the
// library's host code: device memory is host memory, its first MiB filled with
// 0x11, kernels do nothing except host_copy_kernel, whose copies are made, and
// one launch, wait or flag can be made to fail.  Built as libamdhip64.so.7 and loaded
// before the library, in a process of its own.
#include <map>
#include <string>

#include <stdlib.h>
#include <string.h>

#include "w4a8_internal.h"

namespace {
std::map<const void *, std::string> names;
std::string last_name;
unsigned last_grid;
int launches, fail_in, sync_fails, flag_lost, device_error;
struct Config {
  dim3 grid, block;
  size_t shmem;
  hipStream_t stream;
} config;

hipError_t launch(const void *f, dim3 grid, void **args) {
  ++launches;
  last_name = names[f];
  last_grid = grid.x;
  if (fail_in > 0 && --fail_in == 0) return hipErrorLaunchFailure;
  if (names[f].find("host_copy_kernel") != std::string::npos) {
    const w4a8::HostCopy &c = *(const w4a8::HostCopy *)args[0];
    memcpy(c.dst, c.src, (size_t)c.n);
    if (c.flag && !flag_lost) {
      if (device_error) *(int32_t *)c.err = device_error;
      *c.err_out = *c.err;
      *c.flag = c.seq;
    }
  }
  return hipSuccess;
}
hipError_t last = hipSuccess;
hipError_t note(hipError_t e) {
  if (e != hipSuccess) last = e;
  return e;
}
}  // namespace

extern "C" {

// what the tests set and read: the launch that fails (1: the next), whether
// waits fail, whether copies' flags stay down, the error word kernels leave;
// the launches so far, and the last one's kernel and grid
void fake_set(int fail, int sync, int lost, int err) {
  fail_in = fail;
  sync_fails = sync;
  flag_lost = lost;
  device_error = err;
}
int fake_launches(void) { return launches; }
const char *fake_last_kernel(unsigned *grid) {
  *grid = last_grid;
  return last_name.c_str();
}

void **__hipRegisterFatBinary(const void *) {
  static void *module;
  return &module;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *,
                           void *, dim3 *, dim3 *, int *) {
  names[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t n, hipStream_t s) {
  config = Config{g, b, n, s};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *n, hipStream_t *s) {
  *g = config.grid;
  *b = config.block;
  *n = config.shmem;
  *s = config.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3, void **args, size_t, hipStream_t) {
  return note(launch(f, g, args));
}
hipError_t hipExtLaunchKernel(const void *f, dim3 g, dim3, void **args, size_t, hipStream_t,
                              hipEvent_t, hipEvent_t, int) {
  return note(launch(f, g, args));
}
hipError_t hipLaunchCooperativeKernel(const void *f, dim3 g, dim3, void **args, unsigned,
                                      hipStream_t) {
  return note(launch(f, g, args));
}
hipError_t hipGetLastError(void) {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
const char *hipGetErrorString(hipError_t) { return "an error"; }

static hipError_t allocate(void **p, size_t n) {
  *p = aligned_alloc(4096, (n + 4095) / 4096 * 4096);
  memset(*p, 0x11, n < (1 << 20) ? n : 1 << 20);
  return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n) { return allocate(p, n); }
hipError_t hipFree(void *p) {
  free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return allocate(p, n); }
hipError_t hipHostFree(void *p) { return hipFree(p); }
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned) {
  *d = h;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **d, const void *) {
  static char symbol[2 << 20];
  *d = symbol;
  return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) {
  return hipMemcpy(d, s, n, k);
}
hipError_t hipMemset(void *d, int v, size_t n) {
  memset(d, v, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) { return hipMemset(d, v, n); }

hipError_t hipGetDeviceCount(int *n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipGetDevice(int *d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) {
  *v = 256;
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  *s = (hipStream_t)&config;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) {
  return sync_fails ? hipErrorUnknown : hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s) {
  *s = hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorUnknown; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *) { return hipErrorUnknown; }
hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, hipGraphNode_t *, char *, size_t) {
  return hipErrorUnknown;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorUnknown; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *) { return hipErrorUnknown; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipErrorUnknown; }
hipError_t hipEventElapsedTime(float *, hipEvent_t, hipEvent_t) { return hipErrorUnknown; }

}  // extern "C"
