// A stand-in for the HIP runtime that runs no kernel: it hands out addresses
// that nothing may read, and keeps a list of the calls that it got, one line
// each, so that the library's host side (which kernel a call takes, with which
// grid, what it allocates, what it does when a result never arrives or a
// stream is capturing) can be checked where there is no GPU.
//
// Loaded with RTLD_GLOBAL ahead of libwgblas_hip.so, whose calls then bind
// here. 256 compute units, four blocks of any kernel per unit.
#include <hip/hip_runtime_api.h>

#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {

std::string g_log;
std::map<const void *, std::string> g_kernels;
hipStreamCaptureStatus g_capture = hipStreamCaptureStatusNone;
uintptr_t g_next = (uintptr_t)1 << 40;  // device addresses, 256-byte aligned
dim3 g_grid, g_block;
size_t g_shared;
hipStream_t g_stream;

void note(const char *format, ...) {
  char line[256];
  va_list args;
  va_start(args, format);
  std::vsnprintf(line, sizeof(line), format, args);
  va_end(args);
  g_log += line;
  g_log += '\n';
}

}  // namespace

extern "C" {

const char *standin_log() { return g_log.c_str(); }
void standin_clear() { g_log.clear(); }
void standin_capture(int on) { g_capture = on ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone; }

void **__hipRegisterFatBinary(const void *) {
  static void *modules = nullptr;
  return &modules;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, dim3 *,
                           dim3 *, int *) {
  g_kernels[host] = name;
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream) {
  g_grid = grid;
  g_block = block;
  g_shared = shared;
  g_stream = stream;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shared, hipStream_t *stream) {
  *grid = g_grid;
  *block = g_block;
  *shared = g_shared;
  *stream = g_stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *host, dim3 grid, dim3 block, void **, size_t, hipStream_t) {
  note("launch %u %u %u %u %s", grid.x, grid.y, grid.z, block.x, g_kernels[host].c_str());
  return hipSuccess;
}

hipError_t hipMalloc(void **ptr, size_t bytes) {
  note("malloc %zu", bytes);
  *ptr = (void *)g_next;
  g_next += (bytes + 255) / 256 * 256;
  return hipSuccess;
}
hipError_t hipFree(void *) { return hipSuccess; }
hipError_t hipHostMalloc(void **ptr, size_t bytes, unsigned flags) {
  note("host_malloc %zu %u", bytes, flags);
  *ptr = std::calloc(1, bytes);
  return hipSuccess;
}
hipError_t hipHostFree(void *ptr) {
  std::free(ptr);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *, const void *, size_t bytes, hipMemcpyKind, hipStream_t) {
  note("memcpy %zu", bytes);
  return hipSuccess;
}
hipError_t hipMemcpy2DAsync(void *, size_t, const void *, size_t, size_t width, size_t height, hipMemcpyKind,
                            hipStream_t) {
  note("memcpy %zu", width * height);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *, int, size_t bytes, hipStream_t) {
  note("memset %zu", bytes);
  return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t *stream, unsigned) {
  *stream = (hipStream_t)&g_stream;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) {
  note("synchronize");
  return g_capture == hipStreamCaptureStatusNone ? hipSuccess : hipErrorStreamCaptureUnsupported;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *status) {
  *status = g_capture;
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *event) {
  *event = (hipEvent_t)&g_stream;
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
  *ms = 0;
  return hipSuccess;
}

hipError_t hipGetDeviceCount(int *count) {
  *count = 1;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
// (hipGetDeviceProperties is a macro for the versioned name)
hipError_t hipGetDeviceProperties(hipDeviceProp_t *prop, int) {
  std::memset(prop, 0, sizeof(*prop));
  std::snprintf(prop->gcnArchName, sizeof(prop->gcnArchName), "gfx950");
  prop->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **ptr, const void *) {
  *ptr = (void *)((uintptr_t)1 << 39);
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *blocks, const void *, int, size_t) {
  *blocks = 4;
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "error of the stand-in runtime"; }

}  // extern "C"
