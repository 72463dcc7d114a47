// A HIP runtime without a device, for tests of the host side on the CPU: kernels are noted by name and not run (but for
// k_read_back, whose ticket is stored as the kernel would), a launch check can be told to fail, and what happened can be
// read as a list of lines.  Loaded with its symbols global in front of libzen_hip.so, whose calls then end here.
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
struct Dim3 {
  uint32_t x, y, z;
};
std::map<const void *, std::string> g_kernels;
std::string g_log;
int g_fail_at = 0, g_checks = 0;
struct {
  Dim3 grid, block;
  size_t lds;
  void *stream;
} g_config;
}  // namespace

extern "C" {
// The fail_at-th launch check from here on reports an error (0: none does).
void fake_reset(int fail_at) {
  g_log.clear();
  g_fail_at = fail_at;
  g_checks = 0;
}
const char *fake_log() { return g_log.c_str(); }

void **__hipRegisterFatBinary(const void *) {
  static void *handle;
  return &handle;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *, int *) {
  g_kernels[host] = name;
}
void __hipRegisterVar(void **, void *, char *, const char *, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t lds, void *stream) {
  g_config = {grid, block, lds, stream};
  return 0;
}
int __hipPopCallConfiguration(Dim3 *grid, Dim3 *block, size_t *lds, void **stream) {
  *grid = g_config.grid;
  *block = g_config.block;
  *lds = g_config.lds;
  *stream = g_config.stream;
  return 0;
}
int hipLaunchKernel(const void *host, Dim3, Dim3, void **args, size_t, void *stream) {
  const std::string &name = g_kernels[host];
  g_log += "launch " + name + " " + std::to_string(reinterpret_cast<uintptr_t>(stream)) + "\n";
  if (name.find("k_read_back") != std::string::npos) **static_cast<int64_t **>(args[1]) = *static_cast<int64_t *>(args[2]);
  return 0;
}
int hipGetLastError() {
  if (++g_checks != g_fail_at) return 0;
  g_log += "fail\n";
  return 719;
}
const char *hipGetErrorString(int) { return "the device"; }
int hipStreamSynchronize(void *stream) {
  g_log += "wait " + std::to_string(reinterpret_cast<uintptr_t>(stream)) + "\n";
  return 0;
}
int hipStreamQuery(void *) { return 0; }
int hipStreamIsCapturing(void *, int *status) { return *status = 0; }
int hipStreamWaitEvent(void *, void *, unsigned) { return 0; }
int hipEventCreate(void **event) { return (*event = &g_config, 0); }
int hipEventCreateWithFlags(void **event, unsigned) { return (*event = &g_config, 0); }
int hipEventRecord(void *, void *) { return 0; }
int hipEventSynchronize(void *) { return 0; }
int hipEventElapsedTime(float *ms, void *, void *) { return (*ms = 0, 0); }
int hipFuncSetAttribute(const void *, int, int) { return 0; }
int hipGetDevice(int *device) { return *device = 0; }
int hipDeviceGetAttribute(int *value, int, int) { return (*value = 256, 0); }
int hipGetSymbolAddress(void **, const void *) { return 1; }
int hipHostMalloc(void **p, size_t bytes, unsigned) { return (*p = calloc(1, bytes), 0); }
int hipHostFree(void *p) { return (free(p), 0); }
int hipMemcpy(void *, const void *, size_t, int) { return 0; }
int hipMemcpyAsync(void *, const void *, size_t, int, void *) { return 0; }
}
