// A stand-in for the HIP runtime on machines without a device, for tests of the host code: memory is the host's, copies are copies, launches only
// count (by the kernel's name), graphs hold the number of launches that were captured. Loaded with its symbols visible to all (RTLD_GLOBAL) ahead of
// libnerva_hip.so, whose calls then end here. The double_* functions set what it answers and read what it saw; double_log is what streams were given, one
// line each: "kernel 1 name", "graph 1 nodes", "record 1 event", "wait 1 event", "sync 1", "sync event", streams and events numbered as they were created.
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>

#include <atomic>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
int g_cus = 256, g_each = 2;
long g_copies = 0, g_fail_copy = -1;
long g_captured = -1;   // launches since the capture began, or -1
std::map<const void *, std::string> g_names;
std::map<std::string, long> g_launches;
std::string g_log;
std::map<const void *, long> g_numbers;   // of streams and events
long g_streams = 0, g_events = 0;
std::atomic<long> g_held{0}, g_waits{0};
thread_local hipStream_t t_stream;

void log(const char *what, const void *first, const std::string &rest = "") {
  if (g_captured < 0) g_log += std::string(what) + " " + std::to_string(g_numbers[first]) + (rest.empty() ? "" : " " + rest) + "\n";
}
std::string number(const void *of) { return std::to_string(g_numbers[of]); }

struct Graph {
  long nodes;
};
hipError_t copy(void *dst, const void *src, size_t bytes) {
  if (g_copies++ == g_fail_copy) return hipErrorUnknown;
  memcpy(dst, src, bytes);
  return hipSuccess;
}
}  // namespace

extern "C" {
void double_device(int cus, int each) {
  g_cus = cus;
  g_each = each;
}
// The copy with this number, from now on, fails (-1: none does).
void double_fail_copy(long number) {
  g_copies = 0;
  g_fail_copy = number;
}
long double_copies() { return g_copies; }
// Whoever waits for that stream waits until another one is named (0: none); whether somebody does.
void double_hold(long stream) { g_held = stream; }
long double_waits() { return g_waits; }
void double_clear_log() { g_log.clear(); }
const char *double_log() { return g_log.c_str(); }
// Launches of kernels whose names hold `part`.
long double_launches(const char *part) {
  long n = 0;
  for (const auto &entry : g_launches)
    if (entry.first.find(part) != std::string::npos) n += entry.second;
  return n;
}

void **__hipRegisterFatBinary(const void *) {
  static void *handle;
  return &handle;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *, int *) { g_names[host] = name; }
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t stream) {
  t_stream = stream;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *stream) {
  *stream = t_stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *kernel, dim3, dim3, void **, size_t, hipStream_t stream) {
  g_launches[g_names[kernel]] += 1;
  log("kernel", stream, g_names[kernel]);
  if (g_captured >= 0) g_captured += 1;
  return hipSuccess;
}

hipError_t hipGetDeviceCount(int *count) {
  *count = 1;
  return hipSuccess;
}
hipError_t hipGetDevice(int *device) {
  *device = 0;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *value, hipDeviceAttribute_t which, int) {
  *value = which == hipDeviceAttributeMultiprocessorCount ? g_cus : 0;
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *blocks, const void *, int, size_t) {
  *blocks = g_each;
  return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t *prop, int) {
  memset(prop, 0, sizeof(*prop));
  prop->multiProcessorCount = g_cus;
  return hipSuccess;
}
hipError_t hipDeviceGetPCIBusId(char *id, int bytes, int) {
  if (bytes > 0) id[0] = 0;
  return hipSuccess;
}
hipError_t hipDriverGetVersion(int *version) {
  *version = 0;
  return hipSuccess;
}
hipError_t hipRuntimeGetVersion(int *version) {
  *version = 0;
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipMemGetInfo(size_t *free_bytes, size_t *all) {
  *free_bytes = *all = size_t{1} << 38;
  return hipSuccess;
}

hipError_t hipMalloc(void **ptr, size_t bytes) {
  *ptr = aligned_alloc(4096, (bytes + 4095) / 4096 * 4096);
  return *ptr != nullptr ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostMalloc(void **ptr, size_t bytes, unsigned) { return hipMalloc(ptr, bytes); }
hipError_t hipFree(void *ptr) {
  free(ptr);
  return hipSuccess;
}
hipError_t hipHostFree(void *ptr) { return hipFree(ptr); }
hipError_t hipMemcpy(void *dst, const void *src, size_t bytes, hipMemcpyKind) { return copy(dst, src, bytes); }
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t bytes, hipMemcpyKind, hipStream_t) { return copy(dst, src, bytes); }
hipError_t hipMemset(void *dst, int value, size_t bytes) {
  memset(dst, value, bytes);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *dst, int value, size_t bytes, hipStream_t) { return hipMemset(dst, value, bytes); }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *, const void *) { return hipErrorInvalidValue; }
hipError_t hipGetSymbolAddress(void **ptr, const void *) {
  static char scratch[1 << 20];
  *ptr = scratch;
  return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t *stream, unsigned) {
  *stream = reinterpret_cast<hipStream_t>(malloc(1));
  g_numbers[*stream] = ++g_streams;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t stream) {
  free(stream);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t stream) {
  log("sync", stream);
  while (g_held == g_numbers[stream]) g_waits = 1;
  g_waits = 0;
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t stream, hipEvent_t event, unsigned) {
  log("wait", stream, number(event));
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *event, unsigned) {
  *event = reinterpret_cast<hipEvent_t>(malloc(1));
  g_numbers[*event] = ++g_events;
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *event) { return hipEventCreateWithFlags(event, 0); }
hipError_t hipEventDestroy(hipEvent_t event) {
  free(event);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t event, hipStream_t stream) {
  log("record", stream, number(event));
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t event) {
  log("sync event", event);
  return hipSuccess;
}
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
  *ms = 1.0f;
  return hipSuccess;
}

hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
  g_captured = 0;
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *graph) {
  *graph = reinterpret_cast<hipGraph_t>(new Graph{g_captured});
  g_captured = -1;
  return hipSuccess;
}
hipError_t hipGraphGetNodes(hipGraph_t graph, hipGraphNode_t *, size_t *count) {
  *count = static_cast<size_t>(reinterpret_cast<Graph *>(graph)->nodes);
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *exec, hipGraph_t graph, hipGraphNode_t *, char *, size_t) {
  *exec = reinterpret_cast<hipGraphExec_t>(new Graph(*reinterpret_cast<Graph *>(graph)));
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t exec, hipStream_t stream) {
  log("graph", stream, std::to_string(reinterpret_cast<Graph *>(exec)->nodes));
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t graph) {
  delete reinterpret_cast<Graph *>(graph);
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t exec) {
  delete reinterpret_cast<Graph *>(exec);
  return hipSuccess;
}
}
