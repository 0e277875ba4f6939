// Stand-in for the HIP runtime calls of libsoraku_mi355x.so, so that the host
// side of the engine (checks, order of calls, which kernels it launches with
// which grids) runs without a GPU.  Loaded with RTLD_GLOBAL before the library,
// its definitions come first.  Device memory is host memory; a kernel launch is
// only written down, so nothing on the "device" ever changes.
#include <hip/hip_runtime_api.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <map>
#include <new>
#include <string>

namespace {
std::map<const void*, std::string>& names() { static std::map<const void*, std::string> m; return m; }
std::string& calls() { static std::string s; return s; }   // one line per call
std::string fail_name;                                     // this call fails ...
int fail_after = -1;                                       // ... after so many of them (-1: never)
long new_limit = -1;                                       // operator new of more bytes throws (-1: never)
hipError_t last_launch = hipSuccess;
struct { dim3 grid, block; size_t smem; hipStream_t st; } cfg;

hipError_t note(const char* name, const std::string& more = "") {
  calls() += name + more + "\n";
  if (fail_after >= 0 && fail_name == name && fail_after-- == 0) return hipErrorUnknown;
  return hipSuccess;
}
}  // namespace

void* operator new(size_t n) {
  if (new_limit >= 0 && n > (size_t)new_limit) throw std::bad_alloc();
  if (void* p = malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }

extern "C" {

void stub_fail(const char* name, int after) { fail_name = name; fail_after = after; }
void stub_new_limit(long n) { new_limit = n; }
const char* stub_calls() { return calls().c_str(); }
void stub_clear() { calls().clear(); }

void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  names()[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t smem, hipStream_t st) {
  cfg = {g, b, smem, st};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* smem, hipStream_t* st) {
  *g = cfg.grid; *b = cfg.block; *smem = cfg.smem; *st = cfg.st;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void**, size_t, hipStream_t) {
  char t[96];
  snprintf(t, sizeof(t), " %u %u %u %u ", g.x, g.y, g.z, b.x);
  return last_launch = note("hipLaunchKernel", t + names()[f]);
}
hipError_t hipGetLastError() { const hipError_t e = last_launch; last_launch = hipSuccess; return e; }
const char* hipGetErrorString(hipError_t) { return "stub error"; }

hipError_t hipMalloc(void** p, size_t n) {
  *p = aligned_alloc(256, (n + 255) & ~(size_t)255);
  if (*p && n < (1u << 20)) memset(*p, 0, n);   // small ones may be read back (the XCD probe's ids)
  return note("hipMalloc", " " + std::to_string(n));
}
hipError_t hipFree(void* p) { free(p); return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = calloc(1, n); return note("hipHostMalloc"); }
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) { *d = h; return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { memcpy(d, s, n); return note("hipMemcpy"); }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { memcpy(d, s, n); return note("hipMemcpyAsync"); }
hipError_t hipMemset(void* d, int v, size_t n) { memset(d, v, n); return note("hipMemset"); }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { memset(d, v, n); return note("hipMemsetAsync"); }
hipError_t hipGetSymbolAddress(void** p, const void*) { static char* m = (char*)calloc(1, 64 << 20); *p = m; return hipSuccess; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }   // the CU count

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)malloc(8); return note("hipStreamCreateWithFlags"); }
hipError_t hipStreamDestroy(hipStream_t s) { free(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return note("hipStreamSynchronize"); }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return note("hipStreamWaitEvent"); }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* c) { *c = hipStreamCaptureStatusNone; return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return note("hipStreamBeginCapture"); }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { *g = (hipGraph_t)malloc(8); return note("hipStreamEndCapture"); }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t)malloc(8); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return note("hipEventRecord"); }
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t) { *x = (hipGraphExec_t)malloc(8); return note("hipGraphInstantiate"); }
hipError_t hipGraphUpload(hipGraphExec_t, hipStream_t) { return note("hipGraphUpload"); }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return note("hipGraphLaunch"); }
hipError_t hipGraphGetNodes(hipGraph_t, hipGraphNode_t*, size_t* n) { *n = 0; return hipSuccess; }
hipError_t hipGraphNodeGetType(hipGraphNode_t, hipGraphNodeType*) { return hipErrorUnknown; }
hipError_t hipGraphKernelNodeGetParams(hipGraphNode_t, hipKernelNodeParams*) { return hipErrorUnknown; }
hipError_t hipGraphExecKernelNodeSetParams(hipGraphExec_t, hipGraphNode_t, const hipKernelNodeParams*) { return note("hipGraphExecKernelNodeSetParams"); }
hipError_t hipGraphDestroy(hipGraph_t g) { free(g); return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t x) { free(x); return hipSuccess; }
}
