/* A stand-in for the HIP runtime, for tests of the library's host path on a
 * machine without a GPU. Device memory is host memory, copies and clears are
 * done at once, kernels do nothing. What it keeps is which stream still has
 * work that nothing has waited for, by HIP's rules for a null stream and
 * streams that do not block on it:
 *
 *  - hipMemset and hipMemcpy go to the null stream and may return before they
 *    are done (a copy from pageable memory once that has been read), but for a
 *    copy to the host, which waits for the null stream;
 *  - anything with a stream argument, and every launch, is queued there;
 *  - synchronising a stream, an event on it or the device waits, and so does
 *    freeing memory.
 *
 * fake_unordered() counts the calls that queued work on one stream while the
 * other still had some: nothing orders the two. fake_pending() is whether a
 * created stream has unfinished work. fake_fail_in(n) makes the n-th copy from
 * now that is given a stream fail. */
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>
#include <stdlib.h>
#include <string.h>

static int pending[2]; /* 0: the null stream, 1: the created ones */
static long unordered;
static int fail_in;
static int stream_token, event_token, binary_token;

long fake_unordered(void) { return unordered; }
int fake_pending(void) { return pending[1]; }
void fake_fail_in(int n) { fail_in = n; }

static void queue(hipStream_t s) {
  const int k = s != NULL;
  if (pending[!k]) ++unordered;
  pending[k] = 1;
}
static void wait_all(void) { pending[0] = pending[1] = 0; }

hipError_t hipMalloc(void** p, size_t n) { return (*p = calloc(1, n ? n : 1)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipFree(void* p) {
  if (p) wait_all();
  free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned f) { (void)f; return hipMalloc(p, n); }
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned f) { (void)f; *d = h; return hipSuccess; }

hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind k) {
  queue(NULL);
  if (k == hipMemcpyDeviceToHost) pending[0] = 0;
  memmove(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t st) {
  (void)k;
  if (fail_in > 0 && --fail_in == 0) return hipErrorUnknown;
  queue(st);
  memmove(d, s, n);
  return hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n) { queue(NULL); memset(d, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t st) {
  queue(st);
  memset(d, v, n);
  return hipSuccess;
}

hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void** a, size_t m, hipStream_t s) {
  (void)f; (void)g; (void)b; (void)a; (void)m;
  queue(s);
  return hipSuccess;
}
hipError_t hipLaunchCooperativeKernel(const void* f, dim3 g, dim3 b, void** a, unsigned m, hipStream_t s) {
  return hipLaunchKernel(f, g, b, a, m, s);
}
hipError_t hipFuncSetAttribute(const void* f, hipFuncAttribute a, int v) { (void)f; (void)a; (void)v; return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void* f, int b, size_t m) {
  (void)f; (void)b; (void)m;
  *n = 1;
  return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned f) {
  if (f != hipStreamNonBlocking) return hipErrorInvalidValue;
  *s = (hipStream_t)&stream_token;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) { (void)s; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { pending[s != NULL] = 0; return hipSuccess; }
hipError_t hipStreamQuery(hipStream_t s) { return hipStreamSynchronize(s); }
hipError_t hipDeviceSynchronize(void) { wait_all(); return hipSuccess; }
hipError_t hipDeviceReset(void) { wait_all(); return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t)&event_token; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { (void)e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { (void)e; (void)s; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { (void)e; pending[1] = 0; return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b) { (void)a; (void)b; *ms = 0; return hipSuccess; }

hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int d) { (void)d; return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int d) {
  (void)d;
  memset(p, 0, sizeof *p);
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
const char* hipGetErrorString(hipError_t e) { (void)e; return "failed by the test"; }
hipError_t hipGetSymbolAddress(void** p, const void* s) { (void)s; (void)p; return hipErrorNotSupported; }

hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode m) { (void)s; (void)m; return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t* g) { (void)s; (void)g; return hipErrorNotSupported; }

/* What the compiler's launch and registration code calls. */
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t m, hipStream_t s);
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* m, hipStream_t* s);
static struct { dim3 g, b; size_t m; hipStream_t s; } call;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t m, hipStream_t s) {
  call.g = g;
  call.b = b;
  call.m = m;
  call.s = s;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* m, hipStream_t* s) {
  *g = call.g;
  *b = call.b;
  *m = call.m;
  *s = call.s;
  return hipSuccess;
}
void** __hipRegisterFatBinary(const void* d) { (void)d; static void* h = &binary_token; return &h; }
void __hipUnregisterFatBinary(void** h) { (void)h; }
void __hipRegisterFunction(void** h, const void* f, char* n, const char* dn, unsigned t, void* a, void* b, void* c, void* d, int* e) {
  (void)h; (void)f; (void)n; (void)dn; (void)t; (void)a; (void)b; (void)c; (void)d; (void)e;
}
void __hipRegisterVar(void** h, void* v, char* n, char* dn, int e, size_t s, int c, int g) {
  (void)h; (void)v; (void)n; (void)dn; (void)e; (void)s; (void)c; (void)g;
}
