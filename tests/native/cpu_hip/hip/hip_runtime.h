// A HIP runtime on the CPU, for running the library's own kernels and planning
// without a device (test infrastructure).  Device memory is host memory, every
// allocation between two inaccessible pages and ending at the second, so a
// kernel that reads or writes past an array stops there.  A launch runs at once:
// its blocks one after another, a block's threads one after another, both from
// the last to the first with CPU_HIP_ORDER=reverse -- blocks of one launch
// that depend on each other's order then give other results.  A block that
// synchronises runs again from its start with a context per thread (what its
// threads did before the first barrier must not matter when done twice).
#pragma once
#include <math.h>
#include <stddef.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <tuple>

#define __device__
#define __host__
#define __global__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __align__(n) __attribute__((aligned(n)))
#define __shared__ static
#define HIP_SYMBOL(x) (&x)
#define __builtin_amdgcn_readfirstlane(x) (x)

struct dim3 {
  unsigned x, y, z;
  dim3(unsigned a = 1, unsigned b = 1, unsigned c = 1) : x(a), y(b), z(c) {}
};
struct cpu_index { unsigned x, y, z; };
extern cpu_index threadIdx, blockIdx, blockDim, gridDim;

static inline int min(int a, int b) { return a < b ? a : b; }
static inline unsigned min(unsigned a, unsigned b) { return a < b ? a : b; }
static inline int max(int a, int b) { return a > b ? a : b; }
static inline unsigned atomicAdd(unsigned *p, unsigned v) { const unsigned o = *p; *p += v; return o; }
static inline unsigned long long atomicAdd(unsigned long long *p, unsigned long long v)
{
  const unsigned long long o = *p;
  *p += v;
  return o;
}
static inline unsigned long long atomicMin(unsigned long long *p, unsigned long long v)
{
  const unsigned long long o = *p;
  if (v < o) *p = v;
  return o;
}
static inline int __ffs(int v) { return __builtin_ffs(v); }
template <typename V> static inline V __shfl_down(V, int)
{
  fprintf(stderr, "wavefront shuffles do not run on the CPU\n");
  abort();
}
void __syncthreads();

enum hipError_t { hipSuccess = 0, hipErrorNotReady = 600, hipErrorCpu = 1 };
enum { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2, hipHostMallocDefault = 0, hipStreamNonBlocking = 1,
       hipEventDisableTiming = 2, hipStreamCaptureModeThreadLocal = 1 };
typedef struct cpu_stream *hipStream_t;
typedef struct cpu_event *hipEvent_t;
typedef struct cpu_graph *hipGraph_t;
typedef struct cpu_exec *hipGraphExec_t;

hipError_t cpu_malloc(void **p, size_t n);
hipError_t hipFree(void *p);
template <typename V> static inline hipError_t hipMalloc(V **p, size_t n) { return cpu_malloc((void **)p, n); }
static inline hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return cpu_malloc(p, n); }
static inline hipError_t hipHostFree(void *p) { return hipFree(p); }
static inline hipError_t hipMemset(void *p, int v, size_t n) { memset(p, v, n); return hipSuccess; }
static inline hipError_t hipMemcpy(void *d, const void *s, size_t n, int)
{
  if (n) memcpy(d, s, n);
  return hipSuccess;
}
static inline hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, int k, hipStream_t) { return hipMemcpy(d, s, n, k); }
template <typename V> static inline hipError_t hipGetSymbolAddress(void **p, V *s) { *p = (void *)s; return hipSuccess; }
static inline hipError_t hipSetDevice(int) { return hipSuccess; }
static inline hipError_t hipDeviceSynchronize() { return hipSuccess; }
// (an error at every look with CPU_HIP_ERROR=1)
static inline hipError_t hipGetLastError()
{
  const char *e = getenv("CPU_HIP_ERROR");
  return e && e[0] == '1' ? hipErrorCpu : hipSuccess;
}
static inline const char *hipGetErrorString(hipError_t) { return "cpu"; }
static inline hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = (hipStream_t)malloc(1); return hipSuccess; }
static inline hipError_t hipStreamDestroy(hipStream_t s) { free(s); return hipSuccess; }
static inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
static inline hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
static inline hipError_t hipStreamBeginCapture(hipStream_t, int) { return hipErrorCpu; }  // every run launches
static inline hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *) { return hipErrorCpu; }
static inline hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, void *, char *, size_t) { return hipErrorCpu; }
static inline hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorCpu; }
static inline hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
static inline hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
static inline hipError_t hipEventCreate(hipEvent_t *e) { *e = (hipEvent_t)malloc(1); return hipSuccess; }
static inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
static inline hipError_t hipEventDestroy(hipEvent_t e) { free(e); return hipSuccess; }
static inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
static inline hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
static inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
static inline hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 1.0f; return hipSuccess; }

// One launch: run(ctx) is one thread's work.
void cpu_launch(dim3 grid, dim3 block, void (*run)(void *), void *ctx);

template <typename... P, typename... A> static inline void cpu_call(void (*f)(P...), dim3 g, dim3 b, A &&...a)
{
  struct Call { void (*f)(P...); std::tuple<P...> a; } c{f, std::tuple<P...>(static_cast<P>(a)...)};
  cpu_launch(g, b, [](void *p) { std::apply(static_cast<Call *>(p)->f, static_cast<Call *>(p)->a); }, &c);
}
#define hipLaunchKernelGGL(k, g, b, lds, s, ...) cpu_call(k, g, b, __VA_ARGS__)
