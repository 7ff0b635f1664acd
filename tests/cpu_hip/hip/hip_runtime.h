// A host stand-in for the HIP runtime, for tests that run the library's kernels
// on the CPU: one workgroup after another, a work-item per coroutine, with
// guard pages behind every device allocation and array bounds checked
// (emu.cpp, cpu_library.py).  Only what the library uses.
#pragma once
#include <cmath>
#include <cstddef>
#include <cstdint>
#include <cstdlib>
#include <functional>

#define __global__
#define __device__
#define __host__
#define __constant__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __align__(n) __attribute__((aligned(n)))
#define __shared__ thread_local  // one workgroup at a time on the calling thread
#define amdgpu_waves_per_eu(n)
#define HIP_SYMBOL(x) (&(x))
#define __HIP_MEMORY_SCOPE_SYSTEM 0
#define __HIP_MEMORY_SCOPE_AGENT 0
#undef __hip_atomic_store
#undef __hip_atomic_load
#define __hip_atomic_store(p, v, order, scope) ((void)(*(p) = (v)))
#define __hip_atomic_load(p, order, scope) (*(p))
#define __threadfence_system() ((void)0)
#define __threadfence() ((void)0)

struct dim3 {
  unsigned x, y, z;
  dim3(unsigned a = 1, unsigned b = 1, unsigned c = 1) : x(a), y(b), z(c) {}
};
#define EMU_VEC2(T, name, al) struct alignas(al) name { T x, y; }; \
  inline name make_##name(T x, T y) { return name{x, y}; }
#define EMU_VEC4(T, name, al) struct alignas(al) name { T x, y, z, w; }; \
  inline name make_##name(T x, T y, T z, T w) { return name{x, y, z, w}; }
EMU_VEC2(double, double2, 16)
EMU_VEC2(float, float2, 8)
EMU_VEC2(int, int2, 8)
EMU_VEC2(unsigned, uint2, 8)
EMU_VEC2(unsigned short, ushort2, 4)
EMU_VEC4(int, int4, 16)
EMU_VEC4(unsigned, uint4, 16)
EMU_VEC4(float, float4, 16)

// ---- work-item state and wavefront operations
namespace emu {
struct Index {
  unsigned x, y, z;
};
extern Index tid, bid, bdim, gdim;
void barrier();
// every lane of the wavefront gives n bytes and gets the 64 lanes' (stride 16 doubles)
const double *exchange(const void *mine, size_t n);
void run(const void *kernel, dim3 grid, dim3 block, size_t lds, const std::function<void()> &body);
inline int lane() { return tid.x & 63; }
template <class T>
inline T shfl(T v, int src) {
  const double *all = exchange(&v, sizeof(T));
  T r;
  __builtin_memcpy(&r, all + 16 * src, sizeof(T));
  return r;
}
}  // namespace emu
#define threadIdx emu::tid
#define blockIdx emu::bid
#define blockDim emu::bdim
#define gridDim emu::gdim
inline void __syncthreads() { emu::barrier(); }
template <class T>
inline T __shfl(T v, int src, int w = 64) {
  return emu::shfl(v, (emu::lane() & ~(w - 1)) | (src & (w - 1)));
}
template <class T>
inline T __shfl_xor(T v, int m, int = 64) {
  return emu::shfl(v, emu::lane() ^ m);
}
template <class T>
inline T __shfl_up(T v, int d, int w = 64) {
  const int l = emu::lane();
  return emu::shfl(v, (l & (w - 1)) >= d ? l - d : l);
}
unsigned long long __ballot(bool p);
inline int __popcll(unsigned long long x) { return __builtin_popcountll(x); }
#define __builtin_amdgcn_readfirstlane(x) (x)  // used on uniform values only
#define __builtin_amdgcn_sched_barrier(x) ((void)0)
typedef double emu_double4 __attribute__((ext_vector_type(4)));
emu_double4 emu_mfma_f64(double a, double b, emu_double4 c);
#define __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, x, y, z) emu_mfma_f64(a, b, c)
template <class C>
inline C emu_absent(C) {
  std::abort();  // the reduced-precision products are not run here
}
#define __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, x, y, z) emu_absent(c)
#define __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, x, y, z) emu_absent(c)
#define __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, x, y, z) emu_absent(c)
template <class T>
inline T atomicAdd(T *p, T v) {
  const T old = *p;
  *p = old + v;
  return old;
}
inline double unsafeAtomicAdd(double *p, double v) { return atomicAdd(p, v); }
#define EMU_MINMAX(T)                                      \
  inline T min(T a, T b) { return b < a ? b : a; }         \
  inline T max(T a, T b) { return a < b ? b : a; }
EMU_MINMAX(int)
EMU_MINMAX(unsigned)
EMU_MINMAX(long)
EMU_MINMAX(long long)
EMU_MINMAX(unsigned long)
EMU_MINMAX(double)
EMU_MINMAX(float)
inline long long min(long long a, int b) { return min(a, (long long)b); }
inline long long max(long long a, int b) { return max(a, (long long)b); }
using std::abs;

// ---- runtime
enum hipError_t {
  hipSuccess = 0,
  hipErrorInvalidValue = 1,
  hipErrorOutOfMemory = 2,
  hipErrorNotReady = 600,
  hipErrorNotSupported = 801
};
typedef struct emu_stream *hipStream_t;
typedef struct emu_event *hipEvent_t;
typedef struct emu_graph *hipGraph_t;
typedef struct emu_graphexec *hipGraphExec_t;
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost, hipMemcpyDeviceToDevice };
enum hipDeviceAttribute_t { hipDeviceAttributeMaxSharedMemoryPerBlock };
enum hipFuncAttribute { hipFuncAttributeMaxDynamicSharedMemorySize };
enum hipStreamCaptureMode { hipStreamCaptureModeThreadLocal };
enum { hipStreamNonBlocking = 1, hipEventDisableTiming = 2 };
enum { hipHostMallocDefault = 0, hipHostMallocMapped = 2, hipHostMallocCoherent = 0x40000000 };
extern "C" {
hipError_t emu_malloc(void **p, size_t n, int host);
hipError_t hipFree(void *p);
hipError_t hipHostFree(void *p);
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned flags);
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k);
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st);
hipError_t hipMemset(void *d, int v, size_t n);
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t st);
hipError_t hipGetLastError();
const char *hipGetErrorString(hipError_t e);
hipError_t hipSetDevice(int d);
hipError_t hipGetDevice(int *d);
hipError_t hipDeviceSynchronize();
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int d);
hipError_t hipFuncSetAttribute(const void *f, hipFuncAttribute a, int v);
hipError_t hipStreamCreate(hipStream_t *s);
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned flags);
hipError_t hipStreamDestroy(hipStream_t s);
hipError_t hipStreamSynchronize(hipStream_t s);
hipError_t hipStreamQuery(hipStream_t s);
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned flags);
hipError_t hipEventCreate(hipEvent_t *e);
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned flags);
hipError_t hipEventDestroy(hipEvent_t e);
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s);
hipError_t hipEventSynchronize(hipEvent_t e);
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b);
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode m);
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t *g);
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t g, void *n, char *log, size_t z);
hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t s);
hipError_t hipGraphDestroy(hipGraph_t g);
hipError_t hipGraphExecDestroy(hipGraphExec_t x);
}
template <class T>
inline hipError_t hipMalloc(T **p, size_t n) {
  return emu_malloc((void **)p, n, 0);
}
template <class T>
inline hipError_t hipHostMalloc(T **p, size_t n, unsigned = 0) {
  return emu_malloc((void **)p, n, 1);
}
template <class T>
inline hipError_t hipGetSymbolAddress(void **p, T *s) {
  *p = (void *)s;
  return hipSuccess;
}
template <class F, class... A>
inline void hipLaunchKernelGGL(F kernel, dim3 g, dim3 b, size_t lds, hipStream_t, A... a) {
  emu::run((const void *)kernel, g, b, lds, [&] { kernel(a...); });
}
template <class F, class... A>
inline void hipExtLaunchKernelGGL(F kernel, dim3 g, dim3 b, size_t lds, hipStream_t, hipEvent_t, hipEvent_t, unsigned,
                                  A... a) {
  emu::run((const void *)kernel, g, b, lds, [&] { kernel(a...); });
}
