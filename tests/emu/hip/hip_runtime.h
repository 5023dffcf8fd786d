// Stand-in for the HIP headers with which the library's sources build for the CPU: lanes are
// fibers, work-groups run one after another, device memory and LDS are host memory under the
// address sanitizer, and the runtime's calls are logged and can be made to fail.
#pragma once
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>

using std::max;
using std::min;
#define __device__
#define __host__
#define __global__
#define __shared__ static
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __align__(n) __attribute__((aligned(n)))
#define amdgpu_waves_per_eu(...) unused

struct int2 { int x, y; };
struct int4 { int x, y, z, w; };
struct double2 { double x, y; };
inline int2 make_int2(int a, int b) { return {a, b}; }
inline int4 make_int4(int a, int b, int c, int d) { return {a, b, c, d}; }
struct dim3 {
    unsigned x, y, z;
    dim3(unsigned a = 1, unsigned b = 1, unsigned c = 1) : x(a), y(b), z(c) {}
};

typedef int hipError_t;
enum { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorUnknown = 999 };
struct EmuStream { int id, capture; };
struct EmuEvent { int id; };
typedef EmuStream *hipStream_t;
typedef EmuEvent *hipEvent_t;
typedef struct EmuGraph *hipGraph_t;
typedef struct EmuGraphExec *hipGraphExec_t;
enum { hipMemcpyHostToDevice, hipMemcpyDeviceToHost, hipMemcpyDeviceToDevice };
enum { hipStreamNonBlocking, hipEventDisableTiming, hipFuncAttributeMaxDynamicSharedMemorySize, hipStreamCaptureModeThreadLocal };
enum hipStreamCaptureStatus { hipStreamCaptureStatusNone, hipStreamCaptureStatusActive };

namespace emu {
extern dim3 tIdx, bIdx, bDim, gDim;
extern unsigned char *dyn_lds;
// runs fn for every lane of every work-group, or only logs the launch (emu_execute(0))
void launch(const char *name, dim3 g, dim3 b, size_t lds, hipStream_t s, const std::function<void()> &fn);
void wave_barrier();
void block_barrier();
uint64_t exchange(uint64_t v, int off);
uint64_t broadcast(uint64_t v, int src);
unsigned long long ballot(bool p);
int lane();
// logs a runtime call; what it returns (hipSuccess unless emu_fail chose this call)
hipError_t call(const char *name, int stream = -1, int object = -1);
template <class T> uint64_t bits(T v) { uint64_t u = 0; memcpy(&u, &v, sizeof v); return u; }
template <class T> T value(uint64_t u) { T v; memcpy(&v, &u, sizeof v); return v; }
inline int stream_id(hipStream_t s) { return s ? s->id : 0; }
}  // namespace emu

#define threadIdx emu::tIdx
#define blockIdx emu::bIdx
#define blockDim emu::bDim
#define gridDim emu::gDim
template <class T> T __shfl_xor(T v, int off, int) { return emu::value<T>(emu::exchange(emu::bits(v), off)); }
template <class T> T __shfl(T v, int src, int) { return emu::value<T>(emu::broadcast(emu::bits(v), src)); }
inline unsigned long long __ballot(bool p) { return emu::ballot(p); }
inline int __popcll(unsigned long long m) { return __builtin_popcountll(m); }
inline void __syncthreads() { emu::block_barrier(); }
template <class T> T atomicAdd(T *p, T v) { T o = *p; *p += v; return o; }
template <class T> T unsafeAtomicAdd(T *p, T v) { return atomicAdd(p, v); }
#define __HIP_MEMORY_SCOPE_WORKGROUP 0
#define __hip_atomic_fetch_add(p, v, order, scope) atomicAdd(p, v)
#define __builtin_amdgcn_fence(...) (void)0
#define __builtin_amdgcn_wave_barrier() emu::wave_barrier()
inline int __builtin_amdgcn_readfirstlane(int v) { return v; }
inline unsigned emu_mbcnt_lo(unsigned m, unsigned base)
{
    const int l = emu::lane();
    return base + __builtin_popcount(l >= 32 ? m : m & ((1u << l) - 1));
}
inline unsigned emu_mbcnt_hi(unsigned m, unsigned base)
{
    const int l = emu::lane();
    return base + (l <= 32 ? 0 : __builtin_popcount(m & ((1u << (l - 32)) - 1)));
}
#define __builtin_amdgcn_mbcnt_lo emu_mbcnt_lo
#define __builtin_amdgcn_mbcnt_hi emu_mbcnt_hi

// ---- runtime
inline hipError_t hipMalloc(void **p, size_t n)
{
    *p = nullptr;
    if (hipError_t e = emu::call("hipMalloc")) return e;
    *p = malloc(n);
    memset(*p, 0xc3, n);
    return hipSuccess;
}
inline hipError_t hipFree(void *p) { free(p); return emu::call("hipFree"); }
inline hipError_t hipMemcpy(void *d, const void *s, size_t n, int) { memcpy(d, s, n); return emu::call("hipMemcpy"); }
inline hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, int, hipStream_t) { return hipMemcpy(d, s, n, 0); }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned);
inline hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
inline hipError_t hipEventDestroy(hipEvent_t e) { delete e; return emu::call("hipEventDestroy"); }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { return emu::call("hipEventRecord", emu::stream_id(s), e->id); }
inline hipError_t hipEventElapsedTime(float *t, hipEvent_t, hipEvent_t) { *t = 0.0f; return hipSuccess; }
inline hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) { return emu::call("hipStreamWaitEvent", emu::stream_id(s), e->id); }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned);
inline hipError_t hipStreamDestroy(hipStream_t s) { const int id = s->id; delete s; return emu::call("hipStreamDestroy", id); }
inline hipError_t hipStreamSynchronize(hipStream_t s) { return emu::call("hipStreamSynchronize", emu::stream_id(s)); }
inline hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *st)
{
    *st = s && s->capture ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
// (a captured build runs at its capture: its graph holds nothing)
inline hipError_t hipStreamBeginCapture(hipStream_t s, int) { s->capture = 1; return emu::call("hipStreamBeginCapture", s->id); }
inline hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t *g)
{
    s->capture = 0;
    const hipError_t e = emu::call("hipStreamEndCapture", s->id);
    *g = e ? nullptr : reinterpret_cast<hipGraph_t>(s);
    return e;
}
inline hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t g, void *, char *, size_t)
{
    *x = reinterpret_cast<hipGraphExec_t>(g);
    return emu::call("hipGraphInstantiate");
}
inline hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t s) { return emu::call("hipGraphLaunch", emu::stream_id(s)); }
inline hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
inline hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGetLastError();  // of the launches (and calls) since the last
inline hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
inline hipError_t hipFuncSetAttribute(const void *, int, int) { return hipSuccess; }
inline const char *hipGetErrorString(int) { return "injected"; }
#define HIP_SYMBOL(x) (x)
inline hipError_t hipGetSymbolAddress(void **p, void *s) { *p = s; return hipSuccess; }
