// A HIP runtime on the host, for tests without a device: device memory is heap memory of
// the exact size asked for (so AddressSanitizer reports an access outside a buffer), a
// stream runs each call at once, and a kernel launch runs its workgroups one after the
// other, each lane on a stack of its own (simt.cpp). Barriers hold the workgroup's lanes,
// ballots and shuffles the wave's; lanes and workgroups run in a shuffled order. Built with
// g++, so only kernels free of machine builtins can be linked.
#pragma once

#include <cmath>
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <functional>

#define __device__
#define __host__
#define __global__
#define __forceinline__ inline
#define __launch_bounds__(x)
#define __shared__ static

struct alignas(8) float2 { float x, y; };
struct alignas(16) float4 { float x, y, z, w; };
struct alignas(8) int2 { int x, y; };
struct alignas(16) int4 { int x, y, z, w; };
struct alignas(16) uint4 { unsigned x, y, z, w; };
inline float2 make_float2(float a, float b) { return {a, b}; }
inline float4 make_float4(float a, float b, float c, float d) { return {a, b, c, d}; }
inline int2 make_int2(int a, int b) { return {a, b}; }
inline int4 make_int4(int a, int b, int c, int d) { return {a, b, c, d}; }
inline uint4 make_uint4(unsigned a, unsigned b, unsigned c, unsigned d) { return {a, b, c, d}; }
struct dim3 {
  unsigned x = 1, y = 1, z = 1;
  dim3() = default;
  dim3(unsigned a) : x(a) {}
};
extern dim3 threadIdx, blockIdx, gridDim, blockDim;

inline int __float_as_int(float f) { int i; std::memcpy(&i, &f, 4); return i; }
inline float __int_as_float(int i) { float f; std::memcpy(&f, &i, 4); return f; }
inline unsigned __float_as_uint(float f) { unsigned i; std::memcpy(&i, &f, 4); return i; }
inline float __uint_as_float(unsigned i) { float f; std::memcpy(&f, &i, 4); return f; }
inline int __popcll(unsigned long long m) { return __builtin_popcountll(m); }
inline int __ffsll(long long m) { return __builtin_ffsll(m); }
template <class T>
T atomicAdd(T* p, T v) { const T o = *p; *p = o + v; return o; }
template <class T>
T atomicExch(T* p, T v) { const T o = *p; *p = v; return o; }

namespace simt {
enum class Op { kBarrier, kBallot, kShfl };
// Blocks the running lane until its workgroup (kBarrier) or the wave's lanes at the same
// `site` have arrived. kBallot returns the mask of lanes with value != 0, kShfl the value of
// lane `src`; a shuffle from a lane that is not there ends the program.
unsigned long long wait(Op op, unsigned long long value, int src, int site);
void launch(dim3 grid, dim3 block, const std::function<void()>& lane);
extern size_t room;  // the largest device allocation that succeeds
}  // namespace simt

inline void __syncthreads(int site = __builtin_LINE()) { simt::wait(simt::Op::kBarrier, 0, 0, site); }
inline unsigned long long __ballot(int b, int site = __builtin_LINE()) {
  return simt::wait(simt::Op::kBallot, b != 0, 0, site);
}
inline int __shfl(int v, int src, int /*width*/ = 64, int site = __builtin_LINE()) {
  return (int)simt::wait(simt::Op::kShfl, (unsigned)v, src & 63, site);
}
inline unsigned __shfl_up(unsigned v, int n, int /*width*/ = 64, int site = __builtin_LINE()) {
  const int lane = threadIdx.x & 63;
  return (unsigned)simt::wait(simt::Op::kShfl, v, lane >= n ? lane - n : lane, site);
}

template <class... P, class... A>
void hipLaunchKernelGGL(void (*kernel)(P...), dim3 grid, dim3 block, size_t, void*, A... args) {
  simt::launch(grid, block, [&] { kernel(args...); });
}

typedef void* hipStream_t;
typedef void* hipEvent_t;
enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2 };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost, hipMemcpyDeviceToDevice };
enum { hipHostMallocDefault = 0, hipStreamDefault = 0, hipStreamNonBlocking = 1 };
struct hipDeviceProp_t {
  int multiProcessorCount;
  size_t totalGlobalMem;
  char gcnArchName[256];
};
hipError_t hipMalloc(void** p, size_t n);
hipError_t hipFree(void* p);
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return hipMalloc(p, n); }
inline hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind);
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) {
  return hipMemcpy(d, s, n, k);
}
hipError_t hipMemset(void* d, int v, size_t n);
inline hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return hipMemset(d, v, n); }
hipError_t hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h,
                            hipMemcpyKind, hipStream_t);
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int);
inline hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline const char* hipGetErrorString(hipError_t e) { return e == hipSuccess ? "ok" : "error"; }
inline hipError_t hipDeviceSynchronize() { return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipStreamCreateWithFlags(hipStream_t*, unsigned) { return hipErrorInvalidValue; }
inline hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
inline hipError_t hipEventCreate(hipEvent_t*) { return hipErrorInvalidValue; }
inline hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventElapsedTime(float*, hipEvent_t, hipEvent_t) { return hipErrorInvalidValue; }
