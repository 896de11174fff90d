// What the attention kernels need of HIP, on the host: a launch runs a workgroup's threads one after another, each to its end. The
// numbers mean nothing (products leave their sums as they are, loads of global memory give zeros); where LDS is read and written
// and how many barriers came before hangs on sizes and thread numbers alone, and trace.cpp keeps a record of it.
#pragma once
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#define __global__
#define __device__
#define __host__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __shared__ static __attribute__((section("lds")))

struct dim3 {
  unsigned x, y, z;
  dim3(unsigned a = 1, unsigned b = 1, unsigned c = 1) : x(a), y(b), z(c) {}
};
struct uint2 { unsigned x, y; };
struct uint4 { unsigned x, y, z, w; };
struct float4 { float x, y, z, w; };
static inline float4 make_float4(float a, float b, float c, float d) { return {a, b, c, d}; }
static inline uint2 make_uint2(unsigned a, unsigned b) { return {a, b}; }
extern dim3 threadIdx, blockIdx, blockDim, gridDim;

typedef void* hipStream_t;
typedef int hipError_t;
constexpr int hipSuccess = 0;
static inline int hipGetLastError() { return 0; }

// trace.cpp
#define LDS_TRACE
void barrier();
void lds_request(void* p);  // 16 bytes that memory writes there until a wait retires the request
unsigned lds_offset(const void* p);
void lds_request_at(unsigned at);  // the same by its offset
void lds_wait(int newest);  // all of the thread's requests but its newest ones are retired
void run(dim3 grid, dim3 block, void (*thread)(void*), void* what);
extern float trace_weight;                      // what exp2 gives: large, and all sums of softmax weights overflow
static inline void __syncthreads() { barrier(); }
template <class F, class... A>
void launch(F f, dim3 grid, dim3 block, A... a) {
  auto go = [=] { f(a...); };
  run(grid, block, [](void* p) { (*static_cast<decltype(go)*>(p))(); }, &go);
}
#define hipLaunchKernelGGL(f, grid, block, lds, stream, ...) launch(f, grid, block, __VA_ARGS__)

template <class T> T __shfl_xor(T v, int, int) { return v; }
static inline int __any(int v) { return v; }
static inline float __uint_as_float(uint32_t u) { float f; memcpy(&f, &u, 4); return f; }
#define __expf expf
template <class T> T min(T a, T b) { return a < b ? a : b; }
template <class T> T max(T a, T b) { return a < b ? b : a; }

typedef float v16f __attribute__((ext_vector_type(16)));
typedef __bf16 v8b __attribute__((ext_vector_type(8)));
typedef __bf16 v4b __attribute__((ext_vector_type(4)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));
struct __amdgpu_buffer_rsrc_t {};
#define __builtin_amdgcn_readfirstlane(x) (x)
#define __builtin_amdgcn_exp2f(x) ((void)(x), trace_weight)
#define __builtin_amdgcn_rcpf(x) (1.f / (x))
#define __builtin_amdgcn_sched_barrier(x) ((void)0)
#define __builtin_amdgcn_sched_group_barrier(...) ((void)0)
#define __builtin_amdgcn_make_buffer_rsrc(...) __amdgpu_buffer_rsrc_t()
#define __builtin_amdgcn_raw_buffer_load_b128(...) v4u(0)
#define __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, ...) ((void)(a), (void)(b), (c))
#define __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, ...) ((void)(a), (void)(b), (c))
#define __builtin_amdgcn_s_barrier() barrier()
#define __builtin_amdgcn_s_setprio(x) ((void)0)
#define __builtin_amdgcn_fdot2(a, b, c, ...) (c)
#define __builtin_amdgcn_fdot2_f32_bf16(a, b, c, ...) (c)
static inline v4b __builtin_amdgcn_ds_read_tr16_b64_v4bf16(const __attribute__((address_space(3))) v4b* p) {
  return *reinterpret_cast<const v4b*>(reinterpret_cast<uintptr_t>(p));
}
