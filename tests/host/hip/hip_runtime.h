// Host stand-ins for the device language, for kernel_bounds.cpp: every thread of a workgroup is a
// fiber, and a barrier (or a wavefront's fence or shuffle) runs the others up to it.
#pragma once
#include <cmath>
#include <cstdint>
#include <cstring>

#define __device__
#define __host__
#define __global__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __shared__ thread_local  // one copy for the program's one thread, and valid after extern
#define __restrict__

struct dim3 {
  unsigned x = 1, y = 1, z = 1;
  dim3() = default;
  dim3(unsigned a, unsigned b = 1, unsigned c = 1) : x(a), y(b), z(c) {}
};
extern dim3 threadIdx, blockIdx, blockDim, gridDim;

void host_block_barrier();
void host_wave_barrier();
double host_wave_xor(double v, int mask);

inline void __syncthreads() { host_block_barrier(); }
template <class T> inline T __shfl_xor(T v, int mask) { return (T)host_wave_xor((double)v, mask); }
inline uint32_t __umulhi(uint32_t a, uint32_t b) { return (uint32_t)(((uint64_t)a * b) >> 32); }
template <class T> inline T atomicAdd(T* p, T v) {
  const T o = *p;
  *p += v;
  return o;
}
// a wave's lanes meet at the barrier between the two fences
#define __builtin_amdgcn_fence(...) ((void)0)
#define __builtin_amdgcn_wave_barrier() host_wave_barrier()
#define __builtin_amdgcn_readfirstlane(x) (x)
using std::copysign;
using std::exp;
using std::fabs;
using std::fma;
using std::hypot;
using std::isfinite;
using std::isinf;
using std::sqrt;
