// Exact fixed-point accumulation in LDS (see the gridding kernels) and small
// helpers shared by the interpolation sources.
#pragma once
#include "common.h"

namespace {

constexpr int kMaxItemRows = 4096;
constexpr int kFixBits = 50;
constexpr int kPackBits = 30;

// Adding 1.5 * 2^52 to a double of magnitude below 2^51 rounds it to the
// nearest integer and leaves that integer in the low mantissa bits; the low
// word of the constant's bits is zero, so subtracting them is one 32-bit
// subtract of the high word.
constexpr double kMagic = 6755399441055744.0;
constexpr long long kMagicBits = 0x4338000000000000LL;

__device__ __forceinline__ void lds_add(long long* p, long long v) {
  __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

__device__ __forceinline__ double2 to_d2(float2 v) { return make_double2(v.x, v.y); }
__device__ __forceinline__ double2 to_d2(double2 v) { return v; }

// a * b in FP64 (fused multiply-adds)
__device__ __forceinline__ double2 dmul(double2 a, double2 b) {
  return make_double2(__builtin_fma(a.x, b.x, -(a.y * b.y)), __builtin_fma(a.x, b.y, a.y * b.x));
}

// Packed accumulator word of rounded parts re, im (each already offset by
// 1.5 * 2^52, magnitude below 2^31): re + im * 2^32 modulo 2^64.  re's bits
// minus the constant's are re as a 64-bit integer (sign included); im
// enters through its low word only.  The constant's low word is zero, so the
// low word is re's and the high word is one three-operand 32-bit add (written
// out: the compiler otherwise forms a 64-bit add and a second 32-bit add).
__device__ __forceinline__ long long pack_fixed(double re, double im) {
  const unsigned long long rb = (unsigned long long)__double_as_longlong(re);
  const unsigned neg_magic_hi = 0u - (unsigned)((unsigned long long)kMagicBits >> 32);
  unsigned hi;
  asm("v_add3_u32 %0, %1, %2, %3"
      : "=v"(hi)
      : "v"((unsigned)(rb >> 32)), "v"((unsigned)__double_as_longlong(im)), "s"(neg_magic_hi));
  return (long long)(((unsigned long long)hi << 32) | (rb & 0xffffffffull));
}

// Real and imaginary sums of a packed accumulator word.
__device__ __forceinline__ void unpack_fixed(long long v, long long& re, long long& im) {
  re = (long long)(int)(unsigned)(unsigned long long)v;
  im = (long long)((unsigned long long)v - (unsigned long long)re) >> 32;
}

// Max over the workgroup; `red` holds one slot per wave.
template <typename T>
__device__ __forceinline__ T block_max(T v, T* red) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off, 64));
  const int wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  if ((threadIdx.x & 63) == 0) red[wave] = v;
  __syncthreads();
  T r = red[0];
  for (int w = 1; w < nw; ++w) r = fmax(r, red[w]);
  return r;
}

constexpr int kPoisonExp = 0x7fffffff;

// Dynamic LDS above 64 KB must be allowed per kernel before the launch.
template <typename K>
void allow_lds(K kernel, size_t bytes) {
  if (bytes > 65536)
    (void)hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)bytes);
}

}  // namespace
