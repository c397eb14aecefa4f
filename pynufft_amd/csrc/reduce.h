// Sum over a workgroup of 256 threads, shared by the sources that must get the
// same bits from the same partial sums.
#pragma once
#include <hip/hip_runtime.h>

namespace {

// Every thread gets the total; a fixed tree.  red: 4 words of LDS, free again
// on return.  (Shuffles and two barriers: the solve's kernels are a few
// microseconds long, and a tree in LDS is nine barriers.)
__device__ __forceinline__ double2 sum_block256(double2 v, double2* red) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    v.x += __shfl_xor(v.x, off, 64);
    v.y += __shfl_xor(v.y, off, 64);
  }
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  v.x = (red[0].x + red[1].x) + (red[2].x + red[3].x);
  v.y = (red[0].y + red[1].y) + (red[2].y + red[3].y);
  __syncthreads();
  return v;
}

}  // namespace
