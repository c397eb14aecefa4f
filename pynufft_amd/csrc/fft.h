// Line-FFT descriptor shared by the planner (api.hip) and the kernel.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#define PNH_FFT_MAX_PASS 16
// Lengths with kernels compiled for them: even, with a three-radix schedule.
#define PNH_CT_MIN 32
#define PNH_CT_MAX 1024
#define PNH_CT_PARTS 7

// Addressing of one side (source or destination) of a line transform.  Line
// (o0, o1, b), element t lives at o0*o_stride[0] + o1*o_stride[1] +
// b*b_stride + t*t_stride (in elements).
struct FftSide {
  int64_t o_stride[2];
  int64_t b_stride;
  int64_t t_stride;
};

struct FftDesc {
  int n;                // transform length
  int n_in;             // valid input elements per line (rest are zero)
  int n_out;            // outputs kept per line
  int sign;             // -1 forward, +1 inverse
  double scale;         // applied on store
  int64_t n_outer;      // outer lines (split as o0 * o_split + o1)
  int64_t o_split;
  int64_t n_inner;      // inner (contiguous-stride) lines
  FftSide src, dst;
  int sn_side;          // 0 none, 1 multiply on load, 2 multiply on store
  const void* sn;       // real apodization (float or double, matches dtype)
  int64_t sn_o_stride[2];
  int64_t sn_t_stride;
  // per-point factor along the transformed axis (complex, matches dtype), or
  // NULL: the forward transform multiplies point t of its output by mod[t],
  // the inverse point t of its input by conj(mod[t])
  const void* mod;
  int npass;
  uint64_t radices;     // pass p's radix - 1 in bits 4p .. 4p + 3
  int lines_per_block;
  int threads;
  int inner_major;      // 1: threads walk lines fastest (strided axis)
  int ct;               // 1: a kernel is compiled for this length
  int64_t n_blocks;     // workgroups of a launch
  uint32_t lds;         // bytes of LDS of a workgroup
  // compile-time kernels: lines per workgroup as a power of two, workgroups
  // per outer line (inner_major), and the multipliers of the divisions by it,
  // by n_inner and by o_split
  int lg_lines;
  uint32_t blocks_inner;
  uint32_t mul_blocks, mul_inner, mul_split;
  int sh_blocks, sh_inner, sh_split;
};

int pnh_fft_launch(const FftDesc& d, int fp64, const void* in, void* out,
                   const void* tw, const int* skip, hipStream_t stream);
int pnh_fft_factor(int n, uint64_t* radices, int* npass);
__host__ __device__ inline int pnh_fft_radix(uint64_t radices, int p) {
  return (int)(radices >> (4 * p) & 15) + 1;
}
// Line length in elements of the LDS-resident limit of a transform.
__host__ __device__ inline int pnh_fft_lds_line(int n) { return n + (n >> 4) + 1; }
// Line stride in LDS: one pad element per 16 (bank spreading of a line's
// points), odd (bank spreading of the same point of neighbouring lines).
__host__ __device__ inline int pnh_fft_lds_stride(int n) { return (n + (n >> 4) + 1) | 1; }
// Multiplier and shift of the division by d (div_magic).
void pnh_fft_magic(uint32_t d, uint32_t* mul, int* shift);
// Butterflies of a compiled length's first pass, per line.
int pnh_fft_first_pass(int n);
// Threads of a workgroup for a descriptor whose other fields are set.
int pnh_fft_threads(const FftDesc& d);
// Whether a kernel is compiled for transforms of length n.
bool pnh_fft_has_ct(int n);
// LDS bytes of one workgroup: the twiddle table and two line buffers (one
// for a compiled two-pass length).
size_t pnh_fft_lds_bytes(const FftDesc& d, int fp64);
void pnh_fft_allow_lds(const void* kernel, size_t bytes);
