// Kernels of the compile-time transform lengths: every even length from
// PNH_CT_MIN to PNH_CT_MAX with a three-radix schedule.  This source is
// compiled once per part (PNH_CT_PART of PNH_CT_PARTS), the lengths dealt in
// turn.
#include "fft_ct.h"

#include <utility>

namespace {

template <typename T, int N, bool FAST>
__global__ void __launch_bounds__(512)
fft_ct_kernel(FftDesc d, const void* in_, void* out_, const void* __restrict__ tw_,
              const int* __restrict__ skip) {
  if (skip && *skip) return;
  extern __shared__ unsigned char smem_raw[];
  fft_ct_body<T, N, FAST>(d, in_, out_, tw_, xcd_unit(blockIdx.x, gridDim.x), smem_raw);
}

template <typename T, int N>
int launch_ct(const FftDesc& d, const void* in, void* out, const void* tw, const int* skip,
              hipStream_t s) {
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3((unsigned)d.n_blocks), dim3(d.threads), d.lds, s, d, in, out, tw,
                       skip);
    PNH_LAUNCH_CHECK();
    return 0;
  };
  return d.inner_major ? go(fft_ct_kernel<T, N, true>) : go(fft_ct_kernel<T, N, false>);
}

typedef int (*CtLaunch)(const FftDesc&, const void*, void*, const void*, const int*,
                        hipStream_t);

constexpr int kLengths = (PNH_CT_MAX - PNH_CT_MIN) / 2 / PNH_CT_PARTS + 1;

template <typename T, int I>
constexpr CtLaunch entry() {
  constexpr int N = PNH_CT_MIN + 2 * (I * PNH_CT_PARTS + PNH_CT_PART);
  if constexpr (N <= PNH_CT_MAX && radices_of(N).r[0] > 0) return launch_ct<T, N>;
  else return nullptr;
}

template <typename T, int... I>
CtLaunch lookup(int i, std::integer_sequence<int, I...>) {
  static constexpr CtLaunch table[] = {entry<T, I>()...};
  return table[i];
}

}  // namespace

#define PNH_CT_NAME2(p) pnh_fft_ct_part##p
#define PNH_CT_NAME(p) PNH_CT_NAME2(p)

int PNH_CT_NAME(PNH_CT_PART)(const FftDesc& d, int fp64, const void* in, void* out,
                             const void* tw, const int* skip, hipStream_t s) {
  const int i = (d.n - PNH_CT_MIN) / 2 / PNH_CT_PARTS;
  typedef std::make_integer_sequence<int, kLengths> Seq;
  const CtLaunch f = fp64 ? lookup<double>(i, Seq()) : lookup<float>(i, Seq());
  if (!f) {
    pnh_set_error("no compiled transform of length %d", d.n);
    return -2;
  }
  return f(d, in, out, tw, skip, s);
}
