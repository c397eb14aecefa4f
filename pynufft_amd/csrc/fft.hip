// LDS-resident Stockham FFT over lines of a strided N-d array (gfx950).
//
// One launch transforms every line along one axis.  A workgroup takes LB
// lines: the first radix pass reads global memory (zero-filling past n_in, so
// zero-padding is fused, and applying the real apodization factor sn:
// x2xx fused), the passes exchange through LDS, and the last one writes the
// first n_out outputs of each line (cropping, the scale and xx2x fused).
//
// Semantics follow numpy.fft: the forward kernel is exp(-2 pi i t/n), the
// inverse exp(+2 pi i t/n) with the 1/n factors folded into `scale`.  The
// butterflies are forward only: the inverse is conj(F(conj(x))), the
// conjugations riding on the load and the final scale.
//
// The lengths that plans use have kernels compiled for them (fft_ct.h);
// fft_lines_kernel below takes every other length, and the batches.
#include "fft_ct.h"

namespace {

// q = i / n and r = i % n for 0 <= i < 2^22 and 1 <= n, with rcp = 1.0f / n
// (the float estimate is off by at most one; one correction step fixes it)
__device__ __forceinline__ int fdivmod(int i, int n, float rcp, int& r) {
  int q = (int)((float)i * rcp);
  r = i - q * n;
  if (r < 0) { --q; r += n; }
  else if (r >= n) { ++q; r -= n; }
  return q;
}

// One Stockham radix-R pass over LB lines in LDS.  Butterfly (l, j), j <
// n/R, reads points j + r n/R for r < R, applies the twiddles of a stage
// after ns points, and writes points (j / ns) ns R + j % ns + r ns.
template <typename T, int R>
__device__ __forceinline__ void stockham_pass(int n, int LB, int ns, int ld,
                                              const typename cplx<T>::t* tw,
                                              const typename cplx<T>::t* src,
                                              typename cplx<T>::t* dst) {
  typedef typename cplx<T>::t C;
  const int nb = n / R;
  const int twstep = n / (ns * R);
  const int total = LB * nb;
  const float r_nb = 1.0f / (float)nb, r_ns = 1.0f / (float)ns;
  for (int idx = threadIdx.x; idx < total; idx += blockDim.x) {
    int j, k;
    const int l = fdivmod(idx, nb, r_nb, j);
    const int jq = fdivmod(j, ns, r_ns, k);
    const int kt = k * twstep;
    C v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int t = j + r * nb;
      v[r] = src[l * ld + t + (t >> 4)];
    }
#pragma unroll
    for (int r = 1; r < R; ++r) v[r] = cmul_fma(v[r], tw[r * kt]);
    Dft<T, R>::run(v);
    const int o = jq * ns * R + k;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int t = o + r * ns;
      dst[l * ld + t + (t >> 4)] = v[r];
    }
  }
}

// Any length of radices 2 to 16 (run-time schedule).  The lines are copied
// into LDS, transformed there between two buffers, and copied out, so the
// radix switch appears once (with it at the global ends too the kernel was
// 240 KB of code).  in_ and out_ may alias (in-place passes): a workgroup
// reads all its lines before its first store, and other workgroups own other
// lines.  LDS: the twiddle table, then two line buffers of
// LB x pnh_fft_lds_stride(n).
template <typename T>
__device__ __forceinline__ void fft_body(const FftDesc& d, const void* in_, void* out_,
                                         const void* __restrict__ tw_, int64_t blk,
                                         unsigned char* smem_raw) {
  typedef typename cplx<T>::t C;
  const int n = d.n, LB = d.lines_per_block;
  const int ld = pnh_fft_lds_stride(n);
  C* tws = reinterpret_cast<C*>(smem_raw);
  C* src = tws + n;
  C* dst = src + (size_t)LB * ld;
  const C* in = (const C*)in_;
  C* out = (C*)out_;
  const C* __restrict__ tw = (const C*)tw_;
  const int nthr = blockDim.x, tid = threadIdx.x;
  const int64_t line0 = blk * LB;
  const int64_t n_lines = d.n_outer * d.n_inner;
  const int nl = (int)(n_lines - line0 < LB ? n_lines - line0 : LB);  // lines present
  const bool fast = d.inner_major != 0;
  const float r_lb = 1.0f / (float)LB, r_n = 1.0f / (float)n;
  const T cj = d.sign > 0 ? (T)-1 : (T)1;         // inverse: conjugate in and out
  // source, destination and apodization offset of line l of the workgroup
  struct Line { int64_t src, dst, sn; };
  auto line = [&](int l) -> Line {
    const int64_t L = line0 + l;
    int64_t o, b, o0, o1;
    if (n_lines < (1LL << 31)) {
      const uint32_t ou = (uint32_t)L / (uint32_t)d.n_inner;
      o = ou;
      b = (uint32_t)L - ou * (uint32_t)d.n_inner;
      const uint32_t q = ou / (uint32_t)d.o_split;
      o0 = q;
      o1 = ou - q * (uint32_t)d.o_split;
    } else {
      o = L / d.n_inner; b = L - o * d.n_inner;
      o0 = o / d.o_split; o1 = o - o0 * d.o_split;
    }
    return Line{o0 * d.src.o_stride[0] + o1 * d.src.o_stride[1] + b * d.src.b_stride,
                o0 * d.dst.o_stride[0] + o1 * d.dst.o_stride[1] + b * d.dst.b_stride,
                o0 * d.sn_o_stride[0] + o1 * d.sn_o_stride[1]};
  };
  // element i of the copies: consecutive threads on consecutive lines along a
  // strided axis, else along the line
  auto point = [&](int i, int& t) -> int {
    int l;
    if (fast) t = fdivmod(i, LB, r_lb, l);
    else l = fdivmod(i, n, r_n, t);
    return l;
  };
  for (int i = tid; i < n; i += nthr) tws[i] = tw[i];
  const int total = LB * n;
#pragma unroll 4
  for (int i = tid; i < total; i += nthr) {
    int t;
    const int l = point(i, t);
    C v = mk<T>((T)0, (T)0);
    if (l < nl && t < d.n_in) {
      const Line li = line(l);
      v = in[li.src + (int64_t)t * d.src.t_stride];
      if (d.sn_side == 1) {
        const T s = ((const T*)d.sn)[li.sn + (int64_t)t * d.sn_t_stride];
        v.x *= s; v.y *= s;
      }
      if (d.mod && d.sign > 0) {
        C m = ((const C*)d.mod)[t];
        m.y = -m.y;
        v = cmul_fma(v, m);
      }
    }
    v.y *= cj;
    src[l * ld + t + (t >> 4)] = v;
  }
  int ns = 1;
  for (int p = 0; p < d.npass; ++p) {
    __syncthreads();
    const int R = pnh_fft_radix(d.radices, p);
    switch (R) {
#define PNH_R(r) case r: stockham_pass<T, r>(n, LB, ns, ld, tws, src, dst); break;
      PNH_R(2) PNH_R(3) PNH_R(4) PNH_R(5) PNH_R(6) PNH_R(7) PNH_R(8) PNH_R(9) PNH_R(10)
      PNH_R(11) PNH_R(12) PNH_R(13) PNH_R(14) PNH_R(15)
      default: stockham_pass<T, 16>(n, LB, ns, ld, tws, src, dst); break;
#undef PNH_R
    }
    ns *= R;
    C* tmp = src; src = dst; dst = tmp;
  }
  __syncthreads();
  const T scale = (T)d.scale, scale_im = scale * cj;
  const int kept = LB * d.n_out;
  const float r_o = 1.0f / (float)d.n_out;
#pragma unroll 4
  for (int i = tid; i < kept; i += nthr) {
    int l, t;
    if (fast) t = fdivmod(i, LB, r_lb, l);
    else l = fdivmod(i, d.n_out, r_o, t);
    if (l >= nl) continue;
    const Line li = line(l);
    C v = src[l * ld + t + (t >> 4)];
    if (d.sn_side == 2) {
      const T s = ((const T*)d.sn)[li.sn + (int64_t)t * d.sn_t_stride];
      v.x *= s; v.y *= s;
    }
    if (d.mod && d.sign < 0) v = cmul_fma(v, ((const C*)d.mod)[t]);
    out[li.dst + (int64_t)t * d.dst.t_stride] = mk<T>(v.x * scale, v.y * scale_im);
  }
}

template <typename T>
__global__ void __launch_bounds__(256)
fft_lines_kernel(FftDesc d, const void* in_, void* out_,
                 const void* __restrict__ tw_, const int* __restrict__ skip) {
  if (skip && *skip) return;
  extern __shared__ unsigned char smem_raw[];
  fft_body<T>(d, in_, out_, tw_, xcd_unit(blockIdx.x, gridDim.x), smem_raw);
}

template <typename T>
int launch_lines(const FftDesc& d, const void* in, void* out, const void* tw, const int* skip,
                 hipStream_t stream) {
  auto kern = fft_lines_kernel<T>;
  pnh_fft_allow_lds((const void*)kern, d.lds);
  hipLaunchKernelGGL(kern, dim3((unsigned)d.n_blocks), dim3(d.threads), d.lds, stream, d, in, out,
                     tw, skip);
  PNH_LAUNCH_CHECK();
  return 0;
}

}  // namespace

#define PNH_CT_DECL(p) \
  int pnh_fft_ct_part##p(const FftDesc&, int, const void*, void*, const void*, const int*, \
                         hipStream_t);
PNH_CT_DECL(0) PNH_CT_DECL(1) PNH_CT_DECL(2) PNH_CT_DECL(3) PNH_CT_DECL(4) PNH_CT_DECL(5)
PNH_CT_DECL(6)
#undef PNH_CT_DECL

bool pnh_fft_has_ct(int n) {
  return n >= PNH_CT_MIN && n <= PNH_CT_MAX && n % 2 == 0 && radices_of(n).r[0] > 0;
}

int pnh_fft_launch(const FftDesc& d, int fp64, const void* in, void* out,
                   const void* tw, const int* skip, hipStream_t stream) {
  if (d.n_outer * d.n_inner <= 0) return 0;
  if (d.ct) {
    switch ((d.n - PNH_CT_MIN) / 2 % PNH_CT_PARTS) {
      case 0: return pnh_fft_ct_part0(d, fp64, in, out, tw, skip, stream);
      case 1: return pnh_fft_ct_part1(d, fp64, in, out, tw, skip, stream);
      case 2: return pnh_fft_ct_part2(d, fp64, in, out, tw, skip, stream);
      case 3: return pnh_fft_ct_part3(d, fp64, in, out, tw, skip, stream);
      case 4: return pnh_fft_ct_part4(d, fp64, in, out, tw, skip, stream);
      case 5: return pnh_fft_ct_part5(d, fp64, in, out, tw, skip, stream);
      default: return pnh_fft_ct_part6(d, fp64, in, out, tw, skip, stream);
    }
  }
  return fp64 ? launch_lines<double>(d, in, out, tw, skip, stream)
              : launch_lines<float>(d, in, out, tw, skip, stream);
}

void pnh_fft_magic(uint32_t d, uint32_t* mul, int* shift) {
  int L = 0;
  while (L < 32 && (1ULL << L) < d) ++L;        // ceil(log2 d)
  if ((1ULL << L) == d) { *mul = 0; *shift = L; return; }
  *mul = (uint32_t)((((1ULL << L) - d) << 32) / d + 1);
  *shift = L - 1;
}

int pnh_fft_first_pass(int n) { return n / radices_of(n).r[0]; }

int pnh_fft_threads(const FftDesc& d) {
  if (!d.ct) return 256;
  const Radices rs = radices_of(d.n);
  const int rl = rs.r[2] > 1 ? rs.r[2] : rs.r[1];
  // one butterfly per thread in the first pass; in the others one per thread
  // up to 256 threads, or 512 where the workgroups are too few to fill the
  // chip (390 x 462 per transform 9.4 us at 256, 8.9 at 512; 256^3 66.5 at
  // 256, 70.7 at 512)
  const int first = d.n / rs.r[0] << d.lg_lines, most = d.n / rl << d.lg_lines;
  const int cap = d.n_blocks < 512 ? 512 : 256;
  const int want = first > cap ? first : (most < cap ? most : cap);
  return (want + 63) / 64 * 64;
}

size_t pnh_fft_lds_bytes(const FftDesc& d, int fp64) {
  const size_t esz = fp64 ? 16 : 8;
  const int nbuf = d.ct && radices_of(d.n).r[2] == 1 ? 1 : 2;
  return ((size_t)nbuf * d.lines_per_block * pnh_fft_lds_stride(d.n) + d.n) * esz;
}

// Dynamic LDS above 64 KB must be allowed per kernel before the launch.
void pnh_fft_allow_lds(const void* kernel, size_t bytes) {
  if (bytes > 65536)
    (void)hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

// Radices of n (each 2 to 16): the fewest passes, then the smallest sum of
// radices (the least work and the most threads per line), in falling order.
// n <= 4096 in every accepted plan, so three passes usually do.
static void best_radices(int m, int max_r, int left, int* cur, int depth, int sum, int* best,
                         int* best_np, int* best_sum) {
  if (m == 1) {
    if (depth < *best_np || (depth == *best_np && sum < *best_sum)) {
      *best_np = depth;
      *best_sum = sum;
      for (int i = 0; i < depth; ++i) best[i] = cur[i];
    }
    return;
  }
  if (depth >= left || depth >= *best_np) return;
  for (int r = max_r; r >= 2; --r)
    if (m % r == 0) {
      cur[depth] = r;
      best_radices(m / r, r, left, cur, depth + 1, sum + r, best, best_np, best_sum);
    }
}

int pnh_fft_factor(int n, uint64_t* radices, int* npass) {
  int m = n;
  const int primes[6] = {2, 3, 5, 7, 11, 13};
  for (int q = 0; q < 6; ++q)
    while (m % primes[q] == 0 && m > 1) m /= primes[q];
  if (m != 1) {
    pnh_set_error("FFT length %d has a prime factor other than 2, 3, 5, 7, 11, 13", n);
    return -1;
  }
  int cur[PNH_FFT_MAX_PASS], best[PNH_FFT_MAX_PASS];
  int np = PNH_FFT_MAX_PASS + 1, sum = 0;
  best_radices(n, 16, PNH_FFT_MAX_PASS, cur, 0, 0, best, &np, &sum);
  if (np > PNH_FFT_MAX_PASS) {
    pnh_set_error("FFT length %d needs too many passes", n);
    return -1;
  }
  *radices = 0;
  for (int p = 0; p < np; ++p) *radices |= (uint64_t)(best[p] - 1) << (4 * p);
  *npass = np;
  return 0;
}

// ------------------------------------------------------------- batches ----
#include "batch.h"

namespace {

template <typename T>
__global__ void __launch_bounds__(256)
fft_batch_kernel(const BatchProblem* __restrict__ probs, BatchTable t, int axis, int kind,
                 const void* in_, int in_image, void* out_, int out_image,
                 const int* __restrict__ done, const int* __restrict__ all_done) {
  typedef typename cplx<T>::t C;
  if (all_done && *all_done) return;
  const int p = t.tab[blockIdx.x];
  if (done && done[p]) return;
  const int64_t lb = (int64_t)blockIdx.x - t.first[p];
  extern __shared__ unsigned char smem_raw[];
  const BatchProblem& pr = probs[p];
  // a reference into the problem table (uniform loads); a by-value copy
  // selected at run time went to per-thread scratch memory
  const FftDesc& d = kind == BFFT_FWD ? pr.fwd[axis]
                                      : (kind == BFFT_INV ? pr.inv[axis] : pr.inv64[axis]);
  const void* tw = kind == BFFT_INV64 ? pr.tw64[axis] : pr.tw32[axis];
  const C* in = (const C*)in_ + (in_image ? pr.x_off : pr.k_off);
  C* out = (C*)out_ + (out_image ? pr.x_off : pr.k_off);
  fft_body<T>(d, in, out, tw, lb, smem_raw);
}

}  // namespace

int pnh_batch_fft_launch(const BatchProblem* probs, const BatchTable& t, int axis,
                         int kind, int fp64, size_t lds, int threads,
                         const void* in, int in_image, void* out, int out_image,
                         const int* done, const int* all_done, hipStream_t s) {
  if (t.n_blocks == 0) return 0;
  auto go = [&](auto kern) {
    pnh_fft_allow_lds((const void*)kern, lds);
    hipLaunchKernelGGL(kern, dim3((unsigned)t.n_blocks), dim3(threads), lds, s, probs, t, axis,
                       kind, in, in_image, out, out_image, done, all_done);
    PNH_LAUNCH_CHECK();
    return 0;
  };
  return fp64 ? go(fft_batch_kernel<double>) : go(fft_batch_kernel<float>);
}
