// Compile-time parts of the line FFT (gfx950): DFT butterflies in registers
// and the kernel of a transform length known at compile time.
//
// What bounds it: large grids move at HBM rate (128^3 -> 256^3: 352 MB in 67
// us), small ones wait (a pass over a 512^2 grid holds 3 MB; its time is the
// chain load - pass - exchange - pass - exchange - pass - store).  So every
// index is compile-time, the radices are the smallest three (most threads,
// fewest registers), all of a line's loads and the twiddle table's are issued
// before the first wait, and later passes take their twiddles from LDS.  Per
// forward transform (one launch per axis), replayed from a graph, against the
// run-time schedule of radices 16, 8, 4, 2, 3, 5, 7, 11, 13 it replaced: 64^2
// -> 128^2 10.9 -> 6.2 us, 256^2 -> 512^2 15.0 -> 8.7, 195 x 231 -> 390 x 462
// 27.2 -> 8.9, 60 x 75 x 54 -> 120 x 150 x 108 42.4 -> 21.4, 8 coils of 256^2
// 32.8 -> 17.5, 128^3 -> 256^3 75.2 -> 66.5.
#pragma once
#include <type_traits>

#include "common.h"
#include "fft.h"

namespace {

// cos and sin of 2 pi e / R at compile time: reduced to |x| <= pi / 4 by
// quadrants, then Taylor series (below half an ulp of FP64 there).
template <int R>
struct Roots {
  double c[R], s[R];
  constexpr Roots() : c(), s() {
    for (int e = 0; e < R; ++e) {
      const int q = (4 * e + R / 2) / R;               // nearest quadrant
      const double x = 1.57079632679489661923 * (double)(4 * e - q * R) / (double)R;
      double ts = x, tc = 1.0, ss = x, sc = 1.0;
      for (int k = 1; k < 12; ++k) {
        tc *= -x * x / (double)((2 * k - 1) * (2 * k));
        ts *= -x * x / (double)((2 * k) * (2 * k + 1));
        sc += tc;
        ss += ts;
      }
      c[e] = q % 4 == 0 ? sc : (q % 4 == 1 ? -ss : (q % 4 == 2 ? -sc : ss));
      s[e] = q % 4 == 0 ? ss : (q % 4 == 1 ? sc : (q % 4 == 2 ? -ss : -sc));
    }
  }
};
template <int R>
constexpr Roots<R> kRoots = Roots<R>();

template <typename C>
__device__ __forceinline__ C cmul_fma(C a, C b) {
  C z;
  z.x = __builtin_fma(a.x, b.x, -(a.y * b.y));
  z.y = __builtin_fma(a.x, b.y, a.y * b.x);
  return z;
}
template <>
__device__ __forceinline__ float2 cmul_fma(float2 a, float2 b) {
  return make_float2(__builtin_fmaf(a.x, b.x, -(a.y * b.y)),
                     __builtin_fmaf(a.x, b.y, a.y * b.x));
}

template <typename C>
__device__ __forceinline__ C mul_neg_i(C a) {
  C z; z.x = a.y; z.y = -a.x; return z;
}

// Forward DFT of R points in registers, in place.
template <typename T, int R>
struct Dft {
  typedef typename cplx<T>::t C;
  // R = A B: DFTs of A points over x[B n1 + n2], twiddles W_R^(n2 k1), DFTs
  // of B points, output k1 + A k2
  static constexpr int A = R % 4 == 0 ? 4 : (R % 2 == 0 ? 2 : (R % 3 == 0 ? 3 : 5));
  static constexpr int B = R / A;
  static __device__ __forceinline__ void run(C* v) {
    C a[B][A];
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) {
#pragma unroll
      for (int n1 = 0; n1 < A; ++n1) a[n2][n1] = v[B * n1 + n2];
      Dft<T, A>::run(a[n2]);
#pragma unroll
      for (int k1 = 1; k1 < A; ++k1)
        if (n2 > 0) {
          const int e = (n2 * k1) % R;
          a[n2][k1] = cmul_fma(a[n2][k1], mk<T>((T)kRoots<R>.c[e], (T)-kRoots<R>.s[e]));
        }
    }
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) {
      C t[B];
#pragma unroll
      for (int n2 = 0; n2 < B; ++n2) t[n2] = a[n2][k1];
      Dft<T, B>::run(t);
#pragma unroll
      for (int k2 = 0; k2 < B; ++k2) v[k1 + A * k2] = t[k2];
    }
  }
};

template <typename T>
struct Dft<T, 1> {
  typedef typename cplx<T>::t C;
  static __device__ __forceinline__ void run(C*) {}
};

template <typename T>
struct Dft<T, 2> {
  typedef typename cplx<T>::t C;
  static __device__ __forceinline__ void run(C* v) {
    const C a = v[0], b = v[1];
    v[0] = cadd(a, b); v[1] = csub(a, b);
  }
};

template <typename T>
struct Dft<T, 4> {
  typedef typename cplx<T>::t C;
  static __device__ __forceinline__ void run(C* v) {
    const C t0 = cadd(v[0], v[2]), t1 = csub(v[0], v[2]);
    const C t2 = cadd(v[1], v[3]), t3 = mul_neg_i(csub(v[1], v[3]));
    v[0] = cadd(t0, t2);
    v[2] = csub(t0, t2);
    v[1] = cadd(t1, t3);
    v[3] = csub(t1, t3);
  }
};

template <typename T>
struct Dft<T, 8> {
  typedef typename cplx<T>::t C;
  static __device__ __forceinline__ void run(C* v) {
    const T h = (T)0.70710678118654752440;
    C e[4] = {v[0], v[2], v[4], v[6]};
    C o[4] = {v[1], v[3], v[5], v[7]};
    Dft<T, 4>::run(e);
    Dft<T, 4>::run(o);
    // w8^q = exp(-2 pi i q / 8): (1 - i) h, -i, (-1 - i) h
    const C o1 = mk<T>((o[1].x + o[1].y) * h, (o[1].y - o[1].x) * h);
    const C o2 = mul_neg_i(o[2]);
    const C o3 = mk<T>((o[3].y - o[3].x) * h, -(o[3].x + o[3].y) * h);
    v[0] = cadd(e[0], o[0]); v[4] = csub(e[0], o[0]);
    v[1] = cadd(e[1], o1);   v[5] = csub(e[1], o1);
    v[2] = cadd(e[2], o2);   v[6] = csub(e[2], o2);
    v[3] = cadd(e[3], o3);   v[7] = csub(e[3], o3);
  }
};

// Odd prime R: with a_q = x_q + x_(R-q), b_q = x_q - x_(R-q),
// X_k, X_(R-k) = x_0 + sum_q cos(2 pi q k / R) a_q -+ i sum_q sin(..) b_q.
template <typename T, int R>
struct DftPrime {
  typedef typename cplx<T>::t C;
  static __device__ __forceinline__ void run(C* v) {
    constexpr int H = (R - 1) / 2;
    C a[H], b[H];
    C s = v[0];
#pragma unroll
    for (int q = 1; q <= H; ++q) {
      a[q - 1] = cadd(v[q], v[R - q]);
      b[q - 1] = csub(v[q], v[R - q]);
      s = cadd(s, a[q - 1]);
    }
    const C v0 = v[0];
    v[0] = s;
#pragma unroll
    for (int k = 1; k <= H; ++k) {
      T mx = v0.x, my = v0.y, nx = (T)0, ny = (T)0;
#pragma unroll
      for (int q = 1; q <= H; ++q) {
        const T c = (T)kRoots<R>.c[(q * k) % R], sn = (T)kRoots<R>.s[(q * k) % R];
        mx = fma(c, a[q - 1].x, mx);
        my = fma(c, a[q - 1].y, my);
        nx = fma(sn, b[q - 1].x, nx);
        ny = fma(sn, b[q - 1].y, ny);
      }
      v[k] = mk<T>(mx + ny, my - nx);
      v[R - k] = mk<T>(mx - ny, my + nx);
    }
  }
};
template <typename T> struct Dft<T, 3> : DftPrime<T, 3> {};
template <typename T> struct Dft<T, 5> : DftPrime<T, 5> {};
template <typename T> struct Dft<T, 7> : DftPrime<T, 7> {};
template <typename T> struct Dft<T, 11> : DftPrime<T, 11> {};
template <typename T> struct Dft<T, 13> : DftPrime<T, 13> {};

// Radix schedule of a compile-time length, R[0] >= R[1] >= R[2]: three
// radices of the smallest sum (the most threads per line and the fewest
// registers: 128 as 8 4 4 ran 8.0 us per 128^2 -> 256^2 transform in place of
// 11.3 as 16 8), R[0] <= 16, R[1], R[2] <= 10; R[0] = 0 when there is none.
struct Radices { int r[3]; };
constexpr Radices radices_of(int n) {
  Radices best = {{0, 0, 0}};
  int sum = 1 << 30;
  for (int a = 2; a <= 16; ++a)
    for (int b = 2; b <= a && b <= 10; ++b) {
      if (n % (a * b)) continue;
      const int c = n / (a * b);
      if (c < 1 || c > b) continue;
      if (a + b + c < sum) {
        sum = a + b + c;
        best.r[0] = a; best.r[1] = b; best.r[2] = c;
      }
    }
  return best;
}

// q = n / d for n < 2^32 by a host-made multiplier: (n * mul) >> 32 >> shift,
// mul = 0 for powers of two (shift only).
__device__ __forceinline__ uint32_t div_magic(uint32_t n, uint32_t mul, int shift) {
  if (mul == 0) return n >> shift;
  const uint32_t t = __umulhi(n, mul);
  return (((n - t) >> 1) + t) >> shift;
}

// One line transform of compile-time length N.  A workgroup takes 2^lg lines
// (FAST: consecutive inner lines of one outer line, consecutive threads on
// consecutive lines; else consecutive lines, consecutive threads along the
// line).  The first pass takes one butterfly per thread at most, so all of a
// line's loads and the twiddle loads are in flight together.  in_ and out_ may alias (in-place passes): a
// workgroup reads all its lines before its first store, and other workgroups
// own other lines.
template <typename T, int N, bool FAST>
__device__ __forceinline__ void fft_ct_body(const FftDesc& d, const void* in_, void* out_,
                                            const void* __restrict__ tw_, uint32_t blk,
                                            unsigned char* smem_raw) {
  typedef typename cplx<T>::t C;
  constexpr Radices RS = radices_of(N);
  constexpr int R0 = RS.r[0], R1 = RS.r[1], R2 = RS.r[2];
  constexpr int NB0 = N / R0, NB1 = N / R1, NB2 = N / R2;
  constexpr int LD = (N + (N >> 4) + 1) | 1;
  const C* in = (const C*)in_;
  C* out = (C*)out_;
  const C* __restrict__ tw = (const C*)tw_;
  const int lg = d.lg_lines, LB = 1 << lg;
  C* tws = reinterpret_cast<C*>(smem_raw);
  C* buf0 = tws + N;
  C* buf1 = buf0 + LB * LD;
  const int tid = threadIdx.x, nthr = blockDim.x;

  // twiddle table: loaded first, stored to LDS behind the first pass's loads
  constexpr int KT = 4;
  C t[KT];
#pragma unroll
  for (int q = 0; q < KT; ++q) t[q] = tw[min(tid + q * nthr, N - 1)];

  int64_t src0 = 0, dst0 = 0, sn0 = 0;     // FAST: of the workgroup's first line
  uint32_t line0 = 0;
  int nl;
  if (FAST) {
    const uint32_t o = div_magic(blk, d.mul_blocks, d.sh_blocks);
    const uint32_t b0 = (blk - o * d.blocks_inner) << lg;
    const uint32_t o0 = div_magic(o, d.mul_split, d.sh_split);
    const uint32_t o1 = o - o0 * (uint32_t)d.o_split;
    src0 = o0 * d.src.o_stride[0] + o1 * d.src.o_stride[1] + b0;
    dst0 = o0 * d.dst.o_stride[0] + o1 * d.dst.o_stride[1] + b0;
    sn0 = o0 * d.sn_o_stride[0] + o1 * d.sn_o_stride[1];
    nl = (int)min(d.n_inner - (int64_t)b0, (int64_t)LB);
  } else {
    line0 = blk << lg;
    nl = (int)min(d.n_outer * d.n_inner - (int64_t)line0, (int64_t)LB);
  }
  struct Line { int64_t src, dst, sn; };
  auto line = [&](int l) -> Line {
    if (FAST) return Line{src0 + l, dst0 + l, sn0};
    const uint32_t L = line0 + l;
    const uint32_t o = div_magic(L, d.mul_inner, d.sh_inner);
    const uint32_t b = L - o * (uint32_t)d.n_inner;
    const uint32_t o0 = div_magic(o, d.mul_split, d.sh_split);
    const uint32_t o1 = o - o0 * (uint32_t)d.o_split;
    return Line{o0 * d.src.o_stride[0] + o1 * d.src.o_stride[1] + b,
                o0 * d.dst.o_stride[0] + o1 * d.dst.o_stride[1] + b,
                o0 * d.sn_o_stride[0] + o1 * d.sn_o_stride[1]};
  };
  const T cj = d.sign > 0 ? (T)-1 : (T)1;  // inverse: conjugate in and out

  // first pass: global -> buf0
  {
    int l, j;
    if (FAST) { l = tid & (LB - 1); j = tid >> lg; }
    else { l = tid / NB0; j = tid - l * NB0; }
    const bool act = l < nl && j < NB0;
    const Line li = line(act ? l : 0);
    const int64_t st = d.src.t_stride;
    const C* p = in + li.src + (int64_t)(act ? j : 0) * st;
    const int64_t inc = (int64_t)NB0 * st;
    C v[R0];
    // straight-line loads (a conditional one would wait for itself): points
    // past n_in read the buffer's first element and count as zero
    auto load = [&](auto cnt) {
      constexpr int L = decltype(cnt)::value;
      T s[L];
#pragma unroll
      for (int r = 0; r < L; ++r) v[r] = *(act && j + r * NB0 < d.n_in ? p + r * inc : in);
      if (d.mod && d.sign > 0) {
        const C* mod = (const C*)d.mod;
        C m[L];
#pragma unroll
        for (int r = 0; r < L; ++r) m[r] = mod[min(j + r * NB0, N - 1)];
#pragma unroll
        for (int r = 0; r < L; ++r) { m[r].y = -m[r].y; v[r] = cmul_fma(v[r], m[r]); }
      }
      if (d.sn_side == 1) {
        const T* sn = (const T*)d.sn;
        const int64_t s0 = li.sn + (int64_t)(act ? j : 0) * d.sn_t_stride;
        const int64_t sinc = (int64_t)NB0 * d.sn_t_stride;
#pragma unroll
        for (int r = 0; r < L; ++r) s[r] = sn[j + r * NB0 < d.n_in ? s0 + r * sinc : 0];
      } else {
#pragma unroll
        for (int r = 0; r < L; ++r) s[r] = (T)1;
      }
#pragma unroll
      for (int r = 0; r < R0; ++r) {
        const bool ok = r < L && j + r * NB0 < d.n_in;
        v[r] = mk<T>(ok ? v[r < L ? r : 0].x * s[r < L ? r : 0] : (T)0,
                     ok ? v[r < L ? r : 0].y * s[r < L ? r : 0] : (T)0);
      }
    };
    // zero padding to twice the length leaves the upper half of the points
    constexpr int HALF = (R0 + 1) / 2;
    if (d.n_in <= HALF * NB0) load(std::integral_constant<int, HALF>());
    else load(std::integral_constant<int, R0>());
#pragma unroll
    for (int q = 0; q < KT; ++q)
      if (tid + q * nthr < N) tws[tid + q * nthr] = t[q];
    for (int i = tid + KT * nthr; i < N; i += nthr) tws[i] = tw[i];
    if (l < LB && j < NB0) {
#pragma unroll
      for (int r = 0; r < R0; ++r) v[r].y *= cj;
      Dft<T, R0>::run(v);
#pragma unroll
      for (int r = 0; r < R0; ++r) {
        const int o = j * R0 + r;
        buf0[l * LD + o + (o >> 4)] = v[r];
      }
    }
  }
  __syncthreads();
  // second pass: buf0 -> buf1 (or global when it is the last)
  auto middle = [&](int l, int j, C* v) {
    constexpr int NS = R0, TS = N / (NS * R1);
    const int k = j % NS;
#pragma unroll
    for (int r = 0; r < R1; ++r) {
      const int o = j + r * NB1;
      v[r] = buf0[l * LD + o + (o >> 4)];
    }
#pragma unroll
    for (int r = 1; r < R1; ++r) v[r] = cmul_fma(v[r], tws[r * k * TS]);
    Dft<T, R1>::run(v);
    return (j / NS) * (NS * R1) + k;
  };
  const T scale = (T)d.scale, scale_im = scale * cj;
  auto put = [&](int l, int o, int step, auto& v) {
    constexpr int R = sizeof(v) / sizeof(C);
    const Line li = line(l);
    const int64_t dt = d.dst.t_stride;
    C* p = out + li.dst + (int64_t)o * dt;
    const int64_t inc = (int64_t)step * dt;
    if (d.sn_side == 2) {
      const T* sn = (const T*)d.sn + li.sn;
      T s[R];
#pragma unroll
      for (int r = 0; r < R; ++r)
        s[r] = sn[(int64_t)(o + r * step < d.n_out ? o + r * step : 0) * d.sn_t_stride];
#pragma unroll
      for (int r = 0; r < R; ++r) { v[r].x *= s[r]; v[r].y *= s[r]; }
    }
    if (d.mod && d.sign < 0) {
      const C* mod = (const C*)d.mod;
      C m[R];
#pragma unroll
      for (int r = 0; r < R; ++r) m[r] = mod[o + r * step];
#pragma unroll
      for (int r = 0; r < R; ++r) v[r] = cmul_fma(v[r], m[r]);
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (o + r * step < d.n_out) p[r * inc] = mk<T>(v[r].x * scale, v[r].y * scale_im);
  };
  if constexpr (R2 == 1) {
    for (int idx = tid; idx < NB1 << lg; idx += nthr) {
      int l, j;
      if (FAST) { l = idx & (LB - 1); j = idx >> lg; }
      else { l = idx / NB1; j = idx - l * NB1; }
      C v[R1];
      const int o = middle(l, j, v);
      if (l < nl) put(l, o, R0, v);
    }
  } else {
    for (int idx = tid; idx < NB1 << lg; idx += nthr) {
      const int l = idx / NB1, j = idx - l * NB1;
      C v[R1];
      const int o = middle(l, j, v);
#pragma unroll
      for (int r = 0; r < R1; ++r) {
        const int q = o + r * R0;
        buf1[l * LD + q + (q >> 4)] = v[r];
      }
    }
    __syncthreads();
    for (int idx = tid; idx < NB2 << lg; idx += nthr) {
      constexpr int NS = R0 * R1;          // N / (NS R2) = 1
      int l, j;
      if (FAST) { l = idx & (LB - 1); j = idx >> lg; }
      else { l = idx / NB2; j = idx - l * NB2; }
      C v[R2];
#pragma unroll
      for (int r = 0; r < R2; ++r) {
        const int o = j + r * NB2;
        v[r] = buf1[l * LD + o + (o >> 4)];
      }
#pragma unroll
      for (int r = 1; r < R2; ++r) v[r] = cmul_fma(v[r], tws[r * j]);
      Dft<T, R2>::run(v);
      if (l < nl) put(l, j, NS, v);
    }
  }
}

// Block of a launch of nblk -> work unit, so that the units of one XCD
// (workgroups b, b + 8, ... share one and its L2) are neighbours: along a
// strided axis neighbouring line groups share 128-byte lines.
__device__ __forceinline__ uint32_t xcd_unit(uint32_t b, uint32_t nblk) {
  const uint32_t x = b & 7, per = nblk >> 3, rem = nblk & 7;
  return x * per + (x < rem ? x : rem) + (b >> 3);
}

}  // namespace
