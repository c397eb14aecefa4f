// Interpolation (k2y), gridding (y2k) and P^H P with real factors (real.h),
// compiled once per dimension (PNH_D) and
// precision (PNH_F64).
//
// The work list is the gridding's (tile ownership): a row belongs to the tile
// that holds its first support cell, a work item is a run of rows of one
// tile, and the item's padded box (tile + J - 1 cells on an axis cut into
// tiles, the whole axis otherwise) holds every support cell of its rows.
//
// k2y copies the box into LDS and gathers every row from it.  y2k grids every
// row into an LDS accumulator of the box with exact 64-bit fixed-point integer
// atomics (order-independent, hence bit-reproducible), writes it to the item's
// partial slot, and a gather sums the slots that cover each grid cell in a
// fixed order.  P^H P does both for one item: the samples stay in registers.
//
// A row's support is walked by S lanes, each taking every S-th cell of the
// last axis (dispatch() chooses).
#include <stddef.h>

#include <type_traits>

#include "batch.h"
#include "common.h"
#include "fixed.h"
#include "interp.h"
#include "real.h"
#include "reduce.h"

#if !defined(PNH_D) || !defined(PNH_F64)
#error "compile with PNH_D = 1, 2 or 3 and PNH_F64 = 0 (complex64) or 1 (complex128)"
#endif

namespace {

constexpr int kMaxCl = 8;                // coils of one pass at most

template <typename C>
__device__ __forceinline__ C conj_mul(C a, C b) {        // a conj(b)
  C z;
  z.x = fma(a.x, b.x, a.y * b.y);
  z.y = fma(a.y, b.x, -(a.x * b.y));
  return z;
}
template <typename C>
__device__ __forceinline__ C cmul_f(C a, C b) {
  C z;
  z.x = fma(a.x, b.x, -(a.y * b.y));
  z.y = fma(a.x, b.y, a.y * b.x);
  return z;
}

// A value from LDS.  Complex64 is read as one 64-bit word that the compiler
// leaves alone: pairs fused into ds_read2_b64 take longer than the two reads
// (3-D 256^3 interpolation, 2 097 152 samples: LDS busy for 72.8M cycles
// fused, 47.8M so, half of them bank conflicts).
__device__ __forceinline__ float2 lds_get(const float2* p) {
  typedef const volatile __attribute__((address_space(3))) unsigned long long* At;
  const unsigned long long w = *(At)p;
  return make_float2(__uint_as_float((unsigned)w), __uint_as_float((unsigned)(w >> 32)));
}
__device__ __forceinline__ double2 lds_get(const double2* p) { return *p; }

// q = i / n, r = i % n for 0 <= i < 2^22, rcp = 1.0f / n
__device__ __forceinline__ int fdiv(int i, int n, float rcp, int& r) {
  int q = (int)((float)i * rcp);
  r = i - q * n;
  if (r < 0) { --q; r += n; }
  else if (r >= n) { ++q; r -= n; }
  return q;
}

// Origin of the tile.
template <int D>
struct Frame {
  int T0[3];
  __device__ __forceinline__ Frame(const RealArgs& a, int tile) {
#pragma unroll
    for (int d = D - 1; d >= 0; --d) {
      const int tg = a.tgrid[d];
      const int q = tile / tg;
      T0[d] = (tile - q * tg) * a.tile[d];
      tile = q;
    }
  }
};

// The factors and box cells of one row and coil (for lane `sub` of its S
// lanes).  JM bounds the leading axes' support, JL the last axis's; EX: they
// are exactly that.  PAD, how the support's cells lie in the box:
//   > 0: every axis is cut into tiles, boxes of that extent, one coil: the
//        offsets from the first cell are compile-time;
//   -1:  every axis is cut into tiles: the offsets are uniform;
//   0:   an axis spanned by one tile wraps inside the box (the factor takes
//        mod's sign there): an index per support cell and axis.
template <typename T, int D, int JM, int JL, bool EX, int CP, int PAD>
struct Row {
  static constexpr int S = (JL + CP - 1) / CP;
  static constexpr bool WR = PAD == 0;
  // the last axis's support is exactly JL (4 and 16 also take smaller ones)
  static constexpr bool LX = EX || (JL >= 5 && JL <= 8);
  T c0[D > 1 ? JM : 1], c1[D > 2 ? JM : 1], cl[CP];
  int o0[WR && D > 1 ? JM : 1], o1[WR && D > 2 ? JM : 1], ol[WR || !LX ? CP : 1];
  int lin;

  __device__ __forceinline__ static int tail(const RealArgs& a) {
    if (EX) return (D - 1) * JM + JL;
    int t = a.J[0];
    if (D > 1) t += a.J[1];
    if (D > 2) t += a.J[2];
    return t;
  }

  __device__ __forceinline__ void load(const RealArgs& a, int r, int sub, int clc, int c) {
    const T* __restrict__ p =
        (const T*)__builtin_assume_aligned((const T*)a.rec + (int64_t)r * a.rw, 16);
    const int J0 = EX ? JM : a.J[0], J1 = EX ? JM : a.J[1];
    const int JR = LX ? JL : a.J[D - 1];
    const int b1 = J0, bl = D == 1 ? 0 : (D == 2 ? J0 : J0 + J1);
    if (D > 1) {
#pragma unroll
      for (int j = 0; j < JM; ++j) c0[j] = p[EX ? j : min(j, J0 - 1)];
    }
    if (D > 2) {
#pragma unroll
      for (int j = 0; j < JM; ++j) c1[j] = p[b1 + (EX ? j : min(j, J1 - 1))];
    }
    static_assert(JL % S == 0, "whole cells per lane");
    int jl[CP];
#pragma unroll
    for (int i = 0; i < CP; ++i) {
      jl[i] = LX ? sub + S * i : min(sub + S * i, JR - 1);
      cl[i] = p[bl + jl[i]];
      if (!LX && sub + S * i >= JR) cl[i] = (T)0;
    }
    int x0, x1 = 0, x2 = 0;
    const int t = tail(a);
    if constexpr (sizeof(T) == 4) {
      const int w = __float_as_int(p[t + 2]);
      x0 = w & 0xffff;
      x1 = (unsigned)w >> 16;
      if (D > 2) x2 = __float_as_int(p[t + 3]);
    } else {
      const long long w = __double_as_longlong(p[t]);
      x0 = (int)(w & 0xffff);
      x1 = (int)(w >> 16 & 0xffff);
      x2 = (int)(w >> 32 & 0xffff);
    }
    if constexpr (!WR) {
      lin = x0;
      if (D > 1) lin = lin * (PAD > 0 ? PAD : a.pad[1]) + x1;
      if (D > 2) lin = lin * (PAD > 0 ? PAD : a.pad[2]) + x2;
      if (LX) lin += sub;
      if (PAD < 0) lin = lin * clc + c;
      if constexpr (!LX) {
#pragma unroll
        for (int i = 0; i < CP; ++i) ol[i] = jl[i] * clc;
      }
    } else {
      const int P1 = D > 1 ? a.pad[1] : 1, P2 = D > 2 ? a.pad[2] : 1;
      // box index of support offset j on an axis; mod's sign where it wraps
      auto at = [&](int d, int x, T& cf) {
        if (a.tgrid[d] == 1 && x >= a.K[d]) {
          x -= a.K[d];
          if (a.flip[d]) cf = -cf;
        }
        return x * clc;
      };
      if (D > 1) {
#pragma unroll
        for (int j = 0; j < JM; ++j) o0[j] = at(0, x0 + j, c0[j]) * P1 * P2;
      }
      if (D > 2) {
#pragma unroll
        for (int j = 0; j < JM; ++j) o1[j] = at(1, x1 + j, c1[j]) * P2;
      }
      const int xl = D == 1 ? x0 : (D == 2 ? x1 : x2);
#pragma unroll
      for (int i = 0; i < CP; ++i) ol[i] = at(D - 1, xl + jl[i], cl[i]) + c;
    }
  }
  // box element of leading offsets j0, j1 and the lane's i-th last-axis cell
  __device__ __forceinline__ int cell(const RealArgs& a, int clc, int j0, int j1, int i) const {
    if constexpr (WR) {
      int q = ol[i];
      if (D > 1) q += o0[j0];
      if (D > 2) q += o1[j1];
      return q;
    } else {
      const int n = PAD > 0 ? 1 : clc;
      const int s1 = D < 3 ? 0 : (PAD > 0 ? PAD : a.pad[2] * n);
      const int s0 = D == 1 ? 0 : (PAD > 0 ? (D == 2 ? PAD : PAD * PAD)
                                           : a.pad[1] * (D == 2 ? n : s1));
      const int last = LX ? S * i * n : ol[LX ? 0 : i];
      return lin + j0 * s0 + j1 * s1 + last;
    }
  }
  // sum over this lane's cells of coefficient times box value
  template <typename C>
  __device__ __forceinline__ C gather(const RealArgs& a, const C* __restrict__ box,
                                      int clc) const {
    const int J0 = EX ? JM : a.J[0], J1 = EX ? JM : a.J[1];
    auto get = [&](int j0, int j1, int i) -> C {
      return lds_get(box + cell(a, clc, j0, j1, i));
    };
    C acc = mk<T>((T)0, (T)0);
    // CP == 1 factors the last axis out of the sums
    auto last = [&](int j0, int j1) -> C {
      if (CP == 1) return get(j0, j1, 0);
      C s = mk<T>((T)0, (T)0);
#pragma unroll
      for (int i = 0; i < CP; ++i) {
        const C v = get(j0, j1, i);
        s.x = fma(cl[i], v.x, s.x);
        s.y = fma(cl[i], v.y, s.y);
      }
      return s;
    };
    if (D == 1) {
      acc = last(0, 0);
    } else if (D == 2) {
#pragma unroll
      for (int j0 = 0; j0 < JM; ++j0)
        if (EX || j0 < J0) {
          const C s = last(j0, 0);
          acc.x = fma(c0[j0], s.x, acc.x);
          acc.y = fma(c0[j0], s.y, acc.y);
        }
    } else {
#pragma unroll
      for (int j0 = 0; j0 < JM; ++j0)
        if (EX || j0 < J0) {
          C s0 = mk<T>((T)0, (T)0);
#pragma unroll
          for (int j1 = 0; j1 < JM; ++j1)
            if (EX || j1 < J1) {
              const C s = last(j0, j1);
              s0.x = fma(c1[j1], s.x, s0.x);
              s0.y = fma(c1[j1], s.y, s0.y);
            }
          acc.x = fma(c0[j0], s0.x, acc.x);
          acc.y = fma(c0[j0], s0.y, acc.y);
        }
    }
    if (CP == 1) { acc.x *= cl[0]; acc.y *= cl[0]; }
    return acc;
  }
  // adds coefficient times v (scaled for the accumulator) to this lane's
  // cells; the products are formed in FP64 and rounded once, onto the
  // fixed-point grid.  Complex64 operators pack a cell's real and imaginary
  // sums into one word, complex128 keeps two.
  __device__ __forceinline__ void grid(const RealArgs& a, long long* __restrict__ acc, int clc,
                                       double2 v) const {
    constexpr int CW = sizeof(T) == 4 ? 1 : 2;
    const int J0 = EX ? JM : a.J[0], J1 = EX ? JM : a.J[1];
    auto add = [&](int j0, int j1, int i, double f, double2 w) {
      long long* at = acc + cell(a, clc, j0, j1, i) * CW;
      const double re = __builtin_fma(f, w.x, kMagic), im = __builtin_fma(f, w.y, kMagic);
      if (CW == 1) {
        lds_add(at, pack_fixed(re, im));
      } else {
        lds_add(at, __double_as_longlong(re) - kMagicBits);
        lds_add(at + 1, __double_as_longlong(im) - kMagicBits);
      }
    };
    double d0[D > 1 ? JM : 1], d1[D > 2 ? JM : 1];
    if (D > 1) {
#pragma unroll
      for (int j = 0; j < JM; ++j) d0[j] = (double)c0[j];
    }
    if (D > 2) {
#pragma unroll
      for (int j = 0; j < JM; ++j) d1[j] = (double)c1[j];
    }
    const int JR = LX ? JL : a.J[D - 1];
#pragma unroll
    for (int i = 0; i < CP; ++i) {
      const double l = (double)cl[i];
      // a lane's cells past the support add nothing (their factor is zero)
      if (!LX && CP > 1 && S * i >= JR) continue;
      if (D == 1) {
        add(0, 0, i, l, v);
        continue;
      }
      const double2 w = make_double2(l * v.x, l * v.y);
      if (D == 2) {
#pragma unroll
        for (int j0 = 0; j0 < JM; ++j0)
          if (EX || j0 < J0) add(j0, 0, i, d0[j0], w);
        continue;
      }
#pragma unroll
      for (int j0 = 0; j0 < JM; ++j0)
        if (EX || j0 < J0) {
          const double2 w0 = make_double2(d0[j0] * w.x, d0[j0] * w.y);
#pragma unroll
          for (int j1 = 0; j1 < JM; ++j1)
            if (EX || j1 < J1) add(j0, j1, i, d1[j1], w0);
        }
    }
  }
};

// Sample index and phase of row r.
template <typename T>
__device__ __forceinline__ typename cplx<T>::t row_phase(const RealArgs& a, int tail, int r) {
  if constexpr (sizeof(T) == 4) {
    const float* p = (const float*)a.rec + (int64_t)r * a.rw + tail;
    return make_float2(p[0], p[1]);
  } else {
    return ((const double2*)a.ph)[r];
  }
}
template <typename T, int D>
__device__ __forceinline__ int row_sample(const RealArgs& a, int tail, int r) {
  if constexpr (sizeof(T) == 4)
    return __float_as_int(((const float*)a.rec)[(int64_t)r * a.rw + tail + (D == 3 ? 4 : 3)]);
  else
    return a.perm[r];
}

// The item's padded box of the grid -> LDS ([cell][coil]).  A thread keeps one
// place of the trailing axes and walks the leading one, so a cell costs a
// load, a store and an address step; U loads are in flight at once.  note(v)
// sees every value.
template <typename T, int D, bool STAGE, typename F>
__device__ __forceinline__ void load_box_t(const RealArgs& a, const Frame<D>& f, int clc,
                                           typename cplx<T>::t* __restrict__ box,
                                           const typename cplx<T>::t* __restrict__ grid,
                                           F&& note) {
  typedef typename cplx<T>::t C;
  constexpr int U = 4;
  const int tid = threadIdx.x, nthr = blockDim.x;
  const int P0 = a.pad[0], P1 = D > 1 ? a.pad[1] : 1, P2 = D > 2 ? a.pad[2] : 1;
  const int64_t s0 = (D == 1 ? 1 : (D == 2 ? (int64_t)a.K[1] : (int64_t)a.K[1] * a.K[2])) * a.nb;
  const int I = P1 * P2 * clc;                     // elements of a leading plane
  const int K0 = a.K[0], T0 = f.T0[0], flip0 = a.flip[0];
  auto column = [&](int i, int from, int by) {
    const int t = i / clc, c = i - t * clc;
    // grid place of the trailing coordinates; mod changes sign across the edge
    int neg = 0;
    int64_t gt = 0;
    C mt = mk<T>((T)1, (T)0);
    auto at = [&](int d, int x) {
      int g = f.T0[d] + x;
      if (g >= a.K[d]) { g -= a.K[d]; neg ^= a.flip[d]; }
      return g;
    };
    if (D == 2) {
      const int g1 = at(1, t);
      gt = g1;
      if (STAGE) mt = ((const C*)a.mod[1])[g1];
    }
    if (D == 3) {
      const int x1 = t / P2;
      const int g1 = at(1, x1), g2 = at(2, t - x1 * P2);
      gt = (int64_t)g1 * a.K[2] + g2;
      if (STAGE) mt = cmul_f(((const C*)a.mod[1])[g1], ((const C*)a.mod[2])[g2]);
    }
    const C* __restrict__ col = grid + gt * a.nb + a.c0 + c;
    for (int x0 = from; x0 < P0; x0 += U * by) {
      C v[U], m[U];
      int n[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        int g0 = T0 + min(x0 + u * by, P0 - 1);
        n[u] = neg;
        if (g0 >= K0) { g0 -= K0; n[u] ^= flip0; }
        v[u] = col[g0 * s0];
        if (STAGE) m[u] = ((const C*)a.mod[0])[g0];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (STAGE) v[u] = cmul_f(v[u], cmul_f(m[u], mt));
        const T sg = n[u] ? (T)-1 : (T)1;
        if (x0 + u * by < P0) box[(x0 + u * by) * I + i] = mk<T>(v[u].x * sg, v[u].y * sg);
        note(v[u]);
      }
    }
  };
  const int G = nthr / I;
  if (G > 0) {
    const int og = tid / I;
    if (og < G) column(tid - og * I, og, G);
  } else {
    for (int i = tid; i < I; i += nthr) column(i, 0, 1);
  }
}
template <typename T, int D, typename F>
__device__ __forceinline__ void load_box(const RealArgs& a, const Frame<D>& f, int clc,
                                         typename cplx<T>::t* __restrict__ box,
                                         const typename cplx<T>::t* __restrict__ grid, F&& note) {
  if (a.stage) load_box_t<T, D, true>(a, f, clc, box, grid, note);
  else load_box_t<T, D, false>(a, f, clc, box, grid, note);
}
template <typename T, int D>
__device__ __forceinline__ void load_box(const RealArgs& a, const Frame<D>& f, int clc,
                                         typename cplx<T>::t* __restrict__ box,
                                         const typename cplx<T>::t* __restrict__ grid) {
  load_box<T, D>(a, f, clc, box, grid, [](typename cplx<T>::t) {});
}

// Lane and row mapping of a workgroup: pair q = (row, coil) of the item goes
// to S neighbouring lanes, 64 / S pairs to a wave.
template <int S>
struct Lanes {
  int sub, sl, q0, step;
  bool on;
  __device__ __forceinline__ Lanes() {
    constexpr int RW = 64 / S;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    sl = lane / S;
    sub = lane - sl * S;
    on = sl < RW;
    q0 = wave * RW;
    step = (int)(blockDim.x >> 6) * RW;
  }
};

// Sum over a pair's S lanes; lane sub == 0 gets the total.
template <int S, typename C>
__device__ __forceinline__ C lanes_sum(C v, int sub) {
#pragma unroll
  for (int off = 1; off < S; off <<= 1) {
    const auto ox = __shfl_down(v.x, off, 64);
    const auto oy = __shfl_down(v.y, off, 64);
    if (sub + off < S) { v.x += ox; v.y += oy; }
  }
  return v;
}

template <typename T, int D, int JM, int JL, bool EX, int CP, int PAD>
__device__ __forceinline__ void k2y_body(const RealArgs& a, const int4 it, unsigned char* smem,
                                         const void* __restrict__ grid_,
                                         void* __restrict__ y_) {
  typedef typename cplx<T>::t C;
  typedef Row<T, D, JM, JL, EX, CP, PAD> R;
  constexpr int S = R::S;
  const int clc = PAD > 0 ? 1 : a.cl;
  const float rcl = 1.0f / (float)clc;
  C* box = reinterpret_cast<C*>(smem);
  C* __restrict__ y = (C*)y_;
  const Lanes<S> ln;
  const int nq = it.z * clc;
  const int tail = R::tail(a);
  R rd;
  int q = ln.q0 + ln.sl, c = 0;
  auto row_of = [&](int qq, int& cc) {
    if (PAD > 0) { cc = 0; return it.y + qq; }
    return it.y + fdiv(qq, clc, rcl, cc);
  };
  int r = 0;
  if (ln.on && q < nq) {
    r = row_of(q, c);
    rd.load(a, r, ln.sub, clc, c);
  }
  load_box<T, D>(a, Frame<D>(a, it.x), clc, box, (const C*)grid_);
  __syncthreads();
  for (int q0 = ln.q0; q0 < nq; q0 += ln.step) {
    const bool valid = ln.on && q < nq;
    C s = mk<T>((T)0, (T)0);
    if (valid) s = rd.gather(a, box, clc);
    s = lanes_sum<S>(s, ln.sub);
    if (valid && ln.sub == 0) {
      const int64_t m = row_sample<T, D>(a, tail, r);
      y[m * a.nb + a.c0 + c] = cmul_f(s, row_phase<T>(a, tail, r));
    }
    q += ln.step;
    if (ln.on && q < nq) {
      r = row_of(q, c);
      rd.load(a, r, ln.sub, clc, c);
    }
  }
}

// Fraction bits of the accumulators: complex128 50, complex64 31 (a cell's real
// and imaginary sums are the halves of one word).  2^31 is reached by no sum:
// the exponent leaves 2^-18 of it for the rounding of up to 4096 summands.
template <typename T>
constexpr int kBits = sizeof(T) == 4 ? 31 : kFixBits;

// Fixed-point exponent from a bound of the summands: 2^e above it.
__device__ __forceinline__ int fix_exponent(double ymax, double bound) {
  if (!(ymax <= 1.0e300)) return kPoisonExp;
  const double B = ymax * bound * (1.0 + 0x1p-18);
  int e = 0;
  if (B > 0.0) (void)frexp(B, &e);       // B < 2^e
  return e < -960 ? -960 : e;
}

// |Re| + |Im|, or infinity where it is not a finite number
template <typename C>
__device__ __forceinline__ double magnitude(C v) {
  const double s = fabs((double)v.x) + fabs((double)v.y);
  return s <= 1.0e300 ? s : __builtin_inf();
}

// Per-coil maximum over the workgroup of each thread's m (for its coil c);
// mx: kMaxCl words of LDS, red: 16.  Every thread calls it; a barrier on the
// way also orders what the workgroup wrote to LDS before.
__device__ __forceinline__ void coil_max(double m, int clc, double* red,
                                         unsigned long long* mx) {
  // one coil: over the waves; several went to mx by atomics already
  if (clc == 1) {
    m = block_max(m, red);
    if (threadIdx.x == 0) mx[0] = (unsigned long long)__double_as_longlong(m);
  }
  __syncthreads();
}

// Accumulator -> partial slot, scaled back; a non-finite sample poisons its
// coil's cells of the slot.
template <typename T>
__device__ __forceinline__ void flush_slot(const RealArgs& a, const int4 it, int clc,
                                           const long long* __restrict__ acc, const int* ex,
                                           void* __restrict__ part_) {
  typedef typename cplx<T>::t C;
  constexpr int FB = kBits<T>;
  const int plane = a.pad_cells * clc;
  C* __restrict__ part = (C*)part_ + (int64_t)it.w * plane;
  const float rcl = 1.0f / (float)clc;
  int e0 = ex[0];
  double un = ldexp(1.0, (e0 == kPoisonExp ? 0 : e0) - FB);
  const T nan = (T)__builtin_nan("");
  for (int i = threadIdx.x; i < plane; i += blockDim.x) {
    if (clc > 1) {
      int c;
      fdiv(i, clc, rcl, c);
      e0 = ex[c];
      un = ldexp(1.0, (e0 == kPoisonExp ? 0 : e0) - FB);
    }
    long long re, im;
    if (sizeof(T) == 4) {
      unpack_fixed(acc[i], re, im);
    } else {
      re = acc[2 * i];
      im = acc[2 * i + 1];
    }
    C v = mk<T>((T)((double)re * un), (T)((double)im * un));
    if (e0 == kPoisonExp) v = mk<T>(nan, nan);
    part[i] = v;
  }
}

// Scratch after an accumulator of `words` 64-bit words: wave maxima, coil
// maxima, coil exponents.
struct Scratch {
  double* red;
  unsigned long long* mx;
  int* ex;
  __device__ __forceinline__ explicit Scratch(unsigned char* p) {
    red = reinterpret_cast<double*>(p);
    mx = reinterpret_cast<unsigned long long*>(p + 128);
    ex = reinterpret_cast<int*>(p + 128 + 8 * kMaxCl);
  }
};
constexpr int kScratchBytes = 256;

// Gridding of one item.  item_e: the exponents made ahead ([item][coil]) with
// the samples in row order in ys, or null.
template <typename T, int D, int JM, int JL, bool EX, int CP, int PAD>
__device__ __forceinline__ void y2k_body(const RealArgs& a, const int4 it, int item,
                                         unsigned char* smem, const void* __restrict__ y_,
                                         void* __restrict__ part, const int* __restrict__ item_e,
                                         const void* __restrict__ ys_) {
  typedef typename cplx<T>::t C;
  typedef Row<T, D, JM, JL, EX, CP, PAD> R;
  constexpr int S = R::S;
  constexpr int CW = sizeof(T) == 4 ? 1 : 2;
  constexpr int FB = kBits<T>;
  const int clc = PAD > 0 ? 1 : a.cl;
  const float rcl = 1.0f / (float)clc;
  long long* acc = reinterpret_cast<long long*>(smem);
  const int words = a.pad_cells * clc * CW;
  const Scratch sc(smem + (size_t)words * 8);
  const C* __restrict__ y = (const C*)y_;
  const C* __restrict__ ys = (const C*)ys_;
  const Lanes<S> ln;
  const int nq = it.z * clc;
  const int tail = R::tail(a);
  auto row_of = [&](int qq, int& cc) {
    if (PAD > 0) { cc = 0; return it.y + qq; }
    return it.y + fdiv(qq, clc, rcl, cc);
  };
  auto sample = [&](int r, int c) -> C {
    if (item_e) return ys[(int64_t)r * clc + c];
    return y[(int64_t)row_sample<T, D>(a, tail, r) * a.nb + a.c0 + c];
  };
  // the first row's record and sample are under way before the zeroing
  R rd;
  C yv = mk<T>((T)0, (T)0);
  int q = ln.q0 + ln.sl, c = 0, r = 0;
  if (ln.on && q < nq) {
    r = row_of(q, c);
    rd.load(a, r, ln.sub, clc, c);
    yv = sample(r, c);
  }
  for (int i = threadIdx.x; i < words; i += blockDim.x) acc[i] = 0;
  if (item_e) {
    if ((int)threadIdx.x < clc) sc.ex[threadIdx.x] = item_e[item * clc + threadIdx.x];
    __syncthreads();
  } else {
    if (clc > 1) {
      if (threadIdx.x < kMaxCl) sc.mx[threadIdx.x] = 0;
      __syncthreads();
    }
    double m = 0.0;
    for (int qq = q; ln.on && ln.sub == 0 && qq < nq; qq += ln.step) {
      int cc;
      const int rr = row_of(qq, cc);
      const double s = magnitude(qq == q ? yv : sample(rr, cc));
      if (clc == 1) m = fmax(m, s);
      else atomicMax(sc.mx + cc, (unsigned long long)__double_as_longlong(s));
    }
    coil_max(m, clc, sc.red, sc.mx);
    if ((int)threadIdx.x < clc) {
      const double ymax = __longlong_as_double((long long)sc.mx[threadIdx.x]);
      sc.ex[threadIdx.x] = fix_exponent(ymax, sizeof(T) == 4 ? a.item_bound[item] : a.u_bound);
    }
    __syncthreads();
  }
  while (ln.on && q < nq) {
    const int e = sc.ex[c];
    if (e != kPoisonExp) {
      const double scale = ldexp(1.0, FB - e);
      const C ph = row_phase<T>(a, tail, r);
      // conj(phase) y, scaled (exactly), in FP64
      const double yx = (double)yv.x * scale, yy = (double)yv.y * scale;
      const double px = ph.x, py = ph.y;
      rd.grid(a, acc, clc, make_double2(__builtin_fma(yx, px, yy * py),
                                           __builtin_fma(yy, px, -(yx * py))));
    }
    q += ln.step;
    if (q < nq) {
      r = row_of(q, c);
      rd.load(a, r, ln.sub, clc, c);
      yv = sample(r, c);
    }
  }
  __syncthreads();
  flush_slot<T>(a, it, clc, acc, sc.ex, part);
}

// P^H P of one item, on the modulated grid (or the plain one, a.stage: the
// box is modulated on its way in, the gather undoes it): the samples of the
// rows from the box, their exponent, then the rows gridded back.  A thread's
// first sample and record stay in registers between the two halves; further
// ones (more rows than threads) go through ybuf, written and read by the same
// thread.  sep: box and accumulator have LDS of their own, else the
// accumulator takes the box's once every row has read it.
template <typename T, int D, int JM, int JL, bool EX, int CP, int PAD>
__device__ __forceinline__ void php_body(const RealArgs& a, const int4 it, int item,
                                         unsigned char* smem, bool sep,
                                         const void* __restrict__ grid_, void* __restrict__ ybuf_,
                                         void* __restrict__ part) {
  typedef typename cplx<T>::t C;
  typedef Row<T, D, JM, JL, EX, CP, PAD> R;
  constexpr int S = R::S;
  constexpr int CW = sizeof(T) == 4 ? 1 : 2;
  constexpr int FB = kBits<T>;
  const int clc = PAD > 0 ? 1 : a.cl;
  const float rcl = 1.0f / (float)clc;
  C* box = reinterpret_cast<C*>(smem);
  const int words = a.pad_cells * clc * CW;      // box and accumulator alike
  long long* acc = reinterpret_cast<long long*>(smem + (sep ? (size_t)words * 8 : 0));
  const Scratch sc(smem + (size_t)words * (sep ? 16 : 8));
  C* __restrict__ ybuf = (C*)ybuf_;
  const Lanes<S> ln;
  const int nq = it.z * clc;
  auto row_of = [&](int qq, int& cc) {
    if (PAD > 0) { cc = 0; return it.y + qq; }
    return it.y + fdiv(qq, clc, rcl, cc);
  };
  R rd;
  int q = ln.q0 + ln.sl, c = 0;
  if (ln.on && q < nq) {
    const int r = row_of(q, c);
    rd.load(a, r, ln.sub, clc, c);
  }
  load_box<T, D>(a, Frame<D>(a, it.x), clc, box, (const C*)grid_);
  if (sep)
    for (int i = threadIdx.x; i < words; i += blockDim.x) acc[i] = 0;
  if (threadIdx.x < kMaxCl) sc.mx[threadIdx.x] = 0;
  __syncthreads();
  double m = 0.0;
  auto note = [&](C v, int cc) {
    const double s = magnitude(v);
    if (clc == 1) m = fmax(m, s);
    else atomicMax(sc.mx + cc, (unsigned long long)__double_as_longlong(s));
  };
  auto form = [&](const R& row, bool valid, int cc) -> C {
    C s = mk<T>((T)0, (T)0);
    if (valid) s = row.gather(a, box, clc);
    s = lanes_sum<S>(s, ln.sub);
    if (S > 1) {                                   // every lane of the row
      const int src = (int)(threadIdx.x & 63) - ln.sub;
      s.x = __shfl(s.x, src, 64);
      s.y = __shfl(s.y, src, 64);
    }
    if (valid && ln.sub == 0) note(s, cc);
    return s;
  };
  const bool has = ln.on && q < nq;
  const C y0 = form(rd, has, c);
  for (int q0 = ln.q0 + ln.step; q0 < nq; q0 += ln.step) {
    const int qq = q0 + ln.sl;
    const bool valid = ln.on && qq < nq;
    R row;
    int cc = 0, r = 0;
    if (valid) {
      r = row_of(qq, cc);
      row.load(a, r, ln.sub, clc, cc);
    }
    const C s = form(row, valid, cc);
    if (valid && ln.sub == 0) ybuf[(int64_t)r * clc + cc] = s;
  }
  coil_max(m, clc, sc.red, sc.mx);                 // every row has read the box
  if ((int)threadIdx.x < clc) {
    const double ymax = __longlong_as_double((long long)sc.mx[threadIdx.x]);
    sc.ex[threadIdx.x] = fix_exponent(ymax, sizeof(T) == 4 ? a.item_bound[item] : a.u_bound);
  }
  if (!sep)
    for (int i = threadIdx.x; i < words; i += blockDim.x) acc[i] = 0;
  __syncthreads();
  auto back = [&](const R& row, C v, int cc) {
    const int e = sc.ex[cc];
    if (e == kPoisonExp) return;
    const double scale = ldexp(1.0, FB - e);
    row.grid(a, acc, clc, make_double2((double)v.x * scale, (double)v.y * scale));
  };
  if (has) back(rd, y0, c);
  for (int q0 = ln.q0 + ln.step; q0 < nq; q0 += ln.step) {
    const int qq = q0 + ln.sl;
    R row;
    int cc = 0;
    if (ln.on && qq < nq) {
      const int r = row_of(qq, cc);
      row.load(a, r, ln.sub, clc, cc);
      // lanes sub > 0 re-read what their row's first lane wrote: same wave
      back(row, ybuf[(int64_t)r * clc + cc], cc);
    }
  }
  __syncthreads();
  flush_slot<T>(a, it, clc, acc, sc.ex, part);
}

// P^H P of one item in one pass over its rows (complex128, one coil, box and
// accumulator both in LDS): a row is gridded as soon as its sample is formed.
// The exponent is fixed before the first add from a bound of every sample:
// the factors are real, so |Re y| <= row_bound max |Re k| over the box (and Im
// alike).  It depends on the tile's box alone, so the sums do not change with
// how a tile's rows are cut into items.  A sample that is not finite poisons
// the slot.  pq (or null): the item's sum of |y|^2, its part of <k, P^H P k>.
template <int D, int JM, int JL, bool EX, int CP, int PAD>
__device__ __forceinline__ void php1_body(const RealArgs& a, const int4 it, unsigned char* smem,
                                          const void* __restrict__ grid_,
                                          void* __restrict__ part, double2* __restrict__ pq) {
  typedef Row<double, D, JM, JL, EX, CP, PAD> R;
  constexpr int S = R::S;
  double2* box = reinterpret_cast<double2*>(smem);
  const int words = a.pad_cells * 2;
  long long* acc = reinterpret_cast<long long*>(smem + (size_t)words * 8);
  const Scratch sc(smem + (size_t)words * 16);
  const Lanes<S> ln;
  const int nq = it.z;
  R rd;
  int q = ln.q0 + ln.sl;
  if (ln.on && q < nq) rd.load(a, it.y + q, ln.sub, 1, 0);
  double m = 0.0;
  load_box<double, D>(a, Frame<D>(a, it.x), 1, box, (const double2*)grid_, [&](double2 v) {
    // non-finite values are caught in the samples they reach
    const double s = fmax(fabs(v.x), fabs(v.y));
    if (s <= 1.0e300) m = fmax(m, s);
  });
  for (int i = threadIdx.x; i < words; i += blockDim.x) acc[i] = 0;
  if (threadIdx.x == 0) sc.ex[1] = 0;
  m = block_max(m, sc.red);                        // also the barrier after the box
  // (1 + 2^-20): room for the rounding of the products; the plain grid is
  // modulated on its way in, which can raise a part by sqrt(2)
  const double B = fmin(a.row_bound * a.u_bound * m * (a.stage ? 1.5 : 1.0 + 0x1p-20), 1.0e300);
  int e = 0;
  if (B > 0.0) (void)frexp(B, &e);
  if (e < -960) e = -960;
  const double scale = ldexp(1.0, kFixBits - e);
  bool bad = false;
  double sq = 0.0;
  for (int q0 = ln.q0; q0 < nq; q0 += ln.step) {
    const bool valid = ln.on && q < nq;
    double2 s = make_double2(0.0, 0.0);
    if (valid) s = rd.gather(a, box, 1);
    s = lanes_sum<S>(s, ln.sub);
    if (S > 1) {                                   // every lane of the row
      const int src = (int)(threadIdx.x & 63) - ln.sub;
      s.x = __shfl(s.x, src, 64);
      s.y = __shfl(s.y, src, 64);
    }
    if (valid && ln.sub == 0) sq += s.x * s.x + s.y * s.y;
    if (valid) {
      if (fabs(s.x) + fabs(s.y) <= 1.0e300)
        rd.grid(a, acc, 1, make_double2(s.x * scale, s.y * scale));
      else
        bad = true;
    }
    q += ln.step;
    if (ln.on && q < nq) rd.load(a, it.y + q, ln.sub, 1, 0);
  }
  if (bad) sc.ex[1] = 1;
  __syncthreads();                                 // red's maxima have been read
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sq += __shfl_xor(sq, off, 64);
  if ((threadIdx.x & 63) == 0) sc.red[threadIdx.x >> 6] = sq;
  __syncthreads();
  if (threadIdx.x == 0) {
    sc.ex[0] = sc.ex[1] ? kPoisonExp : e;
    if (pq) {
      for (int w = 1; w < (int)(blockDim.x >> 6); ++w) sq += sc.red[w];
      *pq = make_double2(sq, 0.0);
    }
  }
  __syncthreads();
  flush_slot<double>(a, it, 1, acc, sc.ex, part);
}

// Grid cells from the partial slots that cover them.  A cell of tile t sums,
// in a fixed order, the slots of the tiles whose padded box holds it: its own
// and, per set of axes, the tiles below along them, whose padding reaches the
// J_d - 1 lowest cells (across the grid's edge with mod's sign).
template <int D>
struct Tile {
  int td[3], T0[3], E[3], below[3];
  __device__ __forceinline__ Tile(const RealArgs& a, int tile) {
    int rest = tile;
#pragma unroll
    for (int d = D - 1; d >= 0; --d) {
      const int tg = a.tgrid[d], q = rest / tg;
      td[d] = rest - q * tg;
      rest = q;
      T0[d] = td[d] * a.tile[d];
      E[d] = min(a.tile[d], a.K[d] - T0[d]);
      below[d] = tg == 1 ? 0 : a.J[d] - 1;
    }
  }
  // source m (bit d: the tile below along axis d): its slots (first, count),
  // the offset of this tile's cells in them and whether they change sign
  __device__ __forceinline__ int2 source(const RealArgs& a, int m, int& off, bool& neg) const {
    int t = 0;
    bool ok = true;
    off = 0;
    neg = false;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const bool bit = (m >> d) & 1;
      ok &= !bit || below[d] > 0;
      const int q = bit ? (td[d] == 0 ? a.tgrid[d] - 1 : td[d] - 1) : td[d];
      if (bit && td[d] == 0) neg ^= a.flip[d] != 0;
      t = t * a.tgrid[d] + q;
      off = off * (d == 0 ? 1 : a.pad[d]) + (bit ? min(a.tile[d], a.K[d] - q * a.tile[d]) : 0);
    }
    int2 ts = reinterpret_cast<const int2*>(a.tile_slots)[ok ? t : 0];
    if (!ok) ts.y = 0;
    return ts;
  }
  // conj(mod) of a cell (plain grids)
  template <typename C>
  __device__ __forceinline__ C plain(const RealArgs& a, C s, int x0, int x1, int x2) const {
    C m = ((const C*)a.mod[0])[T0[0] + x0];
    if (D > 1) m = cmul_f(m, ((const C*)a.mod[1])[T0[1] + x1]);
    if (D > 2) m = cmul_f(m, ((const C*)a.mod[2])[T0[2] + x2]);
    return conj_mul(s, m);
  }
};

// At most one slot a tile: one workgroup per tile.  A thread keeps one place
// of the trailing axes and walks the leading one, so the sources' predicates
// and addresses are made once, and four planes' loads are in flight (3-D
// 256^3: 118 us with every cell's sources worked out anew, 106 so; 437 MB).
template <typename T, int D>
__device__ __forceinline__ void gather_single(const RealArgs& a, int tile,
                                              const void* __restrict__ part_,
                                              void* __restrict__ grid_) {
  typedef typename cplx<T>::t C;
  const C* __restrict__ part = (const C*)part_;
  C* __restrict__ grid = (C*)grid_;
  const Tile<D> src(a, tile);
  constexpr int NS = 1 << D;
  int slot[NS], cnt[NS], off[NS];
  T sgn[NS];
#pragma unroll
  for (int m = 0; m < NS; ++m) {
    bool neg;
    const int2 ts = src.source(a, m, off[m], neg);
    slot[m] = ts.x;
    cnt[m] = ts.y;
    sgn[m] = neg ? (T)-1 : (T)1;
  }
  const int clc = a.cl;
  constexpr int NT = 1 << (D - 1);                 // trailing sets
  const int P1 = D > 1 ? a.pad[1] : 1, P2 = D > 2 ? a.pad[2] : 1;
  const int E0 = src.E[0], E1 = D > 1 ? src.E[1] : 1, E2 = D > 2 ? src.E[2] : 1;
  const int I = E1 * E2 * clc;                     // elements of a leading plane
  const int64_t s0 = D == 1 ? 1 : (D == 2 ? (int64_t)a.K[1] : (int64_t)a.K[1] * a.K[2]);
  const int64_t stride = (int64_t)a.pad_cells * clc;
  const int pl = P1 * P2 * clc;                    // slot elements of a leading plane
  auto column = [&](int i, int from, int by) {
    const int t = i / clc, c = i - t * clc;
    int x1 = 0, x2 = 0;
    if (D == 2) x1 = t;
    if (D == 3) { x1 = t / E2; x2 = t - x1 * E2; }
    const int tc = (D == 1 ? 0 : (D == 2 ? x1 : x1 * P2 + x2)) * clc + c;
    bool okt[NT];
#pragma unroll
    for (int m = 0; m < NT; ++m)
      okt[m] = (!(m & 1) || x1 < src.below[1]) && (D < 3 || !(m & 2) || x2 < src.below[2]);
    int64_t gt = 0;
    if (D == 2) gt = src.T0[1] + x1;
    if (D == 3) gt = (int64_t)(src.T0[1] + x1) * a.K[2] + src.T0[2] + x2;
    auto put = [&](int x0, C s) {
      if (a.stage) s = src.plain(a, s, x0, x1, x2);
      grid[((src.T0[0] + x0) * s0 + gt) * a.nb + a.c0 + c] = s;
    };
    if (a.n_items == 0) {                          // no slot to read
      for (int x0 = from; x0 < E0; x0 += by) put(x0, mk<T>((T)0, (T)0));
      return;
    }
    // U planes from x0; LEAD: within the leading axis's padding; TS: step of
    // the trailing sets looked at (2: none of axis 1's).  A source that does
    // not apply reads the cell's own place in slot 0 and counts nothing.
    auto planes = [&](auto ucnt, auto lead, auto tstep, int x0) {
      constexpr int U = decltype(ucnt)::value, L = decltype(lead)::value ? 2 : 1;
      constexpr int TS = decltype(tstep)::value, NM = NT / TS;
      C v[U][L][NM];
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int b = 0; b < L; ++b)
#pragma unroll
          for (int m = 0; m < NM; ++m) {
            const int q = b + 2 * m * TS;
            const bool ok = okt[m * TS] && cnt[q] > 0;
            const int64_t own = (int64_t)(x0 + u * by) * pl + tc;
            v[u][b][m] = part[ok ? slot[q] * stride + own + (int64_t)off[q] * clc : own];
          }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        C s = mk<T>((T)0, (T)0);
#pragma unroll
        for (int b = 0; b < L; ++b)
#pragma unroll
          for (int m = 0; m < NM; ++m) {
            const int q = b + 2 * m * TS;
            if (okt[m * TS] && cnt[q] > 0) {
              s.x = fma(sgn[q], v[u][b][m].x, s.x);
              s.y = fma(sgn[q], v[u][b][m].y, s.y);
            }
          }
        put(x0 + u * by, s);
      }
    };
    auto run = [&](auto tstep) {
      typedef std::integral_constant<int, 1> U1;
      typedef std::integral_constant<int, 4> U4;
      int x0 = from;
      for (; x0 < E0 && x0 < src.below[0]; x0 += by)
        planes(U1(), std::integral_constant<bool, true>(), tstep, x0);
      for (; x0 + 3 * by < E0; x0 += 4 * by)
        planes(U4(), std::integral_constant<bool, false>(), tstep, x0);
      for (; x0 < E0; x0 += by) planes(U1(), std::integral_constant<bool, false>(), tstep, x0);
    };
    // 3-D: waves whose lanes all lie past axis 1's padding skip its sources
    if (D == 3 && !__any(okt[NT > 1 ? 1 : 0])) run(std::integral_constant<int, D == 3 ? 2 : 1>());
    else run(std::integral_constant<int, 1>());
  };
  const int tid = threadIdx.x, nthr = blockDim.x;
  if (I <= nthr) {
    const int G = nthr / I, og = tid / I;
    if (og < G) column(tid - og * I, og, G);
  } else {
    for (int i = tid; i < I; i += nthr) column(i, 0, 1);
  }
}

// Tiles of several slots (dense regions, whose rows make many work items):
// one element (cell, coil) per thread.  The workgroup lists the slots of all
// sources (a thread each), then every thread walks the list, sixteen loads at
// a time whichever source they belong to: a dense tile's time is its chain of
// load rounds, every other tile's the few loads on the way to the first sum.
constexpr int kGatherThreads = 256;

//
// out.begin(g) sees the thread's grid element before its sum is formed, every
// thread calls out.middle(), and out.end(g, sum) follows for real elements.
template <typename T, int D, typename O>
__device__ __forceinline__ void gather_multi(const RealArgs& a, int tile, int part_i,
                                             const void* __restrict__ part_, O&& out) {
  typedef typename cplx<T>::t C;
  constexpr int NS = 1 << D;
  __shared__ int4 sources[NS];                     // first slot, slots, offset, sign
  __shared__ long long list[kGatherThreads];       // element offset * 16 + sign * 8 + source
  const C* __restrict__ part = (const C*)part_;
  const Tile<D> src(a, tile);
  const int clc = a.cl, tid = threadIdx.x;
  if (tid < NS) {
    int off;
    bool neg;
    const int2 ts = src.source(a, tid, off, neg);
    sources[tid] = make_int4(ts.x, ts.y, off, neg);
  }
  const int P1 = D > 1 ? a.pad[1] : 1, P2 = D > 2 ? a.pad[2] : 1;
  const int E1 = D > 1 ? src.E[1] : 1, E2 = D > 2 ? src.E[2] : 1;
  const int total = src.E[0] * E1 * E2 * clc;
  const int64_t stride = (int64_t)a.pad_cells * clc;
  const int e0 = part_i * kGatherThreads + tid;
  const int e = min(e0, total - 1);
  const int t = e / clc, c = e - t * clc;
  int x0 = t, x1 = 0, x2 = 0;
  if (D == 2) { x0 = t / E1; x1 = t - x0 * E1; }
  if (D == 3) {
    const int p = t / E2;
    x2 = t - p * E2;
    x0 = p / E1;
    x1 = p - x0 * E1;
  }
  int64_t g = src.T0[0] + x0;
  if (D > 1) g = g * a.K[1] + src.T0[1] + x1;
  if (D > 2) g = g * a.K[2] + src.T0[2] + x2;
  g = g * a.nb + a.c0 + c;
  out.begin(g);
  const int64_t own = (int64_t)((x0 * P1 + x1) * P2 + x2) * clc + c;
  unsigned bits = 0;                               // sources that reach the cell
#pragma unroll
  for (int m = 0; m < NS; ++m)
    bits |= ((!(m & 1) || x0 < src.below[0]) && (D < 2 || !(m & 2) || x1 < src.below[1]) &&
             (D < 3 || !(m & 4) || x2 < src.below[2]) ? 1u : 0u) << m;
  C s = mk<T>((T)0, (T)0);
  __syncthreads();
  int n = 0;
#pragma unroll
  for (int m = 0; m < NS; ++m) n += sources[m].y;
  for (int base = 0; base < n; base += kGatherThreads) {
    const int nb = min(n - base, kGatherThreads);
    if (base) __syncthreads();                     // the list is used again
    if (tid < nb) {
      int i = base + tid, m = 0;
      int4 q = sources[0];
      while (i >= q.y) { i -= q.y; q = sources[++m]; }
      list[tid] = ((int64_t)(q.x + i) * stride + (int64_t)q.z * clc) * 16 + q.w * 8 + m;
    }
    __syncthreads();
    auto round = [&](auto nq, int k) {
      constexpr int NQ = decltype(nq)::value;
      C v[NQ];
      T f[NQ];
#pragma unroll
      for (int j = 0; j < NQ; ++j) {
        const long long l = list[min(k + j, nb - 1)];
        const bool use = k + j < nb && (bits >> (l & 7) & 1);
        f[j] = use ? (l & 8 ? (T)-1 : (T)1) : (T)0;
        v[j] = mk<T>((T)0, (T)0);
        if (use) v[j] = part[(l >> 4) + own];
      }
#pragma unroll
      for (int j = 0; j < NQ; ++j) v[j] = mk<T>(v[j].x * f[j], v[j].y * f[j]);
#pragma unroll
      for (int h = NQ / 2; h >= 1; h /= 2)
#pragma unroll
        for (int j = 0; j < h; ++j) v[j] = cadd(v[2 * j], v[2 * j + 1]);
      s = cadd(s, v[0]);
    };
    int k = 0;
    for (; nb - k > 8; k += 16) round(std::integral_constant<int, 16>(), k);
    if (nb - k > 4) round(std::integral_constant<int, 8>(), k);
    else if (nb - k > 0) round(std::integral_constant<int, 4>(), k);
  }
  out.middle();
  if (e0 < total) {
    if (a.stage) s = src.plain(a, s, x0, x1, x2);
    out.end(g, s);
  }
}

// gather_multi's element to the grid
template <typename C>
struct ToGrid {
  C* __restrict__ grid;
  __device__ __forceinline__ void begin(int64_t) {}
  __device__ __forceinline__ void middle() {}
  __device__ __forceinline__ void end(int64_t g, C s) { grid[g] = s; }
};

// gather_multi's element as a step of the conjugate gradients.  STEP: it is
// (P^H P p)[g]; alpha = rho / (p . q) from the items' sums of |P p|^2, then
// x += alpha p, r -= alpha q (q is never stored).  Otherwise it is the right
// side: r = b, x = 0.  sq: the thread's |r|^2.
template <bool STEP>
struct ToCg {
  double2* __restrict__ x;
  double2* __restrict__ r;
  const double2* __restrict__ p;
  const double2* __restrict__ pq;
  int n_pq;
  double rho;
  double2* red;
  double sq;
  double alpha;
  double2 xv, rv, pv, sum;                         // sum: this thread's part of pq
  __device__ __forceinline__ void begin(int64_t g) {
    sq = 0.0;
    if (!STEP) return;
    xv = x[g];
    rv = r[g];
    pv = p[g];
    sum = make_double2(0.0, 0.0);
    for (int i = threadIdx.x; i < n_pq; i += kGatherThreads) sum.x += pq[i].x;
  }
  __device__ __forceinline__ void middle() {
    if (!STEP) return;
    const double t = sum_block256(sum, red).x;
    alpha = rho * t / (t * t);
  }
  __device__ __forceinline__ void end(int64_t g, double2 s) {
    if (STEP) {
      x[g] = make_double2(xv.x + alpha * pv.x, xv.y + alpha * pv.y);
      s = make_double2(rv.x - alpha * s.x, rv.y - alpha * s.y);
    } else {
      x[g] = make_double2(0.0, 0.0);
    }
    r[g] = s;
    sq = s.x * s.x + s.y * s.y;
  }
};

// ---------------------------------------------------------------- kernels --
template <typename T, int D, int JM, int JL, bool EX, int CP, int PAD>
__global__ void __launch_bounds__(1024, D == 3 && sizeof(T) == 4 && PAD != 0 ? 8 : 1)
__attribute__((amdgpu_num_sgpr(80)))
real_k2y_kernel(RealArgs a, const void* __restrict__ grid, void* __restrict__ y,
                const int* __restrict__ skip) {
  if (skip && *skip) return;
  extern __shared__ __align__(16) unsigned char smem[];
  const int4 it = reinterpret_cast<const int4*>(a.items)[blockIdx.x];
  k2y_body<T, D, JM, JL, EX, CP, PAD>(a, it, smem, grid, y);
}

template <typename T, int D, int JM, int JL, bool EX, int CP, int PAD>
__global__ void __launch_bounds__(1024, D == 3 && sizeof(T) == 4 ? 6 : 1)
real_y2k_kernel(RealArgs a, const void* __restrict__ y, void* __restrict__ part,
                const int* __restrict__ item_e, const void* __restrict__ ys,
                const int* __restrict__ skip) {
  if (skip && *skip) return;
  extern __shared__ __align__(16) unsigned char smem[];
  const int4 it = reinterpret_cast<const int4*>(a.items)[blockIdx.x];
  y2k_body<T, D, JM, JL, EX, CP, PAD>(a, it, blockIdx.x, smem, y, part, item_e, ys);
}

template <typename T, int D, int JM, int JL, bool EX, int CP, int PAD>
__global__ void __launch_bounds__(1024)
real_php_kernel(RealArgs a, int sep, const void* __restrict__ grid, void* __restrict__ ybuf,
                void* __restrict__ part, const int* __restrict__ skip) {
  if (skip && *skip) return;
  extern __shared__ __align__(16) unsigned char smem[];
  const int4 it = reinterpret_cast<const int4*>(a.items)[blockIdx.x];
  php_body<T, D, JM, JL, EX, CP, PAD>(a, it, blockIdx.x, smem, sep, grid, ybuf, part);
}

template <int D, int JM, int JL, bool EX, int CP, int PAD>
__global__ void __launch_bounds__(1024)
real_php1_kernel(RealArgs a, const void* __restrict__ grid, void* __restrict__ part,
                 double2* __restrict__ pq, const int* __restrict__ skip) {
  if (skip && *skip) return;
  extern __shared__ __align__(16) unsigned char smem[];
  const int4 it = reinterpret_cast<const int4*>(a.items)[blockIdx.x];
  php1_body<D, JM, JL, EX, CP, PAD>(a, it, smem, grid, part, pq ? pq + blockIdx.x : nullptr);
}

// Exponents of all items ahead of the gridding (long work lists), the samples
// stored in row order on the way.
template <typename T, int D>
__global__ void __launch_bounds__(256)
real_exponent_kernel(RealArgs a, const void* __restrict__ y_, int* __restrict__ item_e,
                     void* __restrict__ ys_, const int* __restrict__ skip) {
  typedef typename cplx<T>::t C;
  if (skip && *skip) return;
  __shared__ double red[16];
  __shared__ unsigned long long mx[kMaxCl];
  const int clc = a.cl;
  const int4 it = reinterpret_cast<const int4*>(a.items)[blockIdx.x];
  const C* __restrict__ y = (const C*)y_;
  C* __restrict__ ys = (C*)ys_;
  if (threadIdx.x < kMaxCl) mx[threadIdx.x] = 0;
  __syncthreads();
  const float rcl = 1.0f / (float)clc;
  double m = 0.0;
  for (int q = threadIdx.x; q < it.z * clc; q += blockDim.x) {
    int c = 0;
    const int r = it.y + (clc == 1 ? q : fdiv(q, clc, rcl, c));
    const C v = y[(int64_t)a.perm[r] * a.nb + a.c0 + c];
    ys[(int64_t)r * clc + c] = v;
    const double s = magnitude(v);
    if (clc == 1) m = fmax(m, s);
    else atomicMax(mx + c, (unsigned long long)__double_as_longlong(s));
  }
  coil_max(m, clc, red, mx);
  if ((int)threadIdx.x < clc) {
    const double ymax = __longlong_as_double((long long)mx[threadIdx.x]);
    item_e[blockIdx.x * clc + threadIdx.x] =
        fix_exponent(ymax, sizeof(T) == 4 ? a.item_bound[blockIdx.x] : a.u_bound);
  }
}

template <typename T, int D>
__global__ void __launch_bounds__(256)
real_gather_kernel(RealArgs a, const void* __restrict__ part, void* __restrict__ grid,
                   const int* __restrict__ skip) {
  if (skip && *skip) return;
  gather_single<T, D>(a, blockIdx.x, part, grid);
}

template <typename T, int D>
__global__ void __launch_bounds__(kGatherThreads)
real_gather_multi_kernel(RealArgs a, int parts, const void* __restrict__ part,
                         void* __restrict__ grid, const int* __restrict__ skip) {
  if (skip && *skip) return;
  const int t = blockIdx.x / parts;
  gather_multi<T, D>(a, t, blockIdx.x - t * parts, part, ToGrid<typename cplx<T>::t>{(typename cplx<T>::t*)grid});
}

// The gather as a step of the conjugate gradients (complex128, one coil).
template <int D, bool STEP>
__global__ void __launch_bounds__(kGatherThreads)
real_gather_cg_kernel(RealArgs a, int parts, const void* __restrict__ part, RealCg cg,
                      const int* __restrict__ skip) {
  if (skip && *skip) return;
  __shared__ double2 red[4];
  ToCg<STEP> o{(double2*)cg.x, (double2*)cg.r, (const double2*)cg.p, (const double2*)cg.pq,
               cg.n_pq, STEP ? *cg.rho : 0.0, red};
  const int t = blockIdx.x / parts;
  gather_multi<double, D>(a, t, blockIdx.x - t * parts, part, o);
  const double2 v = sum_block256(make_double2(o.sq, 0.0), red);
  if (threadIdx.x == 0) ((double2*)cg.rr)[blockIdx.x] = v;
}

// Per item, the largest over its box of the sum over its rows of |coef|, in
// 64-bit fixed point, rounded up (as item_bound_kernel).
template <int D>
__global__ void __launch_bounds__(256)
real_bound_kernel(RealArgs a, double* __restrict__ bound) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ double red[16];
  long long* acc = reinterpret_cast<long long*>(smem);
  const int4 it = reinterpret_cast<const int4*>(a.items)[blockIdx.x];
  for (int i = threadIdx.x; i < a.pad_cells; i += blockDim.x) acc[i] = 0;
  int eu = 0;
  (void)frexp(a.u_bound, &eu);
  const double scale = ldexp(1.0, kFixBits - eu);
  __syncthreads();
  const int J0 = D > 1 ? a.J[0] : 1, J1 = D > 2 ? a.J[1] : 1, JL = a.J[D - 1];
  const int bl = D == 1 ? 0 : (D == 2 ? J0 : J0 + J1), tail = bl + JL;
  const int P1 = D > 1 ? a.pad[1] : 1, P2 = D > 2 ? a.pad[2] : 1;
  auto at = [&](int d, int x) { return a.tgrid[d] == 1 && x >= a.K[d] ? x - a.K[d] : x; };
  const int n = it.z * JL;
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    const int q = i / JL, jl = i - q * JL;
    const float* p = (const float*)a.rec + (int64_t)(it.y + q) * a.rw;
    const int w = __float_as_int(p[tail + 2]);
    const int x0 = w & 0xffff, x1 = (unsigned)w >> 16;
    const int x2 = D > 2 ? __float_as_int(p[tail + 3]) : 0;
    const int xl = D == 1 ? x0 : (D == 2 ? x1 : x2);
    const double wl = fabs((double)p[bl + jl]) * scale;
    for (int j0 = 0; j0 < J0; ++j0) {
      const double w0 = D > 1 ? wl * fabs((double)p[j0]) : wl;
      for (int j1 = 0; j1 < J1; ++j1) {
        const double w1 = D > 2 ? w0 * fabs((double)p[J0 + j1]) : w0;
        int cell = at(D - 1, xl + jl);
        if (D > 1) cell += at(0, x0 + j0) * P1 * P2;
        if (D > 2) cell += at(1, x1 + j1) * P2;
        lds_add(acc + cell, __double_as_longlong(w1 + kMagic) - kMagicBits);
      }
    }
  }
  __syncthreads();
  double m = 0.0;
  for (int i = threadIdx.x; i < a.pad_cells; i += blockDim.x) m = fmax(m, (double)acc[i]);
  m = block_max(m, red);
  if (threadIdx.x == 0)
    bound[blockIdx.x] = (m + 0.5 * n + 1.0) * ldexp(1.0, eu - kFixBits) * (1.0 + 0x1p-20);
}

// Batches: each workgroup looks up its problem and runs the single-problem
// body on that problem's slice of the packed vectors.
template <typename T>
__device__ __forceinline__ const RealArgs& batch_args(const BatchProblem& p) {
  if constexpr (sizeof(T) == 8) return p.ra64;
  else return p.ra;
}

template <typename T, int D, int JM, int JL, bool EX, int CP, int PAD>
__global__ void __launch_bounds__(1024)
real_k2y_batch_kernel(const BatchProblem* __restrict__ probs, const int2* __restrict__ items,
                      const void* __restrict__ k, void* __restrict__ y,
                      const int* __restrict__ done, const int* __restrict__ all_done) {
  typedef typename cplx<T>::t C;
  if (all_done && *all_done) return;
  const int2 pi = items[blockIdx.x];
  const BatchProblem& p = probs[pi.x];
  if (done && done[pi.x]) return;
  extern __shared__ __align__(16) unsigned char smem[];
  const RealArgs a = batch_args<T>(p);             // copied: the stores may alias it
  const int4 it = reinterpret_cast<const int4*>(a.items)[pi.y];
  k2y_body<T, D, JM, JL, EX, CP, PAD>(a, it, smem, (const C*)k + p.k_off, (C*)y + p.y_off);
}

template <typename T, int D, int JM, int JL, bool EX, int CP, int PAD>
__global__ void __launch_bounds__(1024)
real_y2k_batch_kernel(const BatchProblem* __restrict__ probs, const int2* __restrict__ items,
                      const void* __restrict__ y, void* __restrict__ part,
                      const int* __restrict__ done, const int* __restrict__ all_done) {
  typedef typename cplx<T>::t C;
  if (all_done && *all_done) return;
  const int2 pi = items[blockIdx.x];
  const BatchProblem& p = probs[pi.x];
  if (done && done[pi.x]) return;
  extern __shared__ __align__(16) unsigned char smem[];
  const RealArgs a = batch_args<T>(p);             // copied: the stores may alias it
  const int4 it = reinterpret_cast<const int4*>(a.items)[pi.y];
  y2k_body<T, D, JM, JL, EX, CP, PAD>(a, it, pi.y, smem, (const C*)y + p.y_off,
                                      (C*)part + p.part_off, nullptr, nullptr);
}

template <int D, int JM, int JL, bool EX, int CP, int PAD, bool ONE>
__global__ void __launch_bounds__(1024)
real_php_batch_kernel(const BatchProblem* __restrict__ probs, const int2* __restrict__ items,
                      int sep, const void* __restrict__ k, void* __restrict__ ybuf,
                      void* __restrict__ part, double2* __restrict__ pq,
                      const int* __restrict__ done, const int* __restrict__ all_done) {
  if (all_done && *all_done) return;
  const int2 pi = items[blockIdx.x];
  const BatchProblem& p = probs[pi.x];
  if (done && done[pi.x]) return;
  extern __shared__ __align__(16) unsigned char smem[];
  const RealArgs a = p.ra64;                       // copied: the stores may alias it
  const int4 it = reinterpret_cast<const int4*>(a.items)[pi.y];
  if constexpr (ONE)
    php1_body<D, JM, JL, EX, CP, PAD>(a, it, smem, (const double2*)k + p.k_off,
                                      (double2*)part + p.part_off,
                                      pq ? pq + p.item_off + pi.y : nullptr);
  else
    php_body<double, D, JM, JL, EX, CP, PAD>(a, it, pi.y, smem, sep, (const double2*)k + p.k_off,
                                             (double2*)ybuf + p.y_off,
                                             (double2*)part + p.part_off);
}

template <typename T, int D>
__global__ void __launch_bounds__(kGatherThreads)
real_gather_batch_kernel(const BatchProblem* __restrict__ probs, BatchTable t,
                         const void* __restrict__ part, void* __restrict__ k,
                         const int* __restrict__ done, const int* __restrict__ all_done) {
  typedef typename cplx<T>::t C;
  if (all_done && *all_done) return;
  const int pr = t.tab[blockIdx.x];
  if (done && done[pr]) return;
  const BatchProblem& p = probs[pr];
  const RealArgs a = batch_args<T>(p);             // copied: the stores may alias it
  const int lb = (int)(blockIdx.x - t.first[pr]);
  const int parts = pnh_real_gather_parts(a, D);
  const int tile = lb / parts;
  gather_multi<T, D>(a, tile, lb - tile * parts, (const C*)part + p.part_off,
                     ToGrid<C>{(C*)k + p.k_off});
}

template <int D, bool STEP>
__global__ void __launch_bounds__(kGatherThreads)
real_gather_cg_batch_kernel(const BatchProblem* __restrict__ probs, BatchTable t,
                            const void* __restrict__ part, double2* __restrict__ x,
                            double2* __restrict__ r, const double2* __restrict__ p_,
                            const double2* __restrict__ pq, const double* __restrict__ rho,
                            double2* __restrict__ rr, const int* __restrict__ done) {
  const int pr = t.tab[blockIdx.x];
  if (done && done[pr]) return;
  __shared__ double2 red[4];
  const BatchProblem& p = probs[pr];
  const RealArgs a = batch_args<double>(p);        // copied: the stores may alias it
  ToCg<STEP> o{x + p.k_off, r + p.k_off, p_ + p.k_off, pq + p.item_off, (int)a.n_items,
               STEP ? rho[pr] : 0.0, red};
  const int lb = (int)(blockIdx.x - t.first[pr]);
  const int parts = pnh_real_gather_parts(a, D);
  const int tile = lb / parts;
  gather_multi<double, D>(a, tile, lb - tile * parts, (const double2*)part + p.part_off, o);
  const double2 v = sum_block256(make_double2(o.sq, 0.0), red);
  if (threadIdx.x == 0) rr[blockIdx.x] = v;
}

// --------------------------------------------------------------- dispatch --
// Calls f(JM, JL, EX, CP, PAD) for the supports of a: uniform supports of 4
// to 8 exactly, others up to 8 or 16 per axis with guards (the last axis's
// extent exact down to 4).  CP: one lane per row in 1-D and 2-D, one per
// last-axis cell in 3-D.
template <int V> using I = std::integral_constant<int, V>;
template <bool V> using B = std::integral_constant<bool, V>;

// Lanes per row.  1-D and complex64 2-D take one: their launches wait on memory,
// and then every row's record is loaded at once (512x512, 205 824 samples, one
// lane against six: k2y 6.9 us against 10.1, y2k 11.9 against 15.8; eight
// coils, 131 072 samples, 17.6 against 53.4 and 25.3 against 75.5).  3-D and
// complex128 take one lane per last-axis cell, whose runs of neighbouring
// cells conflict least in LDS (batches of P^H P, 2-D complex128: 164 us an
// iteration over all streams against 290 with one lane a row; a single
// problem's 21.5 against 21.0).
template <typename T, int D, typename F>
int dispatch(const int* J, int how, F&& f) {
  constexpr bool wide = D == 1 || (D == 2 && sizeof(T) == 4);
  const int jl = J[D - 1];
  const int jm = D == 1 ? 1 : (D == 2 ? J[0] : (J[0] > J[1] ? J[0] : J[1]));
  bool same = D > 1;
  for (int d = 0; d < D; ++d) same = same && J[d] == jl;
  typedef I<0> Wrap;
  typedef I<-1> Split;
#define PNH_EX(j)                                                                            \
  if (same && jl == j) {                                                                     \
    if (how > 0)                                                                             \
      return f(I<j>(), I<j>(), B<true>(), I<wide ? j : 1>(), I<15 + j>());                 \
    return f(I<j>(), I<j>(), B<true>(), I<wide ? j : 1>(), Split());                       \
  }
#define PNH_GEN(j)                                                                           \
  {                                                                                          \
    if (how != 0) return f(I<D == 1 ? 1 : 8>(), I<j>(), B<false>(), I<wide ? j : 1>(), Split()); \
    return f(I<D == 1 ? 1 : 8>(), I<j>(), B<false>(), I<wide ? j : 1>(), Wrap());          \
  }
  if constexpr (D > 1) {
    if (how != 0) {
      PNH_EX(4) PNH_EX(6) PNH_EX(8)
    }
  }
  if (jm <= 8 && jl <= 8) {
    switch (jl) {
      case 5: PNH_GEN(5)
      case 6: PNH_GEN(6)
      case 7: PNH_GEN(7)
      case 8: PNH_GEN(8)
      default: PNH_GEN(4)
    }
  }
#undef PNH_EX
#undef PNH_GEN
  if (jm <= 16 && jl <= 16)
    return f(I<D == 1 ? 1 : 16>(), I<16>(), B<false>(), I<wide ? 16 : 1>(), I<0>());
  pnh_set_error("interpolator size above 16");
  return -2;
}

// How the supports lie in the boxes: 0, some axis is spanned by one tile; 1,
// every axis is cut into tiles, boxes of 15 + J cells (16-cell tiles) and one
// coil; -1 every axis is cut.
template <int D>
int layout_of(const RealArgs& a) {
  bool fixed = D > 1 && a.cl == 1;
  for (int d = 0; d < D; ++d) {
    if (a.tgrid[d] == 1) return 0;
    fixed = fixed && a.pad[d] == 15 + a.J[d];
  }
  return fixed ? 1 : -1;
}

// Whether the gridding computes the items' exponents in a pass ahead, which
// also stores the samples in row order (one launch more: long work lists).
bool exponent_pass(int fp64, const RealArgs& a, int cl) {
  return a.n_items >= PNH_EXPONENT_PASS_ITEMS && (!fp64 || cl == 1);
}

size_t acc_bytes(const RealArgs& a, size_t esz) { return (size_t)a.pad_cells * a.cl * esz; }

bool threads_ok(int t) {
  if (t >= 64 && t <= 1024 && t % 64 == 0) return true;
  pnh_set_error("workgroup size %d is not a multiple of 64 in 64..1024", t);
  return false;
}

template <typename T>
int launch_gather(const RealArgs& a, const void* slots, void* grid, const int* skip,
                  hipStream_t s) {
  if (a.max_tile_slots <= 1) {
    hipLaunchKernelGGL((real_gather_kernel<T, PNH_D>), dim3((unsigned)a.n_tiles), dim3(256), 0, s,
                       a, slots, grid, skip);
  } else {
    const int parts = pnh_real_gather_parts(a, PNH_D);
    hipLaunchKernelGGL((real_gather_multi_kernel<T, PNH_D>), dim3((unsigned)(a.n_tiles * parts)),
                       dim3(kGatherThreads), 0, s, a, parts, slots, grid, skip);
  }
  PNH_LAUNCH_CHECK();
  return 0;
}

template <typename T>
int launch_k2y(const RealArgs& a, const void* grid, void* y, const int* skip, hipStream_t s) {
  typedef typename cplx<T>::t C;
  const size_t lds = acc_bytes(a, sizeof(C));
  return dispatch<T, PNH_D>(a.J, layout_of<PNH_D>(a), [&](auto jm, auto jl, auto ex, auto cp, auto pad) {
    auto kern = real_k2y_kernel<T, PNH_D, decltype(jm)::value, decltype(jl)::value,
                                decltype(ex)::value, decltype(cp)::value, decltype(pad)::value>;
    allow_lds(kern, lds);
    hipLaunchKernelGGL(kern, dim3((unsigned)a.n_items), dim3(a.k2y_threads), lds, s, a, grid, y,
                       skip);
    PNH_LAUNCH_CHECK();
    return 0;
  });
}

#if PNH_F64
template <bool STEP>
int launch_gather_cg(const RealArgs& a, const void* slots, const RealCg& cg, const int* skip,
                     hipStream_t s) {
  const int parts = pnh_real_gather_parts(a, PNH_D);
  hipLaunchKernelGGL((real_gather_cg_kernel<PNH_D, STEP>), dim3((unsigned)(a.n_tiles * parts)),
                     dim3(kGatherThreads), 0, s, a, parts, slots, cg, skip);
  PNH_LAUNCH_CHECK();
  return 0;
}
#endif

template <typename T>
int launch_y2k(const RealArgs& a, const void* y, void* grid, void* part_, const int* skip,
               hipStream_t s, const RealCg* cg = nullptr) {
  typedef typename cplx<T>::t C;
  char* part = (char*)part_;
  int* item_e = nullptr;
  void* ys = nullptr;
  const int cl0 = pnh_real_coils(sizeof(T) == 8, a, a.nb);   // coils of the first pass
  if (exponent_pass(sizeof(T) == 8, a, cl0)) {
    item_e = (int*)part;
    part += pnh_item_exponent_bytes(a.n_items * cl0);
    ys = part;
    part += ((size_t)a.M * cl0 * sizeof(C) + 255) & ~(size_t)255;
  }
  if (a.n_items > 0) {
    if (item_e) {
      hipLaunchKernelGGL((real_exponent_kernel<T, PNH_D>), dim3((unsigned)a.n_items), dim3(256),
                         0, s, a, y, item_e, ys, skip);
      PNH_LAUNCH_CHECK();
    }
    const size_t lds = acc_bytes(a, sizeof(C)) + kScratchBytes;
    const int rc = dispatch<T, PNH_D>(a.J, layout_of<PNH_D>(a), [&](auto jm, auto jl, auto ex, auto cp, auto pad) {
      auto kern = real_y2k_kernel<T, PNH_D, decltype(jm)::value, decltype(jl)::value,
                                  decltype(ex)::value, decltype(cp)::value, decltype(pad)::value>;
      allow_lds(kern, lds);
      hipLaunchKernelGGL(kern, dim3((unsigned)a.n_items), dim3(a.threads), lds, s, a, y, part,
                         item_e, ys, skip);
      PNH_LAUNCH_CHECK();
      return 0;
    });
    if (rc) return rc;
  }
#if PNH_F64
  if (cg) return launch_gather_cg<false>(a, part, *cg, skip, s);
#else
  (void)cg;
#endif
  return launch_gather<T>(a, part, grid, skip, s);
}

// LDS of P^H P: box and accumulator of their own while several workgroups
// still share a CU, else in turn.
template <typename C>
size_t php_lds(size_t cells, int& sep) {
  const size_t one = cells * sizeof(C);
  sep = 2 * one <= 40960;
  return one * (sep ? 2 : 1) + kScratchBytes;
}

// LDS of the one-pass complex128 P^H P.
size_t php1_lds(size_t cells) { return cells * 32 + kScratchBytes; }

bool php1_ok(const RealArgs& a) {
  return a.cl == 1 && a.row_bound > 0.0 && php1_lds((size_t)a.pad_cells) <= pnh_lds_limit();
}

#if PNH_F64
int launch_php1(const RealArgs& a, const void* k, void* part, void* pq, const int* skip,
                hipStream_t s) {
  const size_t lds = php1_lds((size_t)a.pad_cells);
  return dispatch<double, PNH_D>(a.J, layout_of<PNH_D>(a), [&](auto jm, auto jl, auto ex, auto cp, auto pad) {
    auto kern = real_php1_kernel<PNH_D, decltype(jm)::value, decltype(jl)::value,
                                 decltype(ex)::value, decltype(cp)::value, decltype(pad)::value>;
    allow_lds(kern, lds);
    hipLaunchKernelGGL(kern, dim3((unsigned)a.n_items), dim3(a.threads), lds, s, a, k, part,
                       (double2*)pq, skip);
    PNH_LAUNCH_CHECK();
    return 0;
  });
}
#endif

template <typename T>
int launch_php(const RealArgs& a, const void* k, void* y, void* grid, void* part,
               const int* skip, hipStream_t s) {
  typedef typename cplx<T>::t C;
#if PNH_F64
  if (a.n_items > 0 && php1_ok(a)) {
    const int rc = launch_php1(a, k, part, nullptr, skip, s);
    return rc ? rc : launch_gather<T>(a, part, grid, skip, s);
  }
#endif
  if (a.n_items > 0) {
    int sep;
    const size_t lds = php_lds<C>((size_t)a.pad_cells * a.cl, sep);
    const int rc = dispatch<T, PNH_D>(a.J, layout_of<PNH_D>(a), [&](auto jm, auto jl, auto ex, auto cp, auto pad) {
      auto kern = real_php_kernel<T, PNH_D, decltype(jm)::value, decltype(jl)::value,
                                  decltype(ex)::value, decltype(cp)::value, decltype(pad)::value>;
      allow_lds(kern, lds);
      hipLaunchKernelGGL(kern, dim3((unsigned)a.n_items), dim3(a.threads), lds, s, a, sep, k, y,
                         part, skip);
      PNH_LAUNCH_CHECK();
      return 0;
    });
    if (rc) return rc;
  }
  return launch_gather<T>(a, part, grid, skip, s);
}

}  // namespace

#define PNH_NAME4(n, x, b) n##_##x##d_f##b
#define PNH_NAME3(n, x, b) PNH_NAME4(n, x, b)
#if PNH_F64
typedef double Real;
#define PNH_NAME(n) PNH_NAME3(n, PNH_D, 64)
#else
typedef float Real;
#define PNH_NAME(n) PNH_NAME3(n, PNH_D, 32)
#endif

int PNH_NAME(pnh_real_k2y)(const RealArgs& a, const void* grid, void* y, const int* skip,
                           hipStream_t s) {
  if (a.n_items == 0) return 0;
  if (!threads_ok(a.k2y_threads)) return -1;
  return launch_k2y<Real>(a, grid, y, skip, s);
}

int PNH_NAME(pnh_real_y2k)(const RealArgs& a, const void* y, void* grid, void* part,
                           const int* skip, hipStream_t s) {
  if (!threads_ok(a.threads)) return -1;
  return launch_y2k<Real>(a, y, grid, part, skip, s);
}

int PNH_NAME(pnh_real_php)(const RealArgs& a, const void* k, void* y, void* grid, void* part,
                           const int* skip, hipStream_t s) {
  if (!threads_ok(a.threads)) return -1;
  return launch_php<Real>(a, k, y, grid, part, skip, s);
}

#if PNH_F64
template <bool STEP>
static int batch_gather_cg(const BatchProblem* probs, const BatchTable& gather, const void* part,
                           const RealBatchCg& cg, const int* done, hipStream_t s) {
  if (gather.n_blocks == 0) return 0;
  hipLaunchKernelGGL((real_gather_cg_batch_kernel<PNH_D, STEP>), dim3((unsigned)gather.n_blocks),
                     dim3(kGatherThreads), 0, s, probs, gather, part, cg.x, cg.r, cg.p, cg.pq,
                     cg.rho, cg.rr, done);
  PNH_LAUNCH_CHECK();
  return 0;
}
#endif

int PNH_NAME(pnh_real_batch_y2k)(const int* J, int layout, const BatchProblem* probs,
                                 const int2* items, int64_t n_items, const BatchTable& gather,
                                 int64_t pad_cells, int threads, const void* y, void* k,
                                 void* part, const int* done, const int* all_done,
                                 const RealBatchCg* cg, hipStream_t s) {
  typedef cplx<Real>::t C;
  const size_t lds = (size_t)pad_cells * sizeof(C) + kScratchBytes;
  if (n_items > 0) {
    const int rc = dispatch<Real, PNH_D>(J, layout, [&](auto jm, auto jl, auto ex, auto cp, auto pad) {
      auto kern = real_y2k_batch_kernel<Real, PNH_D, decltype(jm)::value, decltype(jl)::value,
                                        decltype(ex)::value, decltype(cp)::value, decltype(pad)::value>;
      allow_lds(kern, lds);
      hipLaunchKernelGGL(kern, dim3((unsigned)n_items), dim3(threads), lds, s, probs, items, y,
                         part, done, all_done);
      PNH_LAUNCH_CHECK();
      return 0;
    });
    if (rc) return rc;
  }
#if PNH_F64
  if (cg) return batch_gather_cg<false>(probs, gather, part, *cg, done, s);
#else
  (void)cg;
#endif
  if (gather.n_blocks > 0) {
    hipLaunchKernelGGL((real_gather_batch_kernel<Real, PNH_D>), dim3((unsigned)gather.n_blocks),
                       dim3(256), 0, s, probs, gather, part, k, done, all_done);
    PNH_LAUNCH_CHECK();
  }
  return 0;
}

#if PNH_F64
int PNH_NAME(pnh_real_y2k_cg)(const RealArgs& a, const void* y, void* part, const RealCg& cg,
                              hipStream_t s) {
  if (!threads_ok(a.threads)) return -1;
  return launch_y2k<double>(a, y, nullptr, part, nullptr, s, &cg);
}

int PNH_NAME(pnh_real_php_cg)(const RealArgs& a, void* part, const RealCg& cg, const int* skip,
                              hipStream_t s) {
  if (!threads_ok(a.threads)) return -1;
  const int rc = launch_php1(a, cg.p, part, (void*)cg.pq, skip, s);
  return rc ? rc : launch_gather_cg<true>(a, part, cg, skip, s);
}

int PNH_NAME(pnh_real_batch_php)(const int* J, int layout, int bounds, const BatchProblem* probs,
                                 const int2* items, int64_t n_items, const BatchTable& gather,
                                 int64_t pad_cells, int threads, const void* k, void* ybuf,
                                 void* k_out, void* part, const int* done, const int* all_done,
                                 const RealBatchCg* cg, hipStream_t s) {
  int sep = 1;
  size_t lds = php1_lds((size_t)pad_cells);
  const bool one = bounds && lds <= pnh_lds_limit();
  if (!one) lds = php_lds<double2>((size_t)pad_cells, sep);
  if (n_items > 0) {
    const int rc = dispatch<double, PNH_D>(J, layout, [&](auto jm, auto jl, auto ex, auto cp, auto pad) {
      auto go = [&](auto kern) {
        allow_lds(kern, lds);
        hipLaunchKernelGGL(kern, dim3((unsigned)n_items), dim3(threads), lds, s, probs, items, sep,
                           k, ybuf, part, cg ? cg->pq : nullptr, done, all_done);
        PNH_LAUNCH_CHECK();
        return 0;
      };
      constexpr int jmv = decltype(jm)::value, jlv = decltype(jl)::value;
      constexpr bool exv = decltype(ex)::value;
      constexpr int cpv = decltype(cp)::value, padv = decltype(pad)::value;
      if (one) return go(real_php_batch_kernel<PNH_D, jmv, jlv, exv, cpv, padv, true>);
      return go(real_php_batch_kernel<PNH_D, jmv, jlv, exv, cpv, padv, false>);
    });
    if (rc) return rc;
  }
  if (cg) return batch_gather_cg<true>(probs, gather, part, *cg, done, s);
  if (gather.n_blocks > 0) {
    hipLaunchKernelGGL((real_gather_batch_kernel<double, PNH_D>),
                       dim3((unsigned)gather.n_blocks), dim3(256), 0, s, probs, gather, part,
                       k_out, done, all_done);
    PNH_LAUNCH_CHECK();
  }
  return 0;
}
#else
int PNH_NAME(pnh_real_bounds)(const RealArgs& a, double* bound, hipStream_t s) {
  if (a.n_items == 0) return 0;
  const size_t lds = (size_t)a.pad_cells * 8;
  auto kern = real_bound_kernel<PNH_D>;
  allow_lds(kern, lds);
  hipLaunchKernelGGL(kern, dim3((unsigned)a.n_items), dim3(256), lds, s, a, bound);
  PNH_LAUNCH_CHECK();
  return 0;
}

int PNH_NAME(pnh_real_batch_k2y)(const int* J, int layout, const BatchProblem* probs,
                                 const int2* items, int64_t n_items, int64_t pad_cells,
                                 int threads, const void* k, void* y, const int* done,
                                 const int* all_done, hipStream_t s) {
  if (n_items == 0) return 0;
  const size_t lds = (size_t)pad_cells * 8;
  return dispatch<float, PNH_D>(J, layout, [&](auto jm, auto jl, auto ex, auto cp, auto pad) {
    auto kern = real_k2y_batch_kernel<float, PNH_D, decltype(jm)::value, decltype(jl)::value,
                                      decltype(ex)::value, decltype(cp)::value, decltype(pad)::value>;
    allow_lds(kern, lds);
    hipLaunchKernelGGL(kern, dim3((unsigned)n_items), dim3(threads), lds, s, probs, items, k, y,
                       done, all_done);
    PNH_LAUNCH_CHECK();
    return 0;
  });
}
#endif

#if PNH_D == 1 && !PNH_F64
// The dimension-independent entry points.
#define PNH_DECL(x, b)                                                                          \
  int pnh_real_k2y_##x##d_f##b(const RealArgs&, const void*, void*, const int*, hipStream_t);    \
  int pnh_real_y2k_##x##d_f##b(const RealArgs&, const void*, void*, void*, const int*,          \
                               hipStream_t);                                                    \
  int pnh_real_php_##x##d_f##b(const RealArgs&, const void*, void*, void*, void*, const int*,   \
                               hipStream_t);                                                    \
  int pnh_real_batch_y2k_##x##d_f##b(const int*, int, const BatchProblem*, const int2*,         \
                                     int64_t, const BatchTable&, int64_t, int, const void*,     \
                                     void*, void*, const int*, const int*,                      \
                                     const RealBatchCg*, hipStream_t);
#define PNH_DECL1(x)                                                                            \
  PNH_DECL(x, 32)                                                                               \
  PNH_DECL(x, 64)                                                                               \
  int pnh_real_bounds_##x##d_f32(const RealArgs&, double*, hipStream_t);                        \
  int pnh_real_batch_k2y_##x##d_f32(const int*, int, const BatchProblem*, const int2*, int64_t, \
                                    int64_t, int, const void*, void*, const int*, const int*,   \
                                    hipStream_t);                                               \
  int pnh_real_batch_php_##x##d_f64(const int*, int, int, const BatchProblem*, const int2*,     \
                                    int64_t, const BatchTable&, int64_t, int, const void*,      \
                                    void*, void*, void*, const int*, const int*,                \
                                    const RealBatchCg*, hipStream_t);                           \
  int pnh_real_y2k_cg_##x##d_f64(const RealArgs&, const void*, void*, const RealCg&,            \
                                 hipStream_t);                                                  \
  int pnh_real_php_cg_##x##d_f64(const RealArgs&, void*, const RealCg&, const int*, hipStream_t);
PNH_DECL1(1) PNH_DECL1(2) PNH_DECL1(3)
#undef PNH_DECL1
#undef PNH_DECL

// Up to eight complex64 or four (one, two or four) complex128 coils, as many
// as the box or accumulator leaves room for.
int pnh_real_coils(int fp64, const RealArgs& a, int left) {
  const size_t cell = fp64 ? 16 : 8, lim = pnh_lds_limit();
  int c;
  if (fp64) {
    c = left >= 4 ? 4 : (left >= 2 ? 2 : 1);
  } else {
    const int passes = (left + kMaxCl - 1) / kMaxCl;
    c = (left + passes - 1) / passes;
  }
  while (c > 1 && (size_t)a.pad_cells * c * cell + kScratchBytes > lim) c = fp64 ? c / 2 : c - 1;
  return c;
}

size_t pnh_real_part_bytes(int fp64, const RealArgs& a, int64_t n_slots) {
  const size_t esz = fp64 ? 16 : 8;
  const size_t cl = pnh_real_coils(fp64, a, a.nb);
  size_t n = 0;
  if (exponent_pass(fp64, a, (int)cl))
    n = pnh_item_exponent_bytes(a.n_items * cl) + (((size_t)a.M * cl * esz + 255) & ~(size_t)255);
  return n + (size_t)n_slots * a.pad_cells * cl * esz;
}

// Coils in passes.
template <typename F>
static int coil_passes(int fp64, const RealArgs& a0, F&& f) {
  RealArgs a = a0;
  for (int c0 = 0; c0 < a.nb; c0 += a.cl) {
    a.c0 = c0;
    a.cl = pnh_real_coils(fp64, a0, a.nb - c0);
    const int rc = f(a);
    if (rc) return rc;
  }
  return 0;
}

#define PNH_D_F(fn, b, ...)                                                                     \
  (D == 1 ? fn##_1d_f##b(__VA_ARGS__)                                                           \
          : (D == 2 ? fn##_2d_f##b(__VA_ARGS__) : fn##_3d_f##b(__VA_ARGS__)))
#define PNH_BY_D(fn, ...) (fp64 ? PNH_D_F(fn, 64, __VA_ARGS__) : PNH_D_F(fn, 32, __VA_ARGS__))

int pnh_real_k2y(int D, int fp64, const RealArgs& a, const void* grid, void* y, const int* skip,
                 hipStream_t s) {
  return coil_passes(fp64, a, [&](const RealArgs& p) {
    return PNH_BY_D(pnh_real_k2y, p, grid, y, skip, s);
  });
}

int pnh_real_y2k(int D, int fp64, const RealArgs& a, const void* y, void* grid, void* part,
                 const int* skip, hipStream_t s) {
  return coil_passes(fp64, a, [&](const RealArgs& p) {
    return PNH_BY_D(pnh_real_y2k, p, y, grid, part, skip, s);
  });
}

int pnh_real_php(int D, int fp64, const RealArgs& a, const void* k, void* y, void* grid,
                 void* part, const int* skip, hipStream_t s) {
  return coil_passes(fp64, a, [&](const RealArgs& p) {
    return PNH_BY_D(pnh_real_php, p, k, y, grid, part, skip, s);
  });
}

int pnh_real_item_bounds(int D, const RealArgs& a, double* bound, hipStream_t s) {
  return PNH_D_F(pnh_real_bounds, 32, a, bound, s);
}

int pnh_real_batch_k2y(int D, const int* J, int layout, const BatchProblem* probs,
                       const int2* items, int64_t n_items, int64_t pad_cells, int threads,
                       const void* k, void* y, const int* done, const int* all_done,
                       hipStream_t s) {
  return PNH_D_F(pnh_real_batch_k2y, 32, J, layout, probs, items, n_items, pad_cells, threads, k, y,
                  done, all_done, s);
}

int pnh_real_batch_y2k(int D, int fp64, const int* J, int layout, const BatchProblem* probs,
                       const int2* items, int64_t n_items, const BatchTable& gather,
                       int64_t pad_cells, int threads, const void* y, void* k, void* part,
                       const int* done, const int* all_done, const RealBatchCg* cg,
                       hipStream_t s) {
  return PNH_BY_D(pnh_real_batch_y2k, J, layout, probs, items, n_items, gather, pad_cells,
                  threads, y, k, part, done, all_done, cg, s);
}

int pnh_real_batch_php(int D, const int* J, int layout, int bounds, const BatchProblem* probs,
                       const int2* items, int64_t n_items, const BatchTable& gather,
                       int64_t pad_cells, int threads, const void* k, void* ybuf, void* k_out,
                       void* part, const int* done, const int* all_done, const RealBatchCg* cg,
                       hipStream_t s) {
  return PNH_D_F(pnh_real_batch_php, 64, J, layout, bounds, probs, items, n_items, gather,
                  pad_cells, threads, k, ybuf, k_out, part, done, all_done, cg, s);
}

int64_t pnh_real_cg_blocks(int D, const RealArgs& a0) {
  RealArgs a = a0;
  a.cl = 1;
  if (!a.rec || a.nb != 1 || a.n_items == 0 || !(a.row_bound > 0.0)) return 0;
  if ((size_t)a.pad_cells * 32 + kScratchBytes > pnh_lds_limit()) return 0;
  const int64_t n = a.n_tiles * pnh_real_gather_parts(a, D);
  return n <= 4096 && a.n_items <= 4096 ? n : 0;
}

int pnh_real_y2k_cg(int D, const RealArgs& a0, const void* y, void* part, const RealCg& cg,
                    hipStream_t s) {
  RealArgs a = a0;
  a.c0 = 0;
  a.cl = 1;
  return PNH_D_F(pnh_real_y2k_cg, 64, a, y, part, cg, s);
}

int pnh_real_php_cg(int D, const RealArgs& a0, void* part, const RealCg& cg, const int* skip,
                    hipStream_t s) {
  RealArgs a = a0;
  a.c0 = 0;
  a.cl = 1;
  return PNH_D_F(pnh_real_php_cg, 64, a, part, cg, skip, s);
}
#endif
