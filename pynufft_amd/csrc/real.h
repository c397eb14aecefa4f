// Interpolation and gridding with real factors: argument blocks and host
// entry points (kernels in real.hip).
//
// The min-max factor of sample m along an axis of N image and K grid points is
//   u_j = c_j e^{i om / 2} e^{i pi (N - 1) (b + j) / K},   c_j real,
// b + j the support cell counted without wrapping.  With the grid multiplied
// by mod[t] = e^{i pi (N - 1) t / K} along every axis (the modulated grid, which
// the FFT passes write and read at no cost) the interpolator is real up to
// one phase per sample: two multiply-adds per support cell in place of four,
// half the factor bytes, and P^H P needs no phase at all.  Crossing the grid
// edge multiplies mod by e^{i pi (N - 1)}: for even N the sign flips.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "common.h"

struct RealArgs {
  int nb;                      // coils sharing the trajectory
  int c0, cl;                  // first coil and coils of this pass
  int K[PNH_MAXD], J[PNH_MAXD];
  int tile[PNH_MAXD], tgrid[PNH_MAXD], pad[PNH_MAXD];
  int flip[PNH_MAXD];          // 1: mod changes sign across the grid edge
  int pad_cells;               // prod(pad)
  int max_tile_slots;
  int64_t M, n_items, n_tiles;
  // row records, rw elements apart (element type of the operator): c_0[J_0],
  // c_1[J_1], c_2[J_2], then for complex64: phase re, im, x_0 | x_1 << 16
  // (first cell in the tile), x_2 (3-D), the sample index; for complex128:
  // x_0 | x_1 << 16 | x_2 << 32 (phase and sample index from ph, perm)
  const void* rec;
  int rw;
  const void* ph;              // complex128: [M] phase
  const int* perm;             // [M] row -> sample
  const int* items;            // [n_items][4] tile id, first row, rows, slot
  const int* tile_slots;       // [n_tiles][2] first slot, slot count
  const double* item_bound;    // complex64: per item, bound of a cell's sum of |coef|
  double u_bound;              // bound of |coef|
  double row_bound;            // bound of a row's sum of |coef|, or 0
  const void* mod[PNH_MAXD];   // e^{i pi (N_d - 1) t / K_d}, t < K_d
  int stage;                   // 1: the grid given or wanted is the plain one
  int threads, k2y_threads;    // workgroup sizes of gridding and interpolation
};

// Gather workgroups of 256 elements (cell, coil) per tile.
__host__ __device__ inline int pnh_real_gather_parts(const RealArgs& a, int D) {
  int64_t cells = a.cl;
  for (int d = 0; d < D; ++d) cells *= a.tile[d];
  return (int)((cells + 255) / 256);
}

// y = P k
int pnh_real_k2y(int D, int fp64, const RealArgs& a, const void* grid, void* y, const int* skip,
                 hipStream_t s);
// k = P^H y; part as pnh_real_part_bytes
int pnh_real_y2k(int D, int fp64, const RealArgs& a, const void* y, void* grid, void* part,
                 const int* skip, hipStream_t s);
// k_out = P^H P k (k_out may alias k); y: scratch of M * nb elements
int pnh_real_php(int D, int fp64, const RealArgs& a, const void* k, void* y, void* grid,
                 void* part, const int* skip, hipStream_t s);
// Gridding scratch: item exponents, row-ordered samples, partial slots.
size_t pnh_real_part_bytes(int fp64, const RealArgs& a, int64_t n_slots);
// Per-item bounds from the complex64 records.
int pnh_real_item_bounds(int D, const RealArgs& a, double* bound, hipStream_t s);
// Coils of a gridding or interpolation pass when `left` remain.
int pnh_real_coils(int fp64, const RealArgs& a, int left);

// The gridding as a step of the conjugate gradients (complex128, one coil; x,
// r, p: grids): the gather updates x and r where it would have stored the grid,
// and <p, P^H P p> is the sum of |P p|^2 that P^H P leaves per item, so no
// vector is read again for a product.
struct RealCg {
  void* x;
  void* r;
  const void* p;
  const void* pq;              // [n_items] double2, real: sums of |P p|^2
  int n_pq;
  void* rr;                    // [blocks] double2, real: sums of |r|^2
  const double* rho;           // |r|^2 before the step
};
// Gather workgroups (rr's length), or 0: not these plans (no row bound, a box
// too large for the one-pass P^H P, or more partial sums, over 4096, than
// every workgroup should add up itself).
int64_t pnh_real_cg_blocks(int D, const RealArgs& a);
// r = P^H y, x = 0
int pnh_real_y2k_cg(int D, const RealArgs& a, const void* y, void* part, const RealCg& cg,
                    hipStream_t s);
// alpha = rho / sum(pq); x += alpha p, r -= alpha P^H P p
int pnh_real_php_cg(int D, const RealArgs& a, void* part, const RealCg& cg, const int* skip,
                    hipStream_t s);
