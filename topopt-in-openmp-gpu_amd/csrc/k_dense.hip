// Dense FP64 direct solver of the coarsest level (replaces CHOLMOD,
// stencil_assembly.c:366-503).
//
// The coarsest matrix (n = 3 * interior nodes, 4131 at 16x8x8 elements) is
// block tridiagonal over the grid's x-planes (3 ny nz DOFs each, x slowest).
// Per design iteration:
//   1. Cholesky P A P^T = L L^T over 64x64 tiles, with the planes in
//      nested-dissection order (odd-even reduction of the plane chain, each
//      plane padded to whole tiles): every launch eliminates one tile column
//      of every plane of the current independent set, so a 17-plane chain
//      takes 5 levels x 4 columns (+1) launches instead of the 65 of the
//      banded order.  Each workgroup owns one target tile of the update,
//      forms the panel tiles Q = A_XK L_KK^{-T} it needs on FP64 MFMA
//      (v_mfma_f64_16x16x4f64) and applies C_IJ -= sum_K Q_IK Q_JK^T; the
//      workgroup of a diagonal tile eliminated next factors it in LDS right
//      after its update (Cholesky, then the inverse of the 64x64 factor);
//   2. W = L^{-1} (lower triangle, zero outside the reach of each column) by
//      16-column strips and levels of the dissection, beside the Cholesky
//      launches of the next level; W^T is written alongside.
// A V-cycle applies A^{-1} = P^T W^T W P as two triangular GEMVs.
#include <algorithm>

#include "t3d_internal.hpp"

namespace t3d {

constexpr int kNB = kTile;      // tile size
// LDS row stride of a 64x64 tile: rows 16-byte aligned, and the pairs of an MFMA
// operand in distinct banks
constexpr int kLd = kNB + 2;
constexpr int kStrip = 16;      // columns per workgroup of the W = L^{-1} kernel
constexpr int kTriBatch = 64;   // tiles per batch of loads of the triangular products

typedef double double4_t __attribute__((ext_vector_type(4)));

// MFMA operand layout (v_mfma_f64_16x16x4f64, measured on gfx950): lane l
// feeds A[l%16][l/16] and B[l/16][l%16]; accumulator register v of lane l
// holds D[l/16 + 4v][l%16].
__device__ inline double4_t mfma4(double a, double b, double4_t c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// ---------------------------------------------------------------------------
// Cholesky and inverse of one 64x64 SPD tile in LDS, 8 waves (6 of them at work),
// blocked by 16.  The 64 pivots are a serial chain, and a wave alone on its
// SIMD issues one FP64 instruction in about 8 cycles, so the chain costs the
// instructions of one wave.  Wave 0 does nothing else: it holds a 64x16 panel
// in registers, the diagonal block's rows in each of its four rows of 16
// lanes (so that pivot and multipliers are broadcast by DPP) and beside them
// the rows below.  Per panel the 16 columns of the next panel are then updated
// on MFMA by waves 0-2; while wave 0 factors the next panel, waves 1-3 update
// the rest of the trailing triangle and wave 5, on another SIMD than wave 0,
// inverts the finished diagonal block.  The off-diagonal 16x16 blocks of the
// inverse follow on MFMA.  A tile takes 23,000 cycles (10 us), 19,000 of them
// the four panels; with the 16x16 diagonal blocks factored on their own, each
// pivot column sent through LDS, and panel, trailing triangle and inverses
// between barriers, it took about twice that (a launch of one task 33 us
// against 23, and 18 with eight waves for the products before it).
// In: T (lower triangle, as 16x16 blocks; rows/cols beyond the matrix padded
// with identity), X = 0.  Out: T = L (above the diagonal undefined),
// X = L^{-1}.  A non-positive pivot sets *info (and is replaced by 1 so that
// the factorization finishes).

// two neighbouring values in LDS (16-byte aligned)
__device__ __forceinline__ void pair_load(const double *p, double &a, double &b) {
  const double2 v = *reinterpret_cast<const double2 *>(p);
  a = v.x;
  b = v.y;
}
__device__ __forceinline__ void pair_store(double *p, double a, double b) {
  *reinterpret_cast<double2 *>(p) = double2{a, b};
}

// Workgroup barrier for LDS: the wave's LDS accesses complete (lgkmcnt 0; the
// other counters left at their maxima), then s_barrier.  __syncthreads() also
// waits for the wave's global loads and stores.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_s_waitcnt(0xC07F);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// 1/sqrt(x) for x > 0: the hardware estimate and two Newton steps
// y <- y + y (1/2 - (x / 2) y^2)
__device__ inline double rsqrt_refined(double x) {
  double y = __builtin_amdgcn_rsq(x);
  const double xh = 0.5 * x;
#pragma unroll
  for (int it = 0; it < 2; it++) y = fma(y, fma(-xh * y, y, 0.5), y);
  return y;
}

// FP64 instructions with one operand from another lane of the row of 16 lanes
// (DPP row_newbcast), which saves the two v_readlane per broadcast value.
// s_nop 1: a VGPR may be read through DPP two wait states after it was
// written.
template <int N>
__device__ __forceinline__ double row_bcast(double x) {  // lane N's x
  double r;
  asm("s_nop 1\n\tv_mov_b64_dpp %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf"
      : "=v"(r)
      : "v"(x), "n"(N));
  return r;
}
// a[c] -= (lane c's x) m, c = C..15
template <int C>
__device__ __forceinline__ void row_update(double (&a)[16], double x, double m) {
  if constexpr (C + 3 < 16) {
    asm("s_nop 1\n\t"
        "v_fmac_f64_dpp %0, %4, -%5 row_newbcast:%6 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %1, %4, -%5 row_newbcast:%7 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %2, %4, -%5 row_newbcast:%8 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %3, %4, -%5 row_newbcast:%9 row_mask:0xf bank_mask:0xf"
        : "+v"(a[C]), "+v"(a[C + 1]), "+v"(a[C + 2]), "+v"(a[C + 3])
        : "v"(x), "v"(m), "n"(C), "n"(C + 1), "n"(C + 2), "n"(C + 3));
    row_update<C + 4>(a, x, m);
  } else if constexpr (C < 16) {
    asm("s_nop 1\n\tv_fmac_f64_dpp %0, %1, -%2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
        : "+v"(a[C])
        : "v"(x), "v"(m), "n"(C));
    row_update<C + 1>(a, x, m);
  }
}
// x[q] -= (lane M's x[q]) m
template <int M>
__device__ __forceinline__ void row_eliminate(double (&x)[4], double m) {
  asm("s_nop 1\n\t"
      "v_fmac_f64_dpp %0, %0, -%4 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %1, -%4 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %2, %2, -%4 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %3, %3, -%4 row_newbcast:%5 row_mask:0xf bank_mask:0xf"
      : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3])
      : "v"(m), "n"(M));
}

// Pivot J of a panel and those after it: u the diagonal block's rows (the
// same in each row of 16 lanes), v the lane's row below it, ij[j] = 1 / L_jj.
template <int J, bool V>
__device__ __forceinline__ void panel_pivots(double (&u)[16], double (&v)[16], double (&ij)[16],
                                             bool &bad) {
  if constexpr (J < 16) {
    double piv = row_bcast<J>(u[J]);
    const bool ok = piv > 0.0;
    bad = bad || !ok;
    piv = ok ? piv : 1.0;
    ij[J] = rsqrt_refined(piv);
    u[J] *= ij[J];
    row_update<J + 1>(u, u[J], u[J]);
    if constexpr (V) {
      v[J] *= ij[J];
      row_update<J + 1>(v, u[J], v[J]);
    }
    panel_pivots<J + 1, V>(u, v, ij, bad);
  }
}

// Elimination step M of the inverse of a 16x16 factor: u its rows, ij the
// reciprocals of its diagonal, x four columns of the inverse (times its
// row's diagonal), r the lane's row.
template <int M>
__device__ __forceinline__ void inverse_steps(const double (&u)[16], const double (&ij)[16],
                                              double (&x)[4], int r) {
  if constexpr (M < 15) {
    row_eliminate<M>(x, r > M ? u[M] * ij[M] : 0.0);
    inverse_steps<M + 1>(u, ij, x, r);
  }
}

// X block b = inverse of the diagonal block b of L, by one wave: lane l has
// row l % 16 and the columns 4 (l / 16) + q of the inverse.
__device__ __forceinline__ void invert_block(double *X, int b, const double (&u)[16],
                                             const double (&ij)[16], int lane) {
  const int r = lane & 15, g = lane >> 4;
  double x[4], s = 0.0;
#pragma unroll
  for (int q = 0; q < 4; q++) x[q] = r == 4 * g + q ? 1.0 : 0.0;
  inverse_steps<0>(u, ij, x, r);
#pragma unroll
  for (int i = 0; i < 16; i++) s = r == i ? ij[i] : s;
#pragma unroll
  for (int q = 0; q < 4; q++) X[(16 * b + r) * kLd + 16 * b + 4 * g + q] = x[q] * s;
}

// Columns [16 kb, 16 kb + 16) of the factor by one wave: u the diagonal
// block, v the rows below (lane l: row l % 16 of the blocks kb and
// kb + 1 + l / 16); LAST: the last block, whose inverse follows at once.
template <bool LAST>
__device__ __forceinline__ void factor_panel(double *T, double *X, double *inv, int kb, int lane,
                                             int *info) {
  const int r = lane & 15, g = lane >> 4, d0 = 16 * kb;
  const int vrow = 16 * min(kb + 1 + g, 3) + r;
  double u[16], v[16], ij[16];
  bool bad = false;
#pragma unroll
  for (int c = 0; c < 16; c += 2) {
    pair_load(T + (d0 + r) * kLd + d0 + c, u[c], u[c + 1]);
    if constexpr (!LAST) pair_load(T + vrow * kLd + d0 + c, v[c], v[c + 1]);
  }
  panel_pivots<0, !LAST>(u, v, ij, bad);
  if (bad && lane == 0) info[0] = 1;
  if constexpr (LAST) {
    invert_block(X, kb, u, ij, lane);
  } else {
    if (g == 0) {
#pragma unroll
      for (int c = 0; c < 16; c += 2) {
        pair_store(T + (d0 + r) * kLd + d0 + c, u[c], u[c + 1]);
        pair_store(inv + d0 + c, ij[c], ij[c + 1]);  // (16 lanes write the same values)
      }
    }
    if (kb + 1 + g < 4) {
#pragma unroll
      for (int c = 0; c < 16; c += 2) pair_store(T + vrow * kLd + d0 + c, v[c], v[c + 1]);
    }
  }
}

// the inverse of a diagonal block from the factor in LDS
__device__ __forceinline__ void invert_block_lds(const double *T, double *X, const double *inv,
                                                 int b, int lane) {
  double u[16], ij[16];
#pragma unroll
  for (int c = 0; c < 16; c += 2) {
    pair_load(T + (16 * b + (lane & 15)) * kLd + 16 * b + c, u[c], u[c + 1]);
    pair_load(inv + 16 * b + c, ij[c], ij[c + 1]);
  }
  invert_block(X, b, u, ij, lane);
}

// Block (ti, tj) of the trailing triangle minus the product of the panel
// columns [d0, d0 + 16) of its rows and columns.
__device__ __forceinline__ void trail_block(double *T, int ti, int tj, int d0, int lane) {
  const int li = lane & 15, lk = lane >> 4;
  double *C = T + (16 * ti + lk) * kLd + 16 * tj + li;
  double4_t acc;
#pragma unroll
  for (int v = 0; v < 4; v++) acc[v] = C[4 * v * kLd];
#pragma unroll
  for (int k = 0; k < 16; k += 4)
    acc = mfma4(-T[(16 * ti + li) * kLd + d0 + k + lk], T[(16 * tj + li) * kLd + d0 + k + lk], acc);
#pragma unroll
  for (int v = 0; v < 4; v++) C[4 * v * kLd] = acc[v];
}

// y += L_IK X_KJ (16x16 blocks)
__device__ __forceinline__ void inv_term(const double *T, const double *X, int I, int K, int J,
                                         int lane, double4_t &y) {
  const int li = lane & 15, lk = lane >> 4;
#pragma unroll
  for (int k = 0; k < 16; k += 4)
    y = mfma4(T[(16 * I + li) * kLd + 16 * K + k + lk], X[(16 * K + k + lk) * kLd + 16 * J + li],
              y);
}
// X_IJ = -X_II y (the accumulator of y is the B operand as it is: register v
// of lane l holds y[l/16 + 4v][l%16], the B element of k-step v)
__device__ __forceinline__ void inv_block(double *X, int I, int J, int lane, const double4_t &y) {
  const int li = lane & 15, lk = lane >> 4;
  double4_t o = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int v = 0; v < 4; v++) o = mfma4(-X[(16 * I + li) * kLd + 16 * I + 4 * v + lk], y[v], o);
#pragma unroll
  for (int v = 0; v < 4; v++) X[(16 * I + lk + 4 * v) * kLd + 16 * J + li] = o[v];
}

// inv: 64 doubles of LDS.  T and X are complete (barrier) on entry and exit.
__device__ __forceinline__ void factor_tile(double *T, double *X, double *inv, int *info) {
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const double4_t zero = {0.0, 0.0, 0.0, 0.0};
  double4_t y30 = zero;
#pragma unroll 1
  for (int kb = 0; kb < 4; kb++) {
    const int d0 = 16 * kb;
    if (w == 0) {
      if (kb < 3) factor_panel<false>(T, X, inv, kb, lane, info);
      else factor_panel<true>(T, X, inv, kb, lane, info);
    } else if (kb > 0 && w < 6) {
      // what the panel before left: its blocks (ti, tj), kb < tj <= ti, and
      // the inverse of its diagonal block
      if (kb == 1 && w < 4) trail_block(T, w == 1 ? 2 : 3, w == 3 ? 3 : 2, d0 - 16, lane);
      if (kb == 2 && w == 1) trail_block(T, 3, 3, d0 - 16, lane);
      if (w == 5) invert_block_lds(T, X, inv, kb - 1, lane);
      if (kb == 3 && w == 1) {
        double4_t y = zero;
        inv_term(T, X, 1, 0, 0, lane, y);
        inv_block(X, 1, 0, lane, y);
      }
      if (kb == 3 && w == 2) inv_term(T, X, 3, 0, 0, lane, y30);
    }
    lds_barrier();
    if (kb < 3) {  // the next panel's columns
      if (w < 3 - kb) trail_block(T, kb + 1 + w, kb + 1, d0, lane);
      lds_barrier();
    }
  }
  // the rest of X: X_10 and the diagonal blocks are there
  double4_t y = zero;
  if (w == 0) {
    inv_term(T, X, 2, 1, 1, lane, y);
    inv_block(X, 2, 1, lane, y);
  } else if (w == 1) {
    inv_term(T, X, 2, 0, 0, lane, y);
    inv_term(T, X, 2, 1, 0, lane, y);
    inv_block(X, 2, 0, lane, y);
  } else if (w == 2) {
    inv_term(T, X, 3, 1, 0, lane, y30);
  } else if (w == 3) {
    inv_term(T, X, 3, 2, 2, lane, y);
    inv_block(X, 3, 2, lane, y);
  }
  lds_barrier();
  if (w == 1) {
    y = zero;
    inv_term(T, X, 3, 1, 1, lane, y);
    inv_term(T, X, 3, 2, 1, lane, y);
    inv_block(X, 3, 1, lane, y);
  } else if (w == 2) {
    inv_term(T, X, 3, 2, 0, lane, y30);
    inv_block(X, 3, 0, lane, y30);
  }
  lds_barrier();
}

// The blocks C0 and C1 of the row block rb of Q = P D^T for 64x64 tiles in LDS, D
// lower triangular (block cb needs k < 16 (cb + 1) only).
template <int C0, int C1>
__device__ __forceinline__ void panel_product(const double *P, const double *D, int rb, int lane,
                                              double4_t (&q)[2]) {
  const int li = lane & 15, lk = lane >> 4;
  q[0] = q[1] = double4_t{0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int k = 0; k < 16 * (C1 + 1); k += 4) {
    const double av = P[(16 * rb + li) * kLd + k + lk];
    if (k < 16 * (C0 + 1)) q[0] = mfma4(av, D[(16 * C0 + li) * kLd + k + lk], q[0]);
    q[1] = mfma4(av, D[(16 * C1 + li) * kLd + k + lk], q[1]);
  }
}

// acc_b -= (row block rb_b of X) (row block cb_b of Y)^T, b < NB
template <int NB>
__device__ __forceinline__ void update_blocks(const double *X, const double *Y,
                                              const int (&rb)[2], const int (&cb)[2], int lane,
                                              double4_t (&acc)[2]) {
  const int li = lane & 15, lk = lane >> 4;
#pragma unroll
  for (int k = 0; k < kNB; k += 4)
#pragma unroll
    for (int b = 0; b < NB; b++)
      acc[b] = mfma4(-X[(16 * rb[b] + li) * kLd + k + lk], Y[(16 * cb[b] + li) * kLd + k + lk],
                     acc[b]);
}

// One task of an elimination step (one workgroup): the trailing tile (I, J),
// I >= J, receives the updates of the tile columns K[0..nsrc) eliminated in
// this step,
//   C_IJ = A_IJ - sum_K Q_IK Q_JK^T,   Q_XK = A_XK L_KK^{-T}
// (each workgroup forms the two panel tiles it needs on MFMA).  C is loaded
// into the accumulators: two 16x16 blocks per wave, or for a diagonal tile, of
// which only the blocks on and below the diagonal are used, one or two of those.
// Eight waves, two to a SIMD: alone on its SIMD a wave reaches half the FP64 MFMA
// rate (a diagonal task's product and update took 13,400 cycles with four waves,
// 9,900 with eight).  The task of a diagonal tile (I, I) also writes
// L_IK = Q_IK.  With kTaskFactor the tile is complete after this update and
// is factored in LDS right away (Cholesky, then the inverse of the 64x64
// factor, which goes to Dinv); nsrc = 0 factors A_II as it is.
// Matrices are np x np row-major, np a multiple of 64.
// Latency bound: a launch takes as long as its longest chain of loads,
// products and one factorization.
__global__ __launch_bounds__(512) void k_chol_task(double *__restrict__ A, double *__restrict__ Lf,
                                                   double *__restrict__ Dinv, int np,
                                                   const CholTask *__restrict__ tasks,
                                                   int *__restrict__ info) {
  __shared__ __align__(16) double PI[kNB * kLd];
  __shared__ __align__(16) double PJ[kNB * kLd];
  __shared__ __align__(16) double DV[kNB * kLd];
  __shared__ __align__(16) double inv[kNB];
  // the elimination is the set-up's critical path: its waves go first where they
  // share a SIMD with those of the rows of W
  __builtin_amdgcn_s_setprio(3);
  const CholTask tk = tasks[blockIdx.x];
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  const int li = lane & 15, lk = lane >> 4;
  const bool diag = tk.I == tk.J, fac = (tk.flags & kTaskFactor) != 0;
  const int64_t gi = (int64_t)tk.I * kNB, gj = (int64_t)tk.J * kNB;
  double *Cg = A + gi * np + gj;
  // the wave's blocks of the target: of a diagonal tile (row, column) blocks
  // (0,0) (1,1) | (1,0) (2,2) | (2,0) | (2,1) | (3,0) | (3,1) | (3,2) | (3,3),
  // else two neighbours of a row
  int rb[2], cb[2];
  const int nb = diag && w >= 2 ? 1 : 2;
  if (diag) {
    rb[0] = w < 2 ? w : w < 4 ? 2 : 3;
    cb[0] = w < 2 ? 0 : w < 4 ? w - 2 : w - 4;
    rb[1] = cb[1] = w + 1;
  } else {
    rb[0] = rb[1] = w >> 1;
    cb[0] = 2 * (w & 1);
    cb[1] = cb[0] + 1;
  }
  if (fac) {
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int e = 2 * tid + 1024 * q;
      pair_store(PJ + (e >> 6) * kLd + (e & 63), 0.0, 0.0);
    }
  }
  double4_t acc[2];
#pragma unroll
  for (int b = 0; b < 2; b++)
    if (b < nb) {
#pragma unroll
      for (int v = 0; v < 4; v++)
        acc[b][v] = Cg[(int64_t)(16 * rb[b] + lk + 4 * v) * np + 16 * cb[b] + li];
    }
  for (int s = 0; s < tk.nsrc; s++) {
    const int64_t gk = (int64_t)tk.K[s] * kNB;
    // stage A_IK, A_JK and L_KK^{-1}; all loads of a thread are issued before
    // its LDS stores
    double2 ri[4], rj[4], rd[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int e = 2 * tid + 1024 * q, r = e >> 6, c = e & 63;
      ri[q] = *reinterpret_cast<const double2 *>(A + (gi + r) * np + gk + c);
      if (!diag) rj[q] = *reinterpret_cast<const double2 *>(A + (gj + r) * np + gk + c);
      rd[q] = *reinterpret_cast<const double2 *>(Dinv + (int64_t)tk.K[s] * kNB * kNB + e);
    }
    lds_barrier();  // the previous source's products are done with the tiles
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int e = 2 * tid + 1024 * q, o = (e >> 6) * kLd + (e & 63);
      pair_store(PI + o, ri[q].x, ri[q].y);
      if (!diag) pair_store(PJ + o, rj[q].x, rj[q].y);
      pair_store(DV + o, rd[q].x, rd[q].y);
    }
    lds_barrier();
    // Q_I = A_IK L_KK^{-T}, Q_J
    double4_t qi[2], qj[2];
    const int pr = w & 3, pc = w < 4 ? 0 : 1;  // blocks (pr, pc) and (pr, 3 - pc)
    if (w < 4) {
      panel_product<0, 3>(PI, DV, pr, lane, qi);
      if (!diag) panel_product<0, 3>(PJ, DV, pr, lane, qj);
    } else {
      panel_product<1, 2>(PI, DV, pr, lane, qi);
      if (!diag) panel_product<1, 2>(PJ, DV, pr, lane, qj);
    }
    lds_barrier();  // the tiles are read: Q takes their place
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int r = 16 * pr + lk + 4 * v, c = 16 * (b ? 3 - pc : pc) + li;
        PI[r * kLd + c] = qi[b][v];
        if (diag) Lf[(gi + r) * np + gk + c] = qi[b][v];
        else PJ[r * kLd + c] = qj[b][v];
      }
    lds_barrier();
    const double *Y = diag ? PI : PJ;
    if (nb == 2) update_blocks<2>(PI, Y, rb, cb, lane, acc);
    else update_blocks<1>(PI, Y, rb, cb, lane, acc);
  }
  if (fac) lds_barrier();  // L_KK^{-1} is done with, X is cleared
#pragma unroll
  for (int b = 0; b < 2; b++)
    if (b < nb) {
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int r = 16 * rb[b] + lk + 4 * v, c = 16 * cb[b] + li;
        if (fac) DV[r * kLd + c] = acc[b][v];
        else Cg[(int64_t)r * np + c] = acc[b][v];
      }
    }
  if (!fac) return;
  lds_barrier();
  factor_tile(DV, PJ, inv, info);
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int e = 2 * tid + 1024 * q;
    double2 x;
    pair_load(PJ + (e >> 6) * kLd + (e & 63), x.x, x.y);
    *reinterpret_cast<double2 *>(Dinv + (int64_t)tk.I * kNB * kNB + e) = x;
  }
}

// ---------------------------------------------------------------------------
// W = L^{-1}, WT = W^T by 16-column strips, level by level of the elimination
// so that only the last level's rows remain when the factorization ends.  A
// strip [16s, 16s+16) of tile column J has W_JJ = L_JJ^{-1} and, in the tile
// rows I of the reach of J,
//   W_I = -L_II^{-1} sum_{K in ks(I)} L_IK W_K,
// ks(I) the strip's earlier rows with L_IK != 0 (lists from the elimination
// schedule).  k_linv_sums leaves the terms of the lower levels in W_I, level by
// level as their rows are there; k_linv_rows adds those of the row's own level
// (at most the tiles of a plane; all of them for a band), row by row, and
// multiplies by L_II^{-1}.  (One launch after the factorization that walked
// all rows of a strip took 270 us at coarse 16x8x8.)  W is always written;
// WT, W32 and WT32 (FP32 copies) when given.
//
// acc += L_IK W_K for the wave's 16 rows (row block rb) of the strip: lane l
// feeds k = 16 (l/16) + q of MFMA step q, so that its part of L_IK is a run of
// 128 bytes; the next term's loads are issued before this one's products.
struct LinvTerm {
  double a[16], b[16];
};
__device__ __forceinline__ void linv_load(const double *__restrict__ Lf, const double *W, int np,
                                          int I, int K, int rb, int gc, LinvTerm &t) {
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const double2 *pa = reinterpret_cast<const double2 *>(
      Lf + ((int64_t)I * kNB + 16 * rb + li) * np + (int64_t)K * kNB + 16 * lk);
  const double *pb = W + ((int64_t)K * kNB + 16 * lk) * np + gc;
#pragma unroll
  for (int q = 0; q < 8; q++) {
    const double2 v = pa[q];
    t.a[2 * q] = v.x;
    t.a[2 * q + 1] = v.y;
  }
#pragma unroll
  for (int q = 0; q < 16; q++) t.b[q] = pb[(int64_t)q * np];
}
__device__ __forceinline__ void linv_product(const LinvTerm &t, double4_t &acc0, double4_t &acc1) {
#pragma unroll
  for (int q = 0; q < 16; q += 2) {
    acc0 = mfma4(t.a[q], t.b[q], acc0);
    acc1 = mfma4(t.a[q + 1], t.b[q + 1], acc1);
  }
}
// the terms ks[t0], ks[t0 + dt], ... below ks[t1]
__device__ __forceinline__ double4_t linv_terms(const double *__restrict__ Lf, const double *W,
                                                int np, int I, const int *__restrict__ ks, int t0,
                                                int t1, int dt, int rb, int gc) {
  double4_t acc0 = {0.0, 0.0, 0.0, 0.0}, acc1 = {0.0, 0.0, 0.0, 0.0};
  LinvTerm cur, nxt;
  if (t0 < t1) linv_load(Lf, W, np, I, ks[t0], rb, gc, cur);
  for (int t = t0; t < t1; t += dt) {
    if (t + dt < t1) linv_load(Lf, W, np, I, ks[t + dt], rb, gc, nxt);
    linv_product(cur, acc0, acc1);
    cur = nxt;
  }
  return acc0 + acc1;
}

// The terms of level `from` in the rows of the levels above it, added to what the
// lower levels left there: blockIdx.x, tile column J; blockIdx.z, the level;
// blockIdx.y, the row of J in it.  A workgroup forms the 64x64 tile, a wave 16
// rows and 32 columns of it: two waves to a SIMD, which the FP64 MFMA rate takes,
// and W_KJ staged once per term in LDS.  (All terms of a row after the level
// below it, by strips of 16 columns with L_IK loaded again for each, took 64 us
// for the last level at coarse 16x8x8; its terms of the level below alone 29.)
__global__ __launch_bounds__(512) void k_linv_sums(const double *__restrict__ Lf, int np,
                                                   const int2 *__restrict__ colinfo,
                                                   const int *__restrict__ tile_level, int from,
                                                   const int4 *__restrict__ rows,
                                                   const int *__restrict__ klist, double *W) {
  constexpr int kLdB = kNB + 1;  // rows 16 apart in the other half of the banks
  __shared__ double Bs[2][kNB * kLdB];
  const int J = blockIdx.x;
  const int2 ci = colinfo[(size_t)(from + 1 + blockIdx.z) * gridDim.x + J];
  if ((int)blockIdx.y >= ci.y) return;
  const int4 rw = rows[ci.x + blockIdx.y];
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, li = lane & 15, lk = lane >> 4;
  const int rb = w & 3, c0 = 32 * (w >> 2) + li;
  // the row's terms are in the order of the levels: those of `from`
  int t0 = 0, t1 = 0;
  for (int q = 0; q < rw.w; q += 64) {
    const int lev = q + lane < rw.w ? tile_level[klist[rw.y + q + lane]] : from + 1;
    t0 += __popcll(__ballot(lev < from));
    t1 += __popcll(__ballot(lev <= from));
  }
  if (t0 == t1) return;
  const int *ks = klist + rw.y;
  // lane l feeds k = 16 (l / 16) + q of MFMA step q: a run of 128 bytes of L_IK
  const double *pa = Lf + ((int64_t)rw.x * kNB + 16 * rb + li) * np + 16 * lk;
  double2 a[8], na[8], nb[4];
  auto load = [&](int K) {
#pragma unroll
    for (int q = 0; q < 8; q++)
      na[q] = reinterpret_cast<const double2 *>(pa + (int64_t)K * kNB)[q];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int e = 2 * tid + 1024 * q;
      nb[q] = *reinterpret_cast<const double2 *>(W + ((int64_t)K * kNB + (e >> 6)) * np +
                                                 (int64_t)J * kNB + (e & 63));
    }
  };
  double4_t acc[2] = {{0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0}};
  load(ks[t0]);
  double *out = W + ((int64_t)rw.x * kNB + 16 * rb + lk) * np + (int64_t)J * kNB + c0;
  if (t0 > 0) {
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
      for (int v = 0; v < 4; v++) acc[b][v] = out[(int64_t)(4 * v) * np + 16 * b];
  }
  for (int t = t0; t < t1; t++) {
    double *B = Bs[t & 1];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int e = 2 * tid + 1024 * q;
      double *b = B + (e >> 6) * kLdB + (e & 63);
      b[0] = nb[q].x;
      b[1] = nb[q].y;
    }
#pragma unroll
    for (int q = 0; q < 8; q++) a[q] = na[q];
    lds_barrier();  // (the buffer before last is read: every wave has passed the last barrier)
    if (t + 1 < t1) load(ks[t + 1]);
#pragma unroll
    for (int q = 0; q < 16; q++) {
      const double av = q & 1 ? a[q / 2].y : a[q / 2].x;
      const double *b = B + (16 * lk + q) * kLdB + c0;
      acc[0] = mfma4(av, b[0], acc[0]);
      acc[1] = mfma4(av, b[16], acc[1]);
    }
  }
#pragma unroll
  for (int b = 0; b < 2; b++)
#pragma unroll
    for (int v = 0; v < 4; v++) out[(int64_t)(4 * v) * np + 16 * b] = acc[b][v];
}

constexpr int kLinvGroups = 2;  // groups of 4 waves, which take alternate terms
// Rows of a column in a level up to which its part of W stays in LDS (a plane's
// tiles).  A row needs the one before it: read back from memory the four of the
// last level took 43 us at coarse 16x8x8, 34 from LDS, with all lists loaded at
// the start and the next row's L meanwhile.
constexpr int kLinvOwn = 4;

__global__ __launch_bounds__(256 * kLinvGroups) void k_linv_rows(
    const double *__restrict__ Lf, const double *__restrict__ Dinv, int np,
    const int2 *__restrict__ colinfo, const int *__restrict__ tile_level, int level,
    const int4 *__restrict__ rows, const int *__restrict__ klist, double *W,
    double *__restrict__ WT, float *__restrict__ W32, float *__restrict__ WT32) {
  __shared__ double Bx[kLinvGroups][kNB * 17];
  __shared__ double Own[kLinvOwn + 1][kNB * 17];  // W_JJ, then the rows
  const int tid = threadIdx.x, grp = tid >> 8, rb = (tid >> 6) & 3, lane = tid & 63;
  const int li = lane & 15, lk = lane >> 4;
  const int c0 = blockIdx.x * kStrip, J = c0 / kNB, cofs = c0 - J * kNB;
  const int gc = c0 + li;
  auto put = [&](int64_t gr, int c, double v) {
    W[gr * np + c] = v;
    if (WT) WT[(int64_t)c * np + gr] = v;
    if (W32) {
      W32[gr * np + c] = (float)v;
      WT32[(int64_t)c * np + gr] = (float)v;
    }
  };
  if (tile_level[J] == level) {
    for (int e = tid; e < kNB * kStrip; e += 256 * kLinvGroups) {
      const int r = e >> 4, j = e & 15;
      const double v = Dinv[(int64_t)J * kNB * kNB + r * kNB + cofs + j];
      put((int64_t)J * kNB + r, c0 + j, v);
      Own[0][r * 17 + j] = v;
    }
    __syncthreads();
  }
  const int2 ci = colinfo[J];
  if (ci.y <= kLinvOwn) {
    // the rows, and this group's terms of each, at most two: all lists at once
    int4 rws[kLinvOwn];
    int Ks[kLinvOwn][2], slots[kLinvOwn][2];
#pragma unroll
    for (int q = 0; q < kLinvOwn; q++) rws[q] = q < ci.y ? rows[ci.x + q] : int4{0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < kLinvOwn; q++)
#pragma unroll
      for (int x = 0; x < 2; x++) {
        const int t = rws[q].w + grp + kLinvGroups * x;
        Ks[q][x] = t < rws[q].z ? klist[rws[q].y + t] : -1;
      }
#pragma unroll
    for (int q = 0; q < kLinvOwn; q++)
#pragma unroll
      for (int x = 0; x < 2; x++) {  // the place of W_K: 0, K = J
        slots[q][x] = Ks[q][x] < 0 ? -1 : 0;
#pragma unroll
        for (int p = 0; p < q; p++)
          if (Ks[q][x] >= 0 && rws[p].x == Ks[q][x]) slots[q][x] = p + 1;
      }
    double2 a[2][8];
    double4_t sum;
    auto load = [&](const int4 &rw, const int (&K)[2]) {
#pragma unroll
      for (int x = 0; x < 2; x++)
        if (K[x] >= 0) {
          const double2 *pa = reinterpret_cast<const double2 *>(
              Lf + ((int64_t)rw.x * kNB + 16 * rb + li) * np + (int64_t)K[x] * kNB + 16 * lk);
#pragma unroll
          for (int m = 0; m < 8; m++) a[x][m] = pa[m];
        }
      sum = double4_t{0.0, 0.0, 0.0, 0.0};
      if (grp == 0 && rw.w > 0) {
#pragma unroll
        for (int v = 0; v < 4; v++)
          sum[v] = W[((int64_t)rw.x * kNB + 16 * rb + lk + 4 * v) * np + gc];
      }
    };
    load(rws[0], Ks[0]);
#pragma unroll
    for (int q = 0; q < kLinvOwn; q++) {
      if (q >= ci.y) break;
      const int I = rws[q].x;
      double dreg[16];
      if (grp == 0) {
        const double *D = Dinv + (int64_t)I * kNB * kNB;
#pragma unroll
        for (int t = 0; t < 16; t++)
          dreg[t] = (4 * t < 16 * (rb + 1)) ? D[(16 * rb + li) * kNB + 4 * t + lk] : 0.0;
      }
      double4_t acc0 = {0.0, 0.0, 0.0, 0.0}, acc1 = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int x = 0; x < 2; x++)
        if (slots[q][x] >= 0) {
          const double *B = Own[slots[q][x]] + 16 * lk * 17 + li;
#pragma unroll
          for (int m = 0; m < 8; m++) {
            acc0 = mfma4(a[x][m].x, B[34 * m], acc0);
            acc1 = mfma4(a[x][m].y, B[34 * m + 17], acc1);
          }
        }
      sum += acc0 + acc1;
#pragma unroll
      for (int v = 0; v < 4; v++) Bx[grp][(16 * rb + lk + 4 * v) * 17 + li] = sum[v];
      if (q + 1 < kLinvOwn && q + 1 < ci.y) load(rws[(q + 1) % kLinvOwn], Ks[(q + 1) % kLinvOwn]);
      lds_barrier();
      if (grp == 0) {
        double4_t o = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int t = 0; t < 16; t++)
          if (4 * t < 16 * (rb + 1))
            o = mfma4(dreg[t], Bx[0][(4 * t + lk) * 17 + li] + Bx[1][(4 * t + lk) * 17 + li], o);
#pragma unroll
        for (int v = 0; v < 4; v++) {
          put((int64_t)I * kNB + 16 * rb + lk + 4 * v, gc, -o[v]);
          Own[q + 1][(16 * rb + lk + 4 * v) * 17 + li] = -o[v];
        }
      }
      lds_barrier();  // the row is there for the next one, Bx for its sums
    }
    return;
  }
  for (int q = 0; q < ci.y; q++) {
    const int4 rw = rows[ci.x + q];
    const int I = rw.x;
    double dreg[16];  // group 0: rows 16 rb.. of L_II^{-1}, columns k < 16 (rb + 1)
    double4_t sum = {0.0, 0.0, 0.0, 0.0};
    if (grp == 0) {
      const double *D = Dinv + (int64_t)I * kNB * kNB;
#pragma unroll
      for (int t = 0; t < 16; t++)
        dreg[t] = (4 * t < 16 * (rb + 1)) ? D[(16 * rb + li) * kNB + 4 * t + lk] : 0.0;
      if (rw.w > 0) {
#pragma unroll
        for (int v = 0; v < 4; v++)
          sum[v] = W[((int64_t)I * kNB + 16 * rb + lk + 4 * v) * np + gc];
      }
    }
    sum += linv_terms(Lf, W, np, I, klist + rw.y, rw.w + grp, rw.z, kLinvGroups, rb, gc);
#pragma unroll
    for (int v = 0; v < 4; v++) Bx[grp][(16 * rb + lk + 4 * v) * 17 + li] = sum[v];
    __syncthreads();
    if (grp == 0) {
      double4_t o = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int t = 0; t < 16; t++)
        if (4 * t < 16 * (rb + 1))
          o = mfma4(dreg[t], Bx[0][(4 * t + lk) * 17 + li] + Bx[1][(4 * t + lk) * 17 + li], o);
#pragma unroll
      for (int v = 0; v < 4; v++) put((int64_t)I * kNB + 16 * rb + lk + 4 * v, gc, -o[v]);
    }
    __syncthreads();  // W_I is there for the next row, Bx for its sums
  }
}

// C = WT W restricted to m >= max(i, j) (the explicit inverse A^{-1}),
// 64x64 tiles, k staged through LDS in chunks of 16.  C is n x n; W and WT
// have row stride ld.
__global__ __launch_bounds__(256) void k_gemm_wtw(const double *__restrict__ WT,
                                                  const double *__restrict__ W, int n, int ld,
                                                  double *__restrict__ C) {
  __shared__ double As[kNB][17];
  __shared__ double Bs[16][kNB + 1];
  const int nblk = (n + kNB - 1) / kNB;
  const int bi = blockIdx.x / nblk, bj = blockIdx.x % nblk;
  const int i0 = bi * kNB, j0 = bj * kNB;
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  const int li = lane & 15, lk = lane >> 4;
  const int qr = (w >> 1) * 32, qc = (w & 1) * 32;
  double4_t acc[2][2];
#pragma unroll
  for (int x = 0; x < 2; x++)
#pragma unroll
    for (int y = 0; y < 2; y++) acc[x][y] = double4_t{0.0, 0.0, 0.0, 0.0};
  for (int m0 = std::max(i0, j0); m0 < n; m0 += 16) {
    for (int e = tid; e < kNB * 16; e += 256) {
      const int r = e >> 4, k = e & 15;
      As[r][k] = (i0 + r < n && m0 + k < n) ? WT[(int64_t)(i0 + r) * ld + m0 + k] : 0.0;
      const int kk = e >> 6, c = e & 63;
      Bs[kk][c] = (m0 + kk < n && j0 + c < n) ? W[(int64_t)(m0 + kk) * ld + j0 + c] : 0.0;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 16; k += 4) {
      double av[2], bv[2];
#pragma unroll
      for (int x = 0; x < 2; x++) av[x] = As[qr + 16 * x + li][k + lk];
#pragma unroll
      for (int y = 0; y < 2; y++) bv[y] = Bs[k + lk][qc + 16 * y + li];
#pragma unroll
      for (int x = 0; x < 2; x++)
#pragma unroll
        for (int y = 0; y < 2; y++) acc[x][y] = mfma4(av[x], bv[y], acc[x][y]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int x = 0; x < 2; x++)
#pragma unroll
    for (int y = 0; y < 2; y++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int r = i0 + qr + 16 * x + lk + 4 * v, c = j0 + qc + 16 * y + li;
        if (r < n && c < n) C[(int64_t)r * n + c] = acc[x][y][v];
      }
}

// ---------------------------------------------------------------------------
// host side
// A[s][s] = 1 on the padding indices (ipos[s] < 0)
__global__ void k_pad_identity(int np, const int *__restrict__ ipos, double *__restrict__ A) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s < np && ipos[s] < 0) A[(int64_t)s * np + s] = 1.0;
}

bool CoarseFactor::allocate(int n_, int bw_, bool f32, int planes) {
  CoarseSchedule cs;
  if (!build_coarse_schedule(n_, bw_, planes, cs)) {
    set_error(TOP3D_ERR_ARG, "coarse schedule: %s", cs.error.c_str());
    return false;
  }
  n = n_;
  bw = std::max(0, std::min(bw_, n_ - 1));
  np = cs.np;
  nblk = cs.nblk;
  std::vector<int> hipos(np, -1);
  for (int d = 0; d < n; d++) hipos[cs.pos[d]] = d;
  const size_t nn = (size_t)np * np;
  A = (double *)dalloc(sizeof(double) * nn);
  L = (double *)dalloc(sizeof(double) * nn);
  W = (double *)dalloc(sizeof(double) * nn);
  WT = (double *)dalloc(sizeof(double) * nn);
  Dinv = (double *)dalloc(sizeof(double) * (size_t)nblk * kNB * kNB);
  info = (int *)dalloc(sizeof(int) * 4);
  cw64 = (double *)dalloc(sizeof(double) * 2 * (size_t)np);
  pos = (int *)dalloc(sizeof(int) * (size_t)std::max(n, 1));
  ipos = (int *)dalloc(sizeof(int) * (size_t)np);
  std::vector<int> zt;
  for (const CholTask &tk : cs.tasks) {
    zt.push_back(tk.I * cs.nblk + tk.J);
    for (int q = 0; q < tk.nsrc; q++) {
      zt.push_back(tk.I * cs.nblk + tk.K[q]);
      zt.push_back(tk.J * cs.nblk + tk.K[q]);
    }
  }
  std::sort(zt.begin(), zt.end());
  zt.erase(std::unique(zt.begin(), zt.end()), zt.end());
  nztiles = (int)zt.size();
  dztiles = (int *)dalloc(sizeof(int) * std::max<size_t>(1, zt.size()));
  ntask = (int)cs.tasks.size();
  dtasks = (CholTask *)dalloc(sizeof(CholTask) * std::max<size_t>(1, cs.tasks.size()));
  dcolinfo = (int2 *)dalloc(sizeof(int) * cs.lcolinfo.size());
  dlevel = (int *)dalloc(sizeof(int) * cs.tile_level.size());
  for (hipEvent_t &e : ev_level)
    if (!T3D_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming))) return false;
  drows = (int4 *)dalloc(sizeof(int) * std::max<size_t>(4, cs.rows.size()));
  dklist = (int *)dalloc(sizeof(int) * std::max<size_t>(1, cs.klist.size()));
  // (the products read up to kTriBatch entries past a row's list)
  list_stride = cs.list_stride;
  dwlist = (int *)dalloc(sizeof(int) * (cs.wlist.size() + kTriBatch));
  dwtlist = (int *)dalloc(sizeof(int) * (cs.wtlist.size() + kTriBatch));
  if (f32) {
    W32 = (float *)dalloc(sizeof(float) * nn);
    WT32 = (float *)dalloc(sizeof(float) * nn);
    cw32 = (float *)dalloc(sizeof(float) * 2 * (size_t)np);
  }
  if (!(A && L && W && WT && Dinv && info && cw64 && pos && ipos && dtasks && dcolinfo &&
        drows && dklist && dztiles && dwlist && dwtlist && dlevel && (!f32 || (W32 && WT32 && cw32))))
    return false;
  launch_first = cs.launch_first;
  launch_count = cs.launch_count;
  level_launch = cs.level_launch;
  level_rows.assign(cs.nlevels, 0);
  for (int v = 0; v < cs.nlevels; v++)
    for (int J = 0; J < nblk; J++)
      level_rows[v] = std::max(level_rows[v], cs.lcolinfo[2 * ((size_t)v * nblk + J) + 1]);
  hipStream_t s = stream();
  auto up = [&](void *dst, const void *src, size_t bytes) {
    return bytes == 0 || T3D_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s));
  };
  return up(pos, cs.pos.data(), sizeof(int) * n) && up(ipos, hipos.data(), sizeof(int) * np) &&
         up(dztiles, zt.data(), sizeof(int) * zt.size()) &&
         up(dtasks, cs.tasks.data(), sizeof(CholTask) * cs.tasks.size()) &&
         up(drows, cs.rows.data(), sizeof(int) * cs.rows.size()) &&
         up(dklist, cs.klist.data(), sizeof(int) * cs.klist.size()) &&
         up(dcolinfo, cs.lcolinfo.data(), sizeof(int) * cs.lcolinfo.size()) &&
         up(dlevel, cs.tile_level.data(), sizeof(int) * cs.tile_level.size()) &&
         up(dwlist, cs.wlist.data(), sizeof(int) * cs.wlist.size()) &&
         up(dwtlist, cs.wtlist.data(), sizeof(int) * cs.wtlist.size()) &&
         T3D_HIP(hipStreamSynchronize(s));
}

void CoarseFactor::release() {
  for (void *p : {(void *)A, (void *)L, (void *)W, (void *)WT, (void *)Dinv, (void *)info,
                  (void *)cw64, (void *)W32, (void *)WT32, (void *)cw32, (void *)pos,
                  (void *)ipos, (void *)dtasks, (void *)dcolinfo, (void *)drows,
                  (void *)dklist, (void *)dztiles, (void *)dlevel, (void *)dwlist,
                  (void *)dwtlist})
    if (p) dfree(p);
  for (hipEvent_t &e : ev_level) {
    if (e) hipEventDestroy(e);
    e = nullptr;
  }
  dztiles = dlevel = dwlist = dwtlist = nullptr;
  nztiles = 0;
  A = L = W = WT = Dinv = cw64 = nullptr;
  W32 = WT32 = cw32 = nullptr;
  info = pos = ipos = dklist = nullptr;
  dtasks = nullptr;
  dcolinfo = nullptr;
  drows = nullptr;
}

// zero the listed 64x64 tiles of an np x np matrix, one workgroup per tile
__global__ __launch_bounds__(256) void k_zero_tiles(double *__restrict__ A, int np, int nblk,
                                                    const int *__restrict__ tiles) {
  const int tile = tiles[blockIdx.x];
  const int64_t r0 = (int64_t)(tile / nblk) * kNB, c0 = (int64_t)(tile % nblk) * kNB;
  for (int e = threadIdx.x; e < kNB * kNB; e += 256) A[(r0 + (e >> 6)) * np + c0 + (e & 63)] = 0.0;
}

// A = 0 on the tiles the factorization reads, identity on the padding
void CoarseFactor::begin_assembly() {
  if (nztiles > 0)
    hipLaunchKernelGGL(k_zero_tiles, dim3(nztiles), dim3(256), 0, stream(), A, np, nblk,
                       dztiles);
  hipLaunchKernelGGL(k_pad_identity, dim3((np + 255) / 256), dim3(256), 0, stream(), np, ipos,
                     A);
}

int CoarseFactor::factor(bool f32out) {
  factor_async(f32out);
  return check_info();
}

int CoarseFactor::check_info() {
  int hinfo = 0;
  hipStream_t s = stream();
  if (!T3D_HIP(hipMemcpyAsync(&hinfo, info, sizeof(int), hipMemcpyDeviceToHost, s)) ||
      !T3D_HIP(hipStreamSynchronize(s)))
    return TOP3D_ERR_HIP;
  if (hinfo) {
    set_error(TOP3D_ERR_NOT_SPD, "coarse Cholesky: non-positive pivot");
    return TOP3D_ERR_NOT_SPD;
  }
  return TOP3D_OK;
}

void CoarseFactor::factor_async(bool f32out, hipStream_t with_w) {
  hipStream_t s = stream();
  if (!T3D_HIP(hipMemsetAsync(info, 0, sizeof(int), s))) return;
  const bool f32 = f32out && W32;  // FP32 W, W^T for the mixed V-cycle, else FP64 W^T
  const int nlev = (int)level_launch.size(), nlaunch = (int)launch_first.size();
  hipStream_t sw = with_w ? with_w : s;
  const int max_level_rows =
      level_rows.empty() ? 0 : *std::max_element(level_rows.begin(), level_rows.end());
  auto rows_of = [&](int v) {  // level v's rows of W
    hipLaunchKernelGGL(k_linv_rows, dim3(np / kStrip), dim3(256 * kLinvGroups), 0, sw, L, Dinv, np,
                       dcolinfo + (size_t)v * nblk, dlevel, v, drows, dklist, W,
                       f32 ? nullptr : WT, f32 ? W32 : nullptr, f32 ? WT32 : nullptr);
  };
  auto sums_from = [&](int v) {  // its terms in the rows of the levels above
    if (max_level_rows > 0)
      hipLaunchKernelGGL(k_linv_sums, dim3(nblk, max_level_rows, nlev - 1 - v), dim3(512), 0, sw,
                         L, np, dcolinfo, dlevel, v, drows, dklist, W);
  };
  // With a stream of its own, level v's rows of W follow the launch after the
  // level's last one (which completes L in its columns for the sums of the
  // levels above), and the last level's rows the last launch.
  int v = 0;
  for (int q = 0; q < nlaunch; q++) {
    hipLaunchKernelGGL(k_chol_task, dim3(launch_count[q]), dim3(512), 0, s, A, L, Dinv, np,
                       dtasks + launch_first[q], info);
    if (with_w && v + 1 < nlev && q == level_launch[v] + 1) {
      hipEventRecord(ev_level[v & 1], s);
      hipStreamWaitEvent(sw, ev_level[v & 1], 0);
      rows_of(v);
      sums_from(v++);
    }
  }
  if (with_w) {
    hipEventRecord(ev_level[v & 1], s);
    hipStreamWaitEvent(sw, ev_level[v & 1], 0);
  }
  for (; v < nlev; v++) {
    rows_of(v);
    if (v + 1 < nlev) sums_from(v);
  }
}

// ---------------------------------------------------------------------------
// Coarsest solve z = W^T (W r) in the factor's storage order: lower-triangular
// GEMV, upper-triangular GEMV scattered back to the halo layout (the halo of z
// stays zero).  The V-cycle's restriction writes r in storage order; the
// gather is for other callers.
template <typename T>
__global__ void k_gather_interior(int nx, int ny, int nz, int wy, int wz,
                                  const int *__restrict__ pos, const T *__restrict__ in,
                                  T *__restrict__ out) {
  const int64_t nint = (int64_t)nx * ny * nz;
  const int64_t d = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (d >= 3 * nint) return;
  const int64_t p = d / 3;
  const int j = (int)(p % ny), k = (int)((p / ny) % nz), i = (int)(p / ((int64_t)ny * nz));
  out[pos[d]] = in[3 * (((int64_t)(i + 1) * wz + (k + 1)) * wy + (j + 1)) + d % 3];
}

// Two rows of M x per workgroup of 4 waves, FP64 accumulation, over the tiles
// of the rows' tile row that can be non-zero (41% of the triangle at coarse
// 16x8x8): the tile columns come from a list, whose entries all threads load
// at once, and 16 or 32 lanes read a tile's row of M (16 bytes each), so that
// a row takes one wait for the list and one for its loads.  The product is
// bound by those waits.
// s[0], s[1]: the rows' sums, valid in thread 0.
template <typename T>
__device__ __forceinline__ void tri_rows(const T *__restrict__ M, int64_t np, int row0,
                                         const int *__restrict__ list, const T *__restrict__ x,
                                         double (&s)[2]) {
  constexpr int V = 16 / sizeof(T), kLanes = kNB / V;  // values per load, lanes per tile
  constexpr int kTiles = 256 / kLanes;                 // tiles per load of the workgroup
  constexpr int kU = sizeof(T) == 4 ? 4 : 5;           // loads per batch
  static_assert(kU * kTiles <= kTriBatch, "list padding");
  typedef T vec __attribute__((ext_vector_type(V)));
  const int t = threadIdx.x, off = V * (t % kLanes), tile = t / kLanes;
  const T *a0 = M + (int64_t)row0 * np, *a1 = a0 + np;
  const int cnt = list[0];
  s[0] = s[1] = 0.0;
  for (int b = 0; b < cnt; b += kU * kTiles) {  // (uniform)
    int c[kU];
#pragma unroll
    for (int u = 0; u < kU; u++) c[u] = list[1 + b + u * kTiles + tile];
    vec v0[kU], v1[kU], xv[kU];
#pragma unroll
    for (int u = 0; u < kU; u++) {
      const bool in = b + u * kTiles + tile < cnt;
      const int col = in ? kNB * c[u] + off : off;
      v0[u] = *reinterpret_cast<const vec *>(a0 + col);
      v1[u] = *reinterpret_cast<const vec *>(a1 + col);
      xv[u] = *reinterpret_cast<const vec *>(x + col);
      c[u] = in;
    }
#pragma unroll
    for (int u = 0; u < kU; u++)
#pragma unroll
      for (int e = 0; e < V; e++) {
        const double xe = (double)xv[u][e];
        s[0] += c[u] ? (double)v0[u][e] * xe : 0.0;
        s[1] += c[u] ? (double)v1[u][e] * xe : 0.0;
      }
  }
  __shared__ double sm[4][2];
#pragma unroll
  for (int r = 0; r < 2; r++) {
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) s[r] += __shfl_down(s[r], d, 64);
    if ((t & 63) == 0) sm[t >> 6][r] = s[r];
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 2; r++) s[r] = (sm[0][r] + sm[1][r]) + (sm[2][r] + sm[3][r]);
}

// (the tile rows with the longest lists come last in storage order, and first
// in the grid)
template <typename T>
__global__ __launch_bounds__(256) void k_trmv_lower(const T *__restrict__ Wm, int np,
                                                    const int *__restrict__ lists, int stride,
                                                    const T *__restrict__ x, T *__restrict__ y) {
  const int row0 = np - 2 - 2 * (int)blockIdx.x;
  double s[2];
  tri_rows(Wm, np, row0, lists + (row0 / kNB) * stride, x, s);
  if (threadIdx.x == 0) {
    y[row0] = (T)s[0];
    y[row0 + 1] = (T)s[1];
  }
}

template <typename T>
__global__ __launch_bounds__(256) void k_trmv_upper_scatter(int ny, int nz, int wy, int wz,
                                                            const int *__restrict__ ipos,
                                                            const T *__restrict__ WTm, int np,
                                                            const int *__restrict__ lists,
                                                            int stride, const T *__restrict__ y,
                                                            T *__restrict__ out) {
  const int row0 = 2 * blockIdx.x;
  const int d = ipos[row0 + (threadIdx.x & 1)];
  double s[2];
  tri_rows(WTm, np, row0, lists + (row0 / kNB) * stride, y, s);
  if (threadIdx.x < 2 && d >= 0) {
    const int p = d / 3;
    const int j = p % ny, k = (p / ny) % nz, i = p / (ny * nz);
    out[3 * (((int64_t)(i + 1) * wz + (k + 1)) * wy + (j + 1)) + d % 3] =
        (T)(threadIdx.x ? s[1] : s[0]);
  }
}

template <typename T>
void launch_coarse_apply(const DevGrid &g, int l, const CoarseFactor &cf, const T *in, T *out) {
  const Level &L = g.lv[l];
  const int n = cf.n, np = cf.np;
  T *x = cf.cw<T>(), *y = x + np;  // padding entries of x stay zero
  const int bs = 256;
  if (in)
    hipLaunchKernelGGL((k_gather_interior<T>), dim3((n + bs - 1) / bs), dim3(bs), 0, stream(),
                       L.nx, L.ny, L.nz, L.wy, L.wz, cf.pos, in, x);
  hipLaunchKernelGGL((k_trmv_lower<T>), dim3(np / 2), dim3(256), 0, stream(), cf.w<T>(), np,
                     cf.dwlist, cf.list_stride, x, y);
  hipLaunchKernelGGL((k_trmv_upper_scatter<T>), dim3(np / 2), dim3(256), 0, stream(), L.ny, L.nz,
                     L.wy, L.wz, cf.ipos, cf.wt<T>(), np, cf.dwtlist, cf.list_stride, y, out);
}

template void launch_coarse_apply<double>(const DevGrid &, int, const CoarseFactor &,
                                          const double *, double *);
template void launch_coarse_apply<float>(const DevGrid &, int, const CoarseFactor &,
                                         const float *, float *);

}  // namespace t3d

// A (n x n FP64, device, symmetric positive definite with half bandwidth bw)
// <- A^{-1}.
extern "C" int top3d_dense_spd_inverse(double *A_dev, int n, int bw) {
  using namespace t3d;
  if (n <= 0 || bw < 0 || !A_dev) {
    set_error(TOP3D_ERR_ARG, "top3d_dense_spd_inverse: n=%d bw=%d", n, bw);
    return TOP3D_ERR_ARG;
  }
  CoarseFactor cf;
  if (!cf.allocate(n, bw, false, 0)) {
    cf.release();
    return top3d_last_error() ? top3d_last_error() : TOP3D_ERR_HIP;
  }
  cf.begin_assembly();
  int rc = T3D_HIP(hipMemcpy2DAsync(cf.A, sizeof(double) * cf.np, A_dev, sizeof(double) * n,
                                    sizeof(double) * n, n, hipMemcpyDeviceToDevice, stream()))
               ? cf.factor()
               : TOP3D_ERR_HIP;
  if (rc == TOP3D_OK) {
    const int nblk = (n + kNB - 1) / kNB;
    hipLaunchKernelGGL(k_gemm_wtw, dim3(nblk * nblk), dim3(256), 0, stream(), cf.WT, cf.W, n,
                       cf.np, A_dev);
    if (!T3D_HIP(hipStreamSynchronize(stream()))) rc = TOP3D_ERR_HIP;
  }
  cf.release();
  return rc;
}
