// Fine-level operator, element-centric, for gfx950.
//
// Reflection structure.  The element matrix KE commutes with the three
// mirror reflections of the hexahedron.  In the per-component 8-point
// Walsh-Hadamard basis of the element's nodal values,
//   u^[q][c] = sum_p (-1)^{q.p} u[p][c]      (p, q in {0,1}^3, bit 0 = x),
// KE becomes 8 independent 3x3 blocks: block s couples the components c with
// q = s ^ (1 << c).  Blocks 1, 2, 4 contain a rigid translation (zero row and
// column) and blocks 3, 5, 6 split into a 2x2 and a 1x1; with the symmetries of
// the isotropic cube (Blocks) one element product costs 72 + 33 + 8 + 72
// operations (transform, blocks, modulus, inverse transform) instead of 576
// multiply-adds.  The host derives the
// blocks from KE_0 and checks the zero pattern (hadamard_blocks()).
//
// Tiling.  A workgroup owns a tile of TY x TZ element columns in (y, z) and
// marches along x over NX node planes, a thread per column on level 1, a thread
// per node of the columns on the fine level.  Per x-step each thread computes
// its element in the current slab, adds the pending x+ face of the previous
// slab to the x- face of this one, keeps the corner it owns (node (j+1, k+1) of
// element (j, k)) and hands the other three corners to their owners through LDS
// (9 values, one barrier).  Tiles overlap by one element
// in every direction, so every owned node of a tile interior is complete
// without atomics and the result is deterministic.
#include <climits>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <type_traits>
#include <utility>
#include <vector>

#include "t3d_internal.hpp"


namespace t3d {

// kModeJacobiDiag: Jacobi sweep whose inverse diagonal the kernel forms from
// the element moduli it already reads (fine level, solver only)
// kModeFirst: two sweeps from zero in one, in and b being the right-hand side
// and invD the reciprocal of the moduli's sum at each node (k_recip_moduli)
// kModeProlong: a sweep of in + P aux, aux the next level's vector, with invD as
// in kModeFirst
// kModeApplyX: apply with the densities in the place of the moduli, and zeros on
// the padded rows of the output
enum {
  kModeApply = 0,
  kModeJacobi = 1,
  kModeResidual = 2,
  kModeJacobiDiag = 3,
  kModeFirst = 4,
  kModeProlong = 5,
  kModeApplyX = 6
};

// position bits (x, y, z) of the reference's local node n (stencil_utility.h:19-26)
static constexpr int kPos[8][3] = {{0, 1, 0}, {1, 1, 0}, {1, 0, 0}, {0, 0, 0},
                                   {0, 1, 1}, {1, 1, 1}, {1, 0, 1}, {0, 0, 1}};

// Host: 3x3 blocks M[s][c][c'] of  T KE T^T / 64  (T: per-component WHT).
// Returns false if KE does not have the reflection structure.
bool hadamard_blocks(const double *KE, double M[8][3][3]) {
  auto chi = [](int q, int n) {
    const int d = (q & 1) * kPos[n][0] + ((q >> 1) & 1) * kPos[n][1] + ((q >> 2) & 1) * kPos[n][2];
    return (d & 1) ? -1.0 : 1.0;
  };
  double Kt[24][24];
  double scale = 0.0;
  for (int qa = 0; qa < 8; qa++)
    for (int ca = 0; ca < 3; ca++)
      for (int qb = 0; qb < 8; qb++)
        for (int cb = 0; cb < 3; cb++) {
          double s = 0.0;
          for (int a = 0; a < 8; a++)
            for (int b = 0; b < 8; b++)
              s += chi(qa, a) * KE[24 * (3 * a + ca) + 3 * b + cb] * chi(qb, b);
          Kt[3 * qa + ca][3 * qb + cb] = s / 64.0;
          scale = std::fmax(scale, std::fabs(s / 64.0));
        }
  const double tol = 1e-12 * scale;
  auto sig = [](int idx) { return (idx / 3) ^ (1 << (idx % 3)); };
  for (int a = 0; a < 24; a++)
    for (int b = 0; b < 24; b++)
      if (sig(a) != sig(b) && std::fabs(Kt[a][b]) > tol) return false;
  for (int s = 0; s < 8; s++)
    for (int c = 0; c < 3; c++)
      for (int d = 0; d < 3; d++) {
        const int qa = s ^ (1 << c), qb = s ^ (1 << d);
        M[s][c][d] = Kt[3 * qa + c][3 * qb + d];
      }
  // zero pattern used by the kernel: translation rows/cols of the one-bit
  // blocks, decoupled component of the two-bit blocks
  for (int s = 1; s < 7; s++)
    for (int c = 0; c < 3; c++)
      for (int d = 0; d < 3; d++) {
        const bool one_bit = (s & (s - 1)) == 0;
        bool zero;
        if (one_bit)
          zero = (s == (1 << c)) || (s == (1 << d));
        else
          zero = (c != d) && (!((s >> c) & 1) || !((s >> d) & 1));
        if (zero && std::fabs(M[s][c][d]) > tol) return false;
        if (zero) M[s][c][d] = 0.0;
      }
  return true;
}

// The blocks' values: KE of the isotropic cube is the same under the exchange
// of any two axes, which leaves 8 of the 45 non-zeros, and sigma = (1, -1, 1),
// the reference's direction of y, carries all their signs.  With x the inputs
// of block s (fine_blocks() checks every entry of the 8 matrices):
//   s = 0, 7: (a - b) I + b sigma sigma^T          (d0, b0; d7, b7)
//   s = one axis k: p on the diagonal, q sigma_c sigma_d off it, for the two
//     other components c and d; zero for k         (p1, q1)
//   s = two axes c, d: r (1, sigma_c sigma_d)^T (1, sigma_c sigma_d) for
//     these; t for the third                       (r2, t2)
// Held in scalar registers throughout the march; with all 45 the kernels
// loaded most of them again at every slab.
template <typename T>
struct Blocks {
  T d0, b0, p1, q1, r2, t2, d7, b7;
  // 1 / KE[3a+c][3a+c]: the diagonal of KE is the same for all 8 nodes, so
  // the assembled diagonal at a node is KE[c][c] times the sum of the moduli
  // of its elements
  T ikd[3];
};

// The element transform h[q][c] = sum_p (-1)^{q.p} u[p][c] (p, q in {0,1}^3,
// q = qx | qy<<1 | qz<<2) is split along x: with F_px[f][c] the 4-point
// (y, z) transform of the element's face px (f = qy | qz<<1),
//   h[2f] = F_0[f] + F_1[f],   h[2f+1] = F_0[f] - F_1[f].
// A thread marching along x transforms each node plane once and reuses it
// for the two elements that share it; the inverse runs the same way, and the
// two element contributions to a plane are summed before its 4-point
// inverse.

// F[f][c] for the 4 nodes v[py][pz][c] of a face (its own inverse up to 4)
template <typename T>
__device__ __forceinline__ void face_wht(const T (&v)[2][2][3], T (&F)[4][3]) {
#pragma unroll
  for (int c = 0; c < 3; c++) {
    const T a0 = v[0][0][c] + v[1][0][c], a1 = v[0][0][c] - v[1][0][c];
    const T b0 = v[0][1][c] + v[1][1][c], b1 = v[0][1][c] - v[1][1][c];
    F[0][c] = a0 + b0;
    F[1][c] = a1 + b1;
    F[2][c] = a0 - b0;
    F[3][c] = a1 - b1;
  }
}

// node values y[py][pz][c] = sum_f (-1)^{qy py + qz pz} G[f][c]
template <typename T>
__device__ __forceinline__ void face_iwht(const T (&G)[4][3], T (&y)[2][2][3]) {
#pragma unroll
  for (int c = 0; c < 3; c++) {
    const T a0 = G[0][c] + G[2][c], a1 = G[0][c] - G[2][c];  // qz summed: pz = 0, 1
    const T b0 = G[1][c] + G[3][c], b1 = G[1][c] - G[3][c];
    y[0][0][c] = a0 + b0;
    y[1][0][c] = a0 - b0;
    y[0][1][c] = a1 + b1;
    y[1][1][c] = a1 - b1;
  }
}

// g = E (T KE T^T / 64) h for one fine element (transformed in and out)
template <typename T>
__device__ __forceinline__ void element_core(const Blocks<T> &B, T E, const T (&h)[8][3],
                                             T (&g)[8][3]) {
  // (the modulus times the 8 values: fewer products than with the 21 outputs)
  constexpr int sg[3] = {1, -1, 1};
#pragma unroll
  for (int s = 0; s < 8; s += 7) {
    const T d = E * (s ? B.d7 : B.d0), b = E * (s ? B.b7 : B.b0);
    const T x0 = h[s ^ 1][0], x1 = h[s ^ 2][1], x2 = h[s ^ 4][2];
    const T w = b * ((x0 + x2) - x1);
    g[s ^ 1][0] = d * x0 + w;
    g[s ^ 2][1] = d * x1 - w;
    g[s ^ 4][2] = d * x2 + w;
  }
  const T p = E * B.p1, q = E * B.q1, r = E * B.r2, t = E * B.t2;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const int c = k == 0 ? 1 : 0, d = k == 2 ? 1 : 2;  // the other two
    const bool neg = sg[c] * sg[d] < 0;
    const int s1 = 1 << k, s2 = 7 ^ s1;
    const T xc = h[s1 ^ (1 << c)][c], xd = h[s1 ^ (1 << d)][d];
    g[0][k] = 0;
    g[s1 ^ (1 << c)][c] = neg ? p * xc - q * xd : p * xc + q * xd;
    g[s1 ^ (1 << d)][d] = neg ? p * xd - q * xc : p * xd + q * xc;
    const T yc = h[s2 ^ (1 << c)][c], yd = h[s2 ^ (1 << d)][d];
    const T w = r * (neg ? yc - yd : yc + yd);
    g[s2 ^ (1 << c)][c] = w;
    g[s2 ^ (1 << d)][d] = neg ? -w : w;
    g[7][k] = t * h[7][k];
  }
}

// ---------------------------------------------------------------------------
// Level 1.  A level-1 element is 2x2x2 fine elements with moduli E_o
// (o = ox | oy<<1 | oz<<2); its matrix is sum_o E_o KE1[o], KE1[o] the
// Galerkin projection of KE onto sub-cell o.  The sub-cells are mirror images
// of sub-cell 0, so in the transformed basis, with the index of row (q, c)
// relabelled sigma = q ^ (1 << c),
//   (T K T^T / 64)[(sa,ca)][(sb,cb)] = K1[(sa,ca)][(sb,cb)] * Ehat[sa ^ sb],
//   Ehat[d] = sum_o (-1)^{d.o} E_o,
// where K1 is the transformed sub-cell-0 matrix.  K1 has 279 non-zeros in a
// fixed pattern (independent of the Poisson ratio; kK1Mask, checked on the
// host), so an element product costs 279 + 192 multiply-adds plus the three
// transforms, against 8 x 576 for the sum of sub-cell matrices.
static constexpr uint32_t kK1Mask[24] = {
    0x53977, 0x53977, 0x53977, 0x0,      0x653f77, 0xa7b977, 0x653f77, 0x0,
    0xdd3977, 0x650650, 0x650650, 0xffb977, 0xa7b977, 0xdd3977, 0x0,   0xa69820,
    0xfd3f77, 0xa69820, 0xe7bf77, 0xd92900, 0xd92900, 0xe79e70, 0xfd2f50, 0xffb920};
constexpr int kK1Nnz = 279;
// The non-zeros take 20 magnitudes: entry t of the row-major non-zero list is
// kK1Class[t] & 127 of those, negated when bit 7 is set.  The classes hold
// for every Poisson ratio (tests/test_k1_classes.py derives them by sampling
// ratios from 0.05 to 0.49); init_coef checks them against the K1 it computes.
constexpr int kK1Classes = 20;
static constexpr uint8_t kK1Class[kK1Nnz] = {
    0, 1, 129, 2, 130, 3, 130, 4, 3, 2, 132, 5, 1, 0, 1, 3,
    2, 2, 2, 132, 2, 3, 5, 132, 129, 1, 0, 2, 3, 130, 3, 5,
    130, 2, 132, 4, 2, 3, 2, 6, 7, 8, 132, 9, 137, 10, 132, 5,
    11, 12, 13, 141, 130, 2, 3, 7, 6, 4, 5, 11, 136, 132, 137, 10,
    137, 140, 141, 141, 3, 2, 130, 8, 4, 6, 135, 137, 9, 138, 5, 132,
    12, 11, 141, 13, 130, 2, 3, 132, 5, 135, 6, 11, 4, 8, 12, 138,
    9, 137, 13, 141, 9, 137, 14, 142, 13, 141, 137, 9, 137, 9, 142, 14,
    141, 13, 9, 137, 4, 132, 5, 10, 11, 138, 11, 15, 140, 12, 141, 16,
    141, 144, 13, 141, 17, 145, 18, 3, 2, 130, 132, 136, 5, 4, 140, 6,
    7, 137, 10, 137, 11, 141, 141, 2, 3, 2, 5, 132, 132, 8, 12, 7,
    6, 11, 10, 137, 9, 141, 13, 137, 141, 137, 14, 14, 141, 137, 137, 132,
    5, 132, 11, 10, 12, 12, 13, 141, 16, 10, 11, 15, 16, 141, 13, 145,
    18, 145, 137, 141, 137, 14, 14, 141, 137, 137, 5, 132, 4, 12, 140, 11,
    138, 141, 13, 144, 11, 10, 141, 16, 141, 15, 18, 145, 17, 9, 13, 137,
    141, 14, 142, 137, 9, 137, 141, 9, 13, 142, 14, 9, 137, 13, 141, 141,
    137, 9, 17, 141, 137, 145, 137, 18, 19, 146, 18, 141, 13, 13, 9, 137,
    145, 141, 18, 145, 137, 9, 146, 19, 146, 141, 141, 18, 141, 13, 137, 145,
    137, 17, 9, 137, 18, 146, 19,
};

__host__ __device__ constexpr int k1_offset(int row) {
  int o = 0;
  for (int r = 0; r < row; r++) o += __builtin_popcount(kK1Mask[r]);
  return o;
}

// The class values travel as a kernel argument and stay in scalar registers
// for the whole kernel; every non-zero is one of them, up to a sign that
// folds into the multiply-add.
template <typename T>
struct K1Vals {
  T v[kK1Classes];
};

template <typename T, int IDX>
__device__ __forceinline__ T k1coef(const K1Vals<T> &kv) {
  constexpr uint8_t code = kK1Class[IDX];
  const T v = kv.v[code & 127];
  return (code & 128) ? -v : v;
}

// Host: K1 from the sub-cell matrices KE1 (8 x 576, sub-cell index
// 4 ox + 2 oz + oy), checking the mirror relation for all 8 sub-cells and
// the zero pattern.  Returns false if either fails.
bool level1_hadamard(const double *KE1, double *coef) {
  auto chi = [](int q, int n) {
    const int d = (q & 1) * kPos[n][0] + ((q >> 1) & 1) * kPos[n][1] + ((q >> 2) & 1) * kPos[n][2];
    return (d & 1) ? -1.0 : 1.0;
  };
  auto transformed = [&](const double *K, int ra, int rb) {  // ra = 3 q + c
    const int qa = ra / 3, ca = ra % 3, qb = rb / 3, cb = rb % 3;
    double s = 0.0;
    for (int a = 0; a < 8; a++)
      for (int b = 0; b < 8; b++) s += chi(qa, a) * K[24 * (3 * a + ca) + 3 * b + cb] * chi(qb, b);
    return s / 64.0;
  };
  double K1[24][24], scale = 0.0;
  for (int sa = 0; sa < 8; sa++)
    for (int ca = 0; ca < 3; ca++)
      for (int sb = 0; sb < 8; sb++)
        for (int cb = 0; cb < 3; cb++) {
          const double v = transformed(KE1, 3 * (sa ^ (1 << ca)) + ca, 3 * (sb ^ (1 << cb)) + cb);
          K1[3 * sa + ca][3 * sb + cb] = v;
          scale = std::fmax(scale, std::fabs(v));
        }
  const double tol = 1e-12 * scale;
  int k = 0;
  for (int r = 0; r < 24; r++)
    for (int c = 0; c < 24; c++) {
      if ((kK1Mask[r] >> c) & 1) coef[k++] = K1[r][c];
      else if (std::fabs(K1[r][c]) > tol) return false;
    }
  if (k != kK1Nnz) return false;
  for (int ox = 0; ox < 2; ox++)
    for (int oy = 0; oy < 2; oy++)
      for (int oz = 0; oz < 2; oz++) {
        const double *K = KE1 + 576 * (4 * ox + 2 * oz + oy);
        const int o = ox | (oy << 1) | (oz << 2);
        for (int sa = 0; sa < 8; sa++)
          for (int ca = 0; ca < 3; ca++)
            for (int sb = 0; sb < 8; sb++)
              for (int cb = 0; cb < 3; cb++) {
                const double sgn = (__builtin_popcount(o & (sa ^ sb)) & 1) ? -1.0 : 1.0;
                const double v = transformed(K, 3 * (sa ^ (1 << ca)) + ca, 3 * (sb ^ (1 << cb)) + cb);
                if (std::fabs(v - sgn * K1[3 * sa + ca][3 * sb + cb]) > tol) return false;
              }
      }
  return true;
}

// One row (3 sa + ca) of the transformed product: sum over sigma groups sb
// of Ehat[sa ^ sb] * sum_cb K1[row][(sb, cb)] H[sb][cb], expanded at compile
// time over the non-zeros of kK1Mask.
template <typename T, int ROW, int SB>
__device__ __forceinline__ void l1_accum(T &acc, const K1Vals<T> &kv, const T (&Eh)[8],
                                         const T (&H)[8][3]) {
  constexpr uint32_t m = (kK1Mask[ROW] >> (3 * SB)) & 7u;
  if constexpr (m != 0) {
    constexpr int base =
        k1_offset(ROW) + __builtin_popcount(kK1Mask[ROW] & ((1u << (3 * SB)) - 1u));
    T part;
    if constexpr ((m & 1u) != 0) {
      part = k1coef<T, base>(kv) * H[SB][0];
      if constexpr ((m & 2u) != 0) part += k1coef<T, base + 1>(kv) * H[SB][1];
      if constexpr ((m & 4u) != 0)
        part += k1coef<T, base + ((m & 2u) ? 2 : 1)>(kv) * H[SB][2];
    } else if constexpr ((m & 2u) != 0) {
      part = k1coef<T, base>(kv) * H[SB][1];
      if constexpr ((m & 4u) != 0) part += k1coef<T, base + 1>(kv) * H[SB][2];
    } else {
      part = k1coef<T, base>(kv) * H[SB][2];
    }
    acc += Eh[(ROW / 3) ^ SB] * part;
  }
}

template <typename T, int ROW, int... SB>
__device__ __forceinline__ T l1_row(const K1Vals<T> &kv, const T (&Eh)[8], const T (&H)[8][3],
                                    std::integer_sequence<int, SB...>) {
  T acc = 0;
  (l1_accum<T, ROW, SB>(acc, kv, Eh, H), ...);
  return acc;
}

template <typename T, int... ROW>
__device__ __forceinline__ void l1_rows(T (&g)[8][3], const K1Vals<T> &kv, const T (&Eh)[8],
                                        const T (&H)[8][3], std::integer_sequence<int, ROW...>) {
  ((g[(ROW / 3) ^ (1 << (ROW % 3))][ROW % 3] =
        l1_row<T, ROW>(kv, Eh, H, std::make_integer_sequence<int, 8>{})),
   ...);
}

// g = (T (sum_o E_o KE1[o]) T^T / 64) h for one level-1 element, Eh the
// transformed moduli
template <typename T>
__device__ __forceinline__ void element_core_l1(const K1Vals<T> &kv, const T (&Eh)[8],
                                                const T (&h)[8][3], T (&g)[8][3]) {
  T H[8][3];  // relabelled: H[sigma][c] = h[sigma ^ (1 << c)][c]
#pragma unroll
  for (int sg = 0; sg < 8; sg++)
#pragma unroll
    for (int c = 0; c < 3; c++) H[sg][c] = h[sg ^ (1 << c)][c];
  l1_rows<T>(g, kv, Eh, H, std::make_integer_sequence<int, 24>{});
}

// A register copy made at this point of the program (an empty asm with a
// "+v" operand would keep the value in its source register, whose live range
// then overlaps the next step's load of the same variable).
__device__ __forceinline__ float copy_here(float x) {
  float y;
  asm volatile("v_mov_b32 %0, %1" : "=v"(y) : "v"(x));
  return y;
}
__device__ __forceinline__ double copy_here(double x) {
  double y;
  asm volatile("v_mov_b64 %0, %1" : "=v"(y) : "v"(x));
  return y;
}
__device__ __forceinline__ int copy_here(int x) {
  int y;
  asm volatile("v_mov_b32 %0, %1" : "=v"(y) : "v"(x));
  return y;
}

// Workgroup barrier for the LDS exchange of the tile sweeps: the wave's LDS
// accesses complete (lgkmcnt 0; vmcnt and expcnt left at their maxima), then
// s_barrier; the empty asm statements keep the compiler from moving memory
// accesses across it.  __syncthreads() also releases the wave's global
// stores to the workgroup, which waits for every vector memory operation in
// flight, the loads of the next node plane included.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_s_waitcnt(0xC07F);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

struct TileArgs {
  int nelx, nely, nelz;  // elements of the level
  int wy, wz;            // node strides of the level
  int few, fez;          // fine element strides
  int TY, TZ, NX;        // tile: element columns in y and z, node planes in x
  int nty;               // tiles along y
  int stream_out;        // store the output past the caches
  uint32_t out_bytes;    // size of the level's vectors (below 2^32 - 32)
  uint32_t e_bytes;      // size of the moduli (below 2^32)
  int c_wx, c_wy, c_wz;  // kModeProlong: nodes of the next level's vector
  uint32_t c_bytes;      // and its size
  double E0, Emin;       // kModeApplyX: the moduli at densities 1 and 0
  int wx;                // and the planes of the level
};

// The tile of a workgroup of the (slabs, tiles) grid.  The device deals
// workgroups to its 8 XCDs, each with an L2 of its own, in turn: every XCD
// takes an eighth of the tiles in the order y, z, slab, so that the tiles whose
// edges overlap march together behind one L2.  (Dealt by the plain index that
// was so only where the number of slabs is a multiple of 8: an FP32 sweep of
// 88 tiles in 17 slabs took 55.1 us so, 38.4 us in this order.)
struct TilePos {
  int by, bz, slab, dot;  // dot: place of the workgroup's partial sum
};

__device__ __forceinline__ TilePos tile_pos(const TileArgs &a) {
  const uint32_t ntx = gridDim.x, yz = gridDim.y, n = ntx * yz;
  const uint32_t id = blockIdx.y * ntx + blockIdx.x, xcd = id & 7;
  const uint32_t t = xcd * (n >> 3) + min(xcd, n & 7) + (id >> 3);
  const uint32_t slab = t / yz, tile = t - slab * yz;
  TilePos p;
  p.bz = (int)(tile / (uint32_t)a.nty);
  p.by = (int)(tile - p.bz * a.nty);
  p.slab = (int)slab;
  p.dot = (int)(tile * ntx + slab);
  return p;
}

// p[idx] with the byte offset formed in 32 bits, so that the load or store
// takes the uniform base in scalar registers and a 32-bit offset (no 64-bit
// address arithmetic per access); the host checks that every byte offset of
// the level's arrays fits in 32 bits.
template <typename T>
__device__ __forceinline__ const T *at32(const T *p, uint32_t idx) {
  return reinterpret_cast<const T *>(reinterpret_cast<const char *>(p) + idx * (uint32_t)sizeof(T));
}
template <typename T>
__device__ __forceinline__ T *at32(T *p, uint32_t idx) {
  return reinterpret_cast<T *>(reinterpret_cast<char *>(p) + idx * (uint32_t)sizeof(T));
}

// 1 / x: the hardware reciprocal (1 ulp) in FP32, where the inverse
// diagonal only scales a smoother's correction; exact division in FP64.
template <typename T>
__device__ __forceinline__ T recip(T x) {
  if constexpr (sizeof(T) == 4) return __builtin_amdgcn_rcpf(x);
  else return T(1) / x;
}

// Stores the 3 components of a node through a buffer resource of the output
// vector, at per-thread byte offset `off` and uniform byte offset `base`: an
// offset at or beyond its size (the resource's record count) writes nothing,
// which the hardware guarantees for out-of-range buffer stores, so that every
// lane can issue the store without a branch.  kNt: past the caches.
constexpr int kCached = 0, kNt = 2;
template <int AUX = kCached>
__device__ __forceinline__ void store_node(__amdgpu_buffer_rsrc_t r, uint32_t off,
                                           const float (&o)[3], uint32_t base = 0) {
  typedef uint32_t u3 __attribute__((ext_vector_type(3)));
  const u3 v = {__float_as_uint(o[0]), __float_as_uint(o[1]), __float_as_uint(o[2])};
  __builtin_amdgcn_raw_buffer_store_b96(v, r, (int)off, (int)base, AUX);
}
template <int AUX = kCached>
__device__ __forceinline__ void store_node(__amdgpu_buffer_rsrc_t r, uint32_t off,
                                           const double (&o)[3], uint32_t base = 0) {
  typedef uint32_t u4 __attribute__((ext_vector_type(4)));
  typedef uint32_t u2 __attribute__((ext_vector_type(2)));
  const uint64_t b0 = __double_as_longlong(o[0]), b1 = __double_as_longlong(o[1]),
                 b2 = __double_as_longlong(o[2]);
  const u4 lo = {(uint32_t)b0, (uint32_t)(b0 >> 32), (uint32_t)b1, (uint32_t)(b1 >> 32)};
  const u2 hi = {(uint32_t)b2, (uint32_t)(b2 >> 32)};
  __builtin_amdgcn_raw_buffer_store_b128(lo, r, (int)off, (int)base, AUX);
  __builtin_amdgcn_raw_buffer_store_b64(hi, r, (int)(off + 16u), (int)base, AUX);
}

// Loads through a buffer resource: per-thread byte offset `off`, uniform byte
// offset `base` (no address arithmetic per access)
template <typename T>
__device__ __forceinline__ T load1(__amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t base) {
  if constexpr (sizeof(T) == 4)
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, (int)base, 0));
  else
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, (int)base, 0));
}
template <typename T>
__device__ __forceinline__ void load3(__amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t base,
                                      T (&v)[3]) {
  if constexpr (sizeof(T) == 4) {
    const auto q = __builtin_amdgcn_raw_buffer_load_b96(r, (int)off, (int)base, 0);
#pragma unroll
    for (int c = 0; c < 3; c++) v[c] = __uint_as_float(q[c]);
  } else {
    typedef double d2 __attribute__((ext_vector_type(2)));
    const d2 q = __builtin_bit_cast(
        d2, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, (int)base, 0));
    v[0] = q[0];
    v[1] = q[1];
    v[2] = load1<T>(r, off + 16u, base);
  }
}

// Level 1, eight fine moduli per element.  MODE: apply / Jacobi sweep /
// residual.  fixplane[i] != 0 if a node of plane i has a fixed DOF; planes
// without one skip the per-node mask.
template <typename T, int MODE, bool BCSYM>
__device__ __forceinline__ void level1_sweep_body(
    TileArgs a, K1Vals<T> B, const T *__restrict__ E, const T *__restrict__ in,
    T *__restrict__ out, const T *__restrict__ b, const T *__restrict__ invD, T omega,
    const uint8_t *__restrict__ fix, const int *__restrict__ fixplane) {
  // LDS values per thread and buffer, an odd stride so that 64 consecutive
  // threads hit distinct banks
  constexpr int XS = 9;
  extern __shared__ unsigned char smem_raw[];
  T *xch = reinterpret_cast<T *>(smem_raw);  // [2][nthreads][XS]
  const int nthr = a.TY * a.TZ;
  const int t = threadIdx.x;
  const bool active = t < nthr;
  const int ty = t % a.TY, tz = t / a.TY;
  const TilePos w = tile_pos(a);
  const int by = w.by, bz = w.bz;
  const int j = by * (a.TY - 1) + ty;  // element column (halo index)
  const int k = bz * (a.TZ - 1) + tz;
  const int i0 = 1 + w.slab * a.NX;
  const int i1 = min(i0 + a.NX - 1, a.nelx + 1);  // last output plane
  // the element exists in memory (0..nel+1) and may carry a non-zero modulus
  const bool elem_ok = active && j <= a.nely && k <= a.nelz;
  // owned node (j+1, k+1): complete if its other three elements are in the
  // tile or are halo elements beyond the grid
  const bool last_y = (ty == a.TY - 1), last_z = (tz == a.TZ - 1);
  const bool own_ok = elem_ok && (!last_y || j + 1 == a.nely + 1) &&
                      (!last_z || k + 1 == a.nelz + 1);
  // 32-bit offsets: the host checks sizeof(T) * 3 * nodes < 2^32
  const uint32_t sx = (uint32_t)a.wy * (uint32_t)a.wz;
  const uint32_t n00 = (uint32_t)k * a.wy + j;  // node (j, k) within a plane
  // Threads whose element column lies outside the grid read the halo node
  // (0, 0) of each plane and the halo element (i, 0, 0) instead, both in
  // bounds; that element's modulus is 0, so their products are 0 and no
  // branch guards the loads.  (E holds the transformed moduli of
  // k_level1_moduli, 8 per element slot, with strides few, fez of its own.)
  const uint32_t n00c = elem_ok ? n00 : 0u;
  const uint32_t e00c = elem_ok ? (uint32_t)k * a.few + j : 0u;
  const uint32_t noff[2][2] = {{0u, (uint32_t)a.wy}, {1u, (uint32_t)a.wy + 1u}};  // [py][pz]
  const uint32_t nown = (uint32_t)(k + 1) * a.wy + (uint32_t)(j + 1);  // owned node in a plane

  // raw values of the face of node plane i (zero outside the grid)
  auto fetch_face = [&](int i, T (&v)[2][2][3]) {
#pragma unroll
    for (int py = 0; py < 2; py++)
#pragma unroll
      for (int pz = 0; pz < 2; pz++) {
        // (the march only visits planes i <= nelx + 2)
        const uint32_t nd = (uint32_t)i * sx + n00c + (elem_ok ? noff[py][pz] : 0u);
        const T *pn = at32(in, 3u * nd);
        v[py][pz][0] = pn[0];
        v[py][pz][1] = pn[1];
        v[py][pz][2] = pn[2];
      }
  };
  // BCSYM: the fixed DOFs of the face of plane i read as zero (applied when
  // the face is consumed, on the planes that hold fixed DOFs)
  auto mask_face = [&](int i, T (&v)[2][2][3]) {
    if (BCSYM && fixplane[i] != 0) {
#pragma unroll
      for (int py = 0; py < 2; py++)
#pragma unroll
        for (int pz = 0; pz < 2; pz++) {
          const uint32_t nd = (uint32_t)i * sx + n00c + (elem_ok ? noff[py][pz] : 0u);
          const uint8_t m = fix[nd];
          if (m & 1) v[py][pz][0] = 0;
          if (m & 2) v[py][pz][1] = 0;
          if (m & 4) v[py][pz][2] = 0;
        }
    }
  };
  T vq[2][2][3];

  T pendT[4][3];  // transformed x+ face of the previous slab
#pragma unroll
  for (int f = 0; f < 4; f++)
#pragma unroll
    for (int c = 0; c < 3; c++) pendT[f][c] = 0;

  // Every load but the slab's moduli is issued a step ahead of its use, so that its latency
  // hides behind a step of element work; per step, in issue order:
  //   head: wait for the raw face of plane i+1 (issued at the last step's
  //         head), then issue that of the next step;
  //   end:  the owned node's output of plane i, then the loads of the owned
  //         node's operands for step i+1 (b, invD, mask), issued after this
  //         step's operands have been used so that one set is live at a time.
  // Every path through a step issues the same memory operations, so the
  // waits leave the younger ones in flight (the memory counter is in order).
  struct NodeIn {  // the owned node's b, invD and fixed-DOF mask
    T bb[3], di[3];
    uint8_t m;
  };
  auto load_node = [&](int i, NodeIn &sv) {
    // threads that own no node read node 0 of the plane (in bounds) and
    // never use it
    const uint32_t nd = (uint32_t)i * sx + (own_ok ? nown : 0u);
    const uint32_t d0 = 3u * nd;
    if (MODE != kModeApply) {
      const T *pb = at32(b, d0);
      sv.bb[0] = pb[0];
      sv.bb[1] = pb[1];
      sv.bb[2] = pb[2];
    }
    if (MODE == kModeJacobi) {
      const T *pd = at32(invD, d0);
      sv.di[0] = pd[0];
      sv.di[1] = pd[1];
      sv.di[2] = pd[2];
    }
    sv.m = fixplane[i] != 0 ? fix[nd] : uint8_t(0);
  };
  // the output vector as a buffer resource (stride 0, size in bytes); the
  // offset out_bytes addresses nothing
  const __amdgpu_buffer_rsrc_t orsrc =
      __builtin_amdgcn_make_buffer_rsrc(out, (short)0, (int)a.out_bytes, 0x00020000);
  NodeIn nv{};
  // u0: the owned node (j+1, k+1) of plane i, node (1, 1) of this thread's
  // face of plane i; u1: that of plane i+1 (unmasked even when BCSYM masks
  // the faces)
  T u0[3] = {0, 0, 0}, u1[3] = {0, 0, 0};

  // element slab i (node planes i, i+1): Fc the transformed face of plane
  // i, Fn that of plane i+1 (from the raw face in vq)
  auto step = [&](int i, const T (&Fc)[4][3], T (&Fn)[4][3]) {
    const bool emit = i >= i0;  // uniform
    const uint32_t d0 = 3u * ((uint32_t)i * sx + nown);
    // The values of the face are copied into registers of their own here,
    // where they have been waited for: the loads issued below then land in
    // the registers they leave (an empty asm with a "+v" operand fixes the
    // transformed face here).
#pragma unroll
    for (int c = 0; c < 3; c++) u1[c] = copy_here(vq[1][1][c]);
    mask_face(i + 1, vq);
    face_wht<T>(vq, Fn);
#pragma unroll
    for (int f = 0; f < 4; f++)
#pragma unroll
      for (int c = 0; c < 3; c++) asm volatile("" : "+v"(Fn[f][c]));
    // nothing moves across
    __builtin_amdgcn_sched_barrier(0);
    // (unconditional, the last step repeats its plane)
    fetch_face(min(i + 2, i1 + 1), vq);
    T h[8][3];
#pragma unroll
    for (int f = 0; f < 4; f++)
#pragma unroll
      for (int c = 0; c < 3; c++) {
        h[2 * f][c] = Fc[f][c] + Fn[f][c];
        h[2 * f + 1][c] = Fc[f][c] - Fn[f][c];
      }
    // g[0][c] (the element's rigid translations) is zero and is never formed
    // or read below
    T g[8][3];
    // Ehat: the per-element 8-point transform of the element's fine moduli,
    // formed once per set of moduli (k_level1_moduli); zero for halo
    // elements, which threads outside the grid read
    T Eh[8];
    const uint32_t eh = 8u * ((uint32_t)i * (uint32_t)(a.fez * a.few) + e00c);
    if constexpr (sizeof(T) == 4) {
      typedef float f4 __attribute__((ext_vector_type(4)));
      const f4 *pe = reinterpret_cast<const f4 *>(at32(E, eh));
      const f4 lo = pe[0], hi = pe[1];
#pragma unroll
      for (int o = 0; o < 4; o++) {
        Eh[o] = lo[o];
        Eh[o + 4] = hi[o];
      }
    } else {
      typedef double d2 __attribute__((ext_vector_type(2)));
      const d2 *pe = reinterpret_cast<const d2 *>(at32(E, eh));
#pragma unroll
      for (int o = 0; o < 4; o++) {
        const d2 v = pe[o];
        Eh[2 * o] = v[0];
        Eh[2 * o + 1] = v[1];
      }
    }
    element_core_l1<T>(B, Eh, h, g);
    T o[3] = {0, 0, 0};
    const T *bb = nv.bb, *di = nv.di;
    const uint8_t m = nv.m;
    if (emit) {
      // plane i: x- face of slab i plus the pending x+ face of slab i-1,
      // summed in the transformed basis
      T totT[4][3], tot[2][2][3];
#pragma unroll
      for (int c = 0; c < 3; c++) totT[0][c] = g[1][c] + pendT[0][c];
#pragma unroll
      for (int f = 1; f < 4; f++)
#pragma unroll
        for (int c = 0; c < 3; c++) totT[f][c] = (g[2 * f][c] + g[2 * f + 1][c]) + pendT[f][c];
      face_iwht<T>(totT, tot);
      // this thread's slot, formed anew each step (the addresses of its
      // neighbours' slots are then a few adds here rather than registers
      // held across the march)
      const int ts = copy_here(t);
      T *buf = xch + (size_t)(i & 1) * nthr * XS + XS * ts;
      if (active) {
#pragma unroll
        for (int c = 0; c < 3; c++) {
          buf[c] = tot[0][1][c];            // node (j, k+1)  -> thread (ty-1, tz)
          buf[3 + c] = tot[1][0][c];           // node (j+1, k)  -> thread (ty, tz-1)
          buf[6 + c] = tot[0][0][c];           // node (j, k)    -> thread (ty-1, tz-1)
        }
      }
      lds_barrier();
      if (own_ok) {
        T kin[3] = {tot[1][1][0], tot[1][1][1], tot[1][1][2]};
        if (!last_y) {
#pragma unroll
          for (int c = 0; c < 3; c++) kin[c] += buf[XS + c];
        }
        if (!last_z) {
#pragma unroll
          for (int c = 0; c < 3; c++) kin[c] += buf[XS * a.TY + 3 + c];
        }
        if (!last_y && !last_z) {
#pragma unroll
          for (int c = 0; c < 3; c++) kin[c] += buf[XS * (a.TY + 1) + 6 + c];
        }
#pragma unroll
        for (int c = 0; c < 3; c++) {
          const T uc = u0[c];
          T kv = kin[c];
          if ((m >> c) & 1) kv = uc;  // identity row
          if (MODE == kModeApply) {
            o[c] = kv;
          } else if (MODE == kModeJacobi) {
            o[c] = uc + omega * di[c] * (bb[c] - kv);
          } else {
            o[c] = bb[c] - kv;
          }
        }
      }
    }
    // every lane stores (the step's last memory operation, so that the next
    // step's wait for its face leaves it in flight): the owned node of an
    // emitted plane, else nothing
    store_node(orsrc, emit && own_ok ? d0 * (uint32_t)sizeof(T) : a.out_bytes, o);
    load_node(min(i + 1, i1), nv);
#pragma unroll
    for (int c = 0; c < 3; c++) pendT[0][c] = -g[1][c];
#pragma unroll
    for (int f = 1; f < 4; f++)
#pragma unroll
      for (int c = 0; c < 3; c++) pendT[f][c] = g[2 * f][c] - g[2 * f + 1][c];
  };

  // the march; the transformed face of plane i+1 becomes that of plane i
  T Fa[4][3], Fb[4][3];
  fetch_face(i0 - 1, vq);
#pragma unroll
  for (int c = 0; c < 3; c++) u0[c] = vq[1][1][c];
  mask_face(i0 - 1, vq);
  face_wht<T>(vq, Fa);
  // the loads a step's head and end would have issued before the first step
  // (the store writes nothing; the first step emits no plane and leaves the
  // node operands unused)
  fetch_face(i0, vq);
  store_node(orsrc, a.out_bytes, u0);
  load_node(i0 - 1, nv);
  for (int i = i0 - 1; i <= i1; i++) {
    step(i, Fa, Fb);
#pragma unroll
    for (int f = 0; f < 4; f++)
#pragma unroll
      for (int c = 0; c < 3; c++) Fa[f][c] = Fb[f][c];
#pragma unroll
    for (int c = 0; c < 3; c++) u0[c] = u1[c];
  }
}

// Keeps a value that a loop loads again from being loaded inside the loop only
// (the compiler would merge the loads before the loop with those in it and
// issue them where they are used).
template <typename T>
__device__ __forceinline__ void pin(T &x) {
  asm volatile("" : "+v"(x));
}

// The fine level.  A workgroup has a thread per node of its (TY + 1) x (TZ + 1)
// node tile, up to 255 nodes in FP64 and 511 in FP32; each loads its own node of the plane
// and hands it on through LDS with the exchange of the element's corners, under
// the same barrier, and works on the element whose upper corner (j, k) is its
// node (none for the tile's lower edges).  Every LDS array is [value][thread],
// so that a wave's access is contiguous but for the three face nodes of other
// rows.  Every load is issued a step before its value is used, as on level 1;
// every lane forms its node's row, and the store decides by its offset.
//
// What bounds it: the arithmetic in FP32 (about 230 instructions per element,
// of 4 cycles each, and 170 MB per sweep at 257x129x129 nodes: 33-35 us), the
// memory in FP64 (341 MB, more than the memory-side cache holds).  Before,
// with a thread per element that loaded the four nodes of its face through the
// first-level cache, all 45 values of the blocks and masks at every node: 40.0
// us and, FP64, 101 us per sweep and 72.5 us per apply, now 79 and 55-60.  At
// 513x257x257 nodes FP32 317-326 -> 293-298 us, FP64 770 -> 661 and 636 -> 489.
// (FP32 in workgroups of 4 waves: 34.6 and 356 us.)
// threads of a workgroup: two of 8 waves (FP32, 88 registers) or three of 4
// waves (FP64, 168 registers) share a CU
template <typename T>
constexpr int march_threads() {
  return sizeof(T) == 4 ? 512 : 256;
}

// LDS values per thread: two buffers of the exchange (9 corners, in the
// diagonal-forming sweep the modulus too) and of the plane's 3 components
constexpr int march_lds_values(bool diag) { return 2 * ((diag ? 10 : 9) + 3); }

template <typename T, int MODE, bool BCSYM>
__device__ __forceinline__ void fine_march_body(
    TileArgs a, Blocks<T> B, const T *__restrict__ E, const T *__restrict__ in,
    T *__restrict__ out, const T *__restrict__ b, const T *__restrict__ invD, T omega,
    const uint8_t *__restrict__ fix, const int *__restrict__ fixplane,
    double *__restrict__ dotp, void *__restrict__ aux) {
  constexpr bool kDiag = MODE == kModeJacobiDiag, kFirst = MODE == kModeFirst;
  constexpr bool kProl = MODE == kModeProlong, kX = MODE == kModeApplyX;
  constexpr bool kApply = MODE == kModeApply || kX;
  constexpr int N = march_threads<T>(), XV = kDiag ? 10 : 9;
  extern __shared__ unsigned char smem_raw[];
  T *xch = reinterpret_cast<T *>(smem_raw);  // [2][XV][N]; slot N-1: zeros
  T *nodes = xch + 2 * XV * N;               // [2][3][N]
  const int t = threadIdx.x, nrow = a.TY + 1;
  const bool active = t < nrow * (a.TZ + 1);
  const int ty = t % nrow, tz = t / nrow;
  const TilePos w = tile_pos(a);
  const int j = w.by * (a.TY - 1) + ty, k = w.bz * (a.TZ - 1) + tz;  // the node's column
  const int i0 = 1 + w.slab * a.NX;
  const int i1 = min(i0 + a.NX - 1, a.nelx + 1);  // last output plane
  const bool elem_ok = active && ty > 0 && tz > 0 && j - 1 <= a.nely && k - 1 <= a.nelz;
  const bool mat_ok = elem_ok && j > 1 && k > 1;  // kX: not an element of the halo
  const bool last_y = (ty == a.TY), last_z = (tz == a.TZ);
  const bool own_ok = elem_ok && (!last_y || j == a.nely + 1) && (!last_z || k == a.nelz + 1);
  // bytes of a plane of each array
  const uint32_t sx = (uint32_t)a.wy * (uint32_t)a.wz, sv = 3u * sx * (uint32_t)sizeof(T);
  const uint32_t se = (uint32_t)a.fez * (uint32_t)a.few * (uint32_t)sizeof(T);
  // nodes beyond the level's arrays read node 0 of the plane
  const uint32_t node =
      active && j < a.wy && k < a.wz ? (uint32_t)k * a.wy + (uint32_t)j : 0u;
  const uint32_t vnode = 3u * (uint32_t)sizeof(T) * node;
  const uint32_t vout = own_ok ? vnode : a.out_bytes;  // (a store there writes nothing)
  const uint32_t velem =
      elem_ok ? (uint32_t)sizeof(T) * ((uint32_t)(k - 1) * a.few + (uint32_t)(j - 1)) : 0u;
  // node (j - 1, k - 1) of the face
  const int f00 = max(t - nrow - 1, 0), f01 = f00 + nrow;
  // the neighbours' corners: zeros beyond the tile's last element
  const int n01 = last_y ? N - 1 : t + 1;
  const int n10 = last_z ? N - 1 : t + nrow;
  const int n11 = last_y || last_z ? N - 1 : t + nrow + 1;
  double dacc = 0.0;
  T es_prev = 0;
  auto rsrc = [](const void *p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)bytes,
                                             0x00020000);
  };
  const __amdgpu_buffer_rsrc_t rin = rsrc(in, a.out_bytes), re = rsrc(E, a.e_bytes);
  const __amdgpu_buffer_rsrc_t rfix = rsrc(fix, a.out_bytes / (3u * (uint32_t)sizeof(T)));
  const __amdgpu_buffer_rsrc_t rb = rsrc(kApply || kFirst ? in : b, a.out_bytes);
  const __amdgpu_buffer_rsrc_t rd = rsrc(MODE == kModeJacobi || kFirst || kProl ? invD : in,
                                         kFirst || kProl ? a.out_bytes / 3u : a.out_bytes);
  // the planes from plane fbase on with a fixed DOF
  int fbase = i0 - 1;
  auto fixed_planes = [&]() {
    return __ballot(fixplane[min(fbase + (int)__lane_id(), a.nelx + 2)] != 0);
  };
  uint64_t fbits = fixed_planes();
  // the node of a plane as the march carries it: its values; kFirst: its
  // right-hand side, reciprocal and fixed DOFs
  struct Node {
    T u[3], rs;
    uint32_t m;
    bool fixed;  // a fixed DOF in the plane (uniform)
  };
  // operands in flight: the node to hand on, the slab's modulus, the owned
  // node's b, invD and fixed-DOF mask
  struct Operands {
    Node p;
    T e, bb[3], di[3];
    uint32_t m;
    bool fixed;
  } s{};
  auto load_mask = [&](int i, bool &fixed) {
    if (i - fbase >= 64) {
      fbase = i;
      fbits = fixed_planes();
    }
    // (no branch: the merged value would be waited for here)
    fixed = (fbits >> (i - fbase)) & 1;
    return (uint32_t)__builtin_amdgcn_raw_buffer_load_b8(rfix, (int)(fixed ? node : 0u),
                                                         (int)((uint32_t)i * sx), 0);
  };
  auto load_plane = [&](int i_, Node &p) {  // (the march reads planes up to i1 + 1)
    const int i = min(i_, i1 + 1);
    load3<T>(rin, vnode, (uint32_t)i * sv, p.u);
    if constexpr (kFirst) {
      p.rs = load1<T>(rd, vnode / 3u, (uint32_t)i * (sx * (uint32_t)sizeof(T)));
      p.m = load_mask(i, p.fixed);
    }
  };
  // kFirst: the first sweep from zero, x = omega b / diagonal
  auto first_sweep = [&](const Node &n, T (&dd)[3], T (&x)[3]) {
#pragma unroll
    for (int c = 0; c < 3; c++) dd[c] = n.rs * B.ikd[c];
    if (n.fixed) {
#pragma unroll
      for (int c = 0; c < 3; c++)
        if ((n.m >> c) & 1) dd[c] = T(1);
    }
#pragma unroll
    for (int c = 0; c < 3; c++) x[c] = omega * dd[c] * n.u[c];
  };
  auto load_modulus = [&](int i) { return load1<T>(re, velem, (uint32_t)min(i, i1) * se); };
  auto load_node = [&](int i_) {
    const int i = min(i_, i1);
    if (kFirst) return;  // (all carried with the planes)
    if (!kApply) load3<T>(rb, vnode, (uint32_t)i * sv, s.bb);
    if (MODE == kModeJacobi) load3<T>(rd, vnode, (uint32_t)i * sv, s.di);
    if (kProl) s.di[0] = load1<T>(rd, vnode / 3u, (uint32_t)i * (sx * (uint32_t)sizeof(T)));
    s.m = load_mask(i, s.fixed);
  };
  // kProl: the nodes of the coarse plane over the tile, in LDS one at a time, a
  // thread each; Cm, the plane's interpolation in y and z at the thread's node.
  // The march starts at an odd plane, so that step 0 of a turn puts a plane
  // between two coarse ones and step 1 a plane on one.
  T *ctile = nodes + 2 * 3 * N;  // [ncn][3]
  const int cj0 = (w.by * (a.TY - 1) + 1) >> 1, ck0 = (w.bz * (a.TZ - 1) + 1) >> 1;
  const int ncy = ((w.by * (a.TY - 1) + a.TY) >> 1) + 2 - cj0;
  const int ncn = ncy * (((w.bz * (a.TZ - 1) + a.TZ) >> 1) + 2 - ck0);
  const int c11 = active ? (((k + 1) >> 1) - ck0) * ncy + ((j + 1) >> 1) - cj0 : 0;
  const int c12 = c11 + (active && (j & 1) == 0);
  const int c21 = c11 + (active && (k & 1) == 0 ? ncy : 0), c22 = c21 + c12 - c11;
  const __amdgpu_buffer_rsrc_t rc = rsrc(kProl ? aux : in, kProl ? a.c_bytes : 0u);
  const uint32_t vc =
      t < ncn ? 3u * (uint32_t)sizeof(T) *
                    ((uint32_t)min(ck0 + t / ncy, a.c_wz - 1) * (uint32_t)a.c_wy +
                     (uint32_t)min(cj0 + t % ncy, a.c_wy - 1))
              : 0u;
  T cz[3] = {0, 0, 0}, Cm[3] = {0, 0, 0};
  auto load_coarse = [&](int ic, T (&v)[3]) {
    load3<T>(rc, vc, (uint32_t)min(ic, a.c_wx - 1) * (3u * (uint32_t)sizeof(T)) *
                         ((uint32_t)a.c_wy * (uint32_t)a.c_wz), v);
  };
  auto put_coarse = [&](const T (&v)[3]) {
    if (t < ncn) {
#pragma unroll
      for (int c = 0; c < 3; c++) ctile[3 * t + c] = v[c];
    }
  };
  auto get_coarse = [&](T (&C)[3]) {
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const T *q = ctile + c;
      C[c] = T(0.25) * ((q[3 * c11] + q[3 * c12]) + (q[3 * c21] + q[3 * c22]));
    }
  };
  // plane i into LDS buffer P; n: the node as carried; BCSYM: the fixed DOFs
  // are handed on, and read back, as zeros
  auto put_plane = [&](int i, int P, const Node &p, Node &n) {
#pragma unroll
    for (int c = 0; c < 3; c++) n.u[c] = copy_here(p.u[c]);
    T v[3];
    if constexpr (kFirst) {
      n.rs = copy_here(p.rs);
      n.m = (uint32_t)copy_here((int)p.m);
      n.fixed = p.fixed;
      T dd[3];
      first_sweep(n, dd, v);
      if (BCSYM && n.fixed) {
#pragma unroll
        for (int c = 0; c < 3; c++)
          if ((n.m >> c) & 1) v[c] = 0;
      }
    } else {
      if constexpr (kProl) {
        if (P == 0) {
          T Cn[3];
          get_coarse(Cn);
#pragma unroll
          for (int c = 0; c < 3; c++) {
            n.u[c] += T(0.5) * (Cm[c] + Cn[c]);
            Cm[c] = Cn[c];
          }
        } else {
#pragma unroll
          for (int c = 0; c < 3; c++) n.u[c] += Cm[c];
        }
      }
#pragma unroll
      for (int c = 0; c < 3; c++) v[c] = n.u[c];
      if (BCSYM && fixplane[min(i, i1 + 1)] != 0) {
        const uint8_t m = fix[(uint32_t)min(i, i1 + 1) * sx + node];
#pragma unroll
        for (int c = 0; c < 3; c++)
          if ((m >> c) & 1) v[c] = 0;
      }
      if constexpr (BCSYM && !kProl) {
#pragma unroll
        for (int c = 0; c < 3; c++) n.u[c] = v[c];
      }
    }
    T *nb = nodes + P * 3 * N + t;
#pragma unroll
    for (int c = 0; c < 3; c++) nb[c * N] = v[c];
  };
  // transformed face of the plane in LDS buffer P, whose node (j, k) is n
  auto get_face = [&](int P, T (&F)[4][3], const Node &n) {
    const T *nb = nodes + P * 3 * N;
    T v[2][2][3];
#pragma unroll
    for (int c = 0; c < 3; c++) {
      v[0][0][c] = nb[c * N + f00];
      v[1][0][c] = nb[c * N + f00 + 1];
      v[0][1][c] = nb[c * N + f01];
      v[1][1][c] = kFirst || kProl ? nb[c * N + t] : n.u[c];
    }
    face_wht<T>(v, F);
  };

  T pendT[4][3];
#pragma unroll
  for (int f = 0; f < 4; f++)
#pragma unroll
    for (int c = 0; c < 3; c++) pendT[f][c] = 0;

  // element slab i, the (P + 1)th or (P + 3)th, ... of the march: Fc the
  // transformed face of plane i, Fn that of plane i+1; u0, u1, u2 the node of
  // planes i, i+1 and i+2
  auto step = [&](int i, auto par, const T (&Fc)[4][3], T (&Fn)[4][3], const Node &u0,
                  const Node &u1, Node &u2) {
    constexpr int P = decltype(par)::value;
    const bool emit = i >= i0;  // uniform
    T Ee = copy_here(s.e);
    if constexpr (kX)  // (as k_young)
      Ee = mat_ok && i >= 1 && i <= a.nelx ? T(a.Emin + (Ee * Ee * Ee) * (a.E0 - a.Emin)) : T(0);
    s.e = load_modulus(i + 1);
    get_face(1 - P, Fn, u1);
    T hh[8][3];
#pragma unroll
    for (int f = 0; f < 4; f++)
#pragma unroll
      for (int c = 0; c < 3; c++) {
        hh[2 * f][c] = Fc[f][c] + Fn[f][c];
        hh[2 * f + 1][c] = Fc[f][c] - Fn[f][c];
      }
    T g[8][3];
    element_core<T>(B, Ee, hh, g);
    T totT[4][3], tot[2][2][3];
#pragma unroll
    for (int c = 0; c < 3; c++) totT[0][c] = g[1][c] + pendT[0][c];
#pragma unroll
    for (int f = 1; f < 4; f++)
#pragma unroll
      for (int c = 0; c < 3; c++) totT[f][c] = (g[2 * f][c] + g[2 * f + 1][c]) + pendT[f][c];
#pragma unroll
    for (int c = 0; c < 3; c++) pendT[0][c] = -g[1][c];
#pragma unroll
    for (int f = 1; f < 4; f++)
#pragma unroll
      for (int c = 0; c < 3; c++) pendT[f][c] = g[2 * f][c] - g[2 * f + 1][c];
    face_iwht<T>(totT, tot);
    T *buf = xch + P * XV * N;
    if (active) {
#pragma unroll
      for (int c = 0; c < 3; c++) {
        buf[c * N + t] = tot[0][1][c];        // node (j-1, k)    -> its thread
        buf[(3 + c) * N + t] = tot[1][0][c];  // node (j, k-1)
        buf[(6 + c) * N + t] = tot[0][0][c];  // node (j-1, k-1)
      }
      if constexpr (kDiag) buf[9 * N + t] = Ee;
    }
    put_plane(i + 2, P, s.p, u2);
    load_plane(i + 3, s.p);
    if constexpr (kProl && P == 1) {
      put_coarse(cz);
      load_coarse((i + 2 + 3) / 2 + 1, cz);
    }
    lds_barrier();
    // the owned node's row, in every lane: stored where own_ok and emit
    T kin[3] = {tot[1][1][0], tot[1][1][1], tot[1][1][2]}, o[3], uo[3], dd[3];
#pragma unroll
    for (int c = 0; c < 3; c++) kin[c] += buf[c * N + n01];
#pragma unroll
    for (int c = 0; c < 3; c++) kin[c] += buf[(3 + c) * N + n10];
#pragma unroll
    for (int c = 0; c < 3; c++) kin[c] += buf[(6 + c) * N + n11];
    if constexpr (kFirst) {
      first_sweep(u0, dd, uo);
      if (u0.fixed) {
#pragma unroll
        for (int c = 0; c < 3; c++)
          if ((u0.m >> c) & 1) kin[c] = uo[c];  // identity row
      }
#pragma unroll
      for (int c = 0; c < 3; c++) s.bb[c] = u0.u[c];
    } else {
#pragma unroll
      for (int c = 0; c < 3; c++) {
        uo[c] = u0.u[c];
        dd[c] = s.di[c];
      }
    }
    if constexpr (kDiag) {  // the moduli of the two slabs' 4 elements each at the node
      const T es = ((Ee + buf[9 * N + n01]) + buf[9 * N + n10]) + buf[9 * N + n11];
      const T rs = recip<T>(es_prev + es);
      es_prev = es;
#pragma unroll
      for (int c = 0; c < 3; c++) dd[c] = rs * B.ikd[c];
    }
    if constexpr (kProl) {
#pragma unroll
      for (int c = 0; c < 3; c++) dd[c] = s.di[0] * B.ikd[c];
    }
    uint32_t m = s.m;
    if constexpr (!kFirst)
      pin(m);  // (used in the branch only, its copies for the next step would wait for the load)
    if (!kFirst && s.fixed) {
      if (BCSYM && !kProl && m != 0) {  // u0 holds zeros there
        const T *pu = at32(in, 3u * ((uint32_t)i * sx + node));
#pragma unroll
        for (int c = 0; c < 3; c++) uo[c] = pu[c];
      }
#pragma unroll
      for (int c = 0; c < 3; c++)
        if ((m >> c) & 1) {  // identity row
          kin[c] = uo[c];
          if constexpr (kDiag || kProl) dd[c] = T(1);
        }
    }
#pragma unroll
    for (int c = 0; c < 3; c++) {
      if (kApply) o[c] = kin[c];
      else if (MODE == kModeJacobi || kDiag || kFirst || kProl) o[c] = uo[c] + omega * dd[c] * (s.bb[c] - kin[c]);
      else o[c] = s.bb[c] - kin[c];
    }
    if (MODE != kModeResidual && !kFirst && !kProl && dotp) {
      double d = dacc;
#pragma unroll
      for (int c = 0; c < 3; c++)
        d += (double)(kApply ? uo[c] : s.bb[c]) * (double)o[c];
      dacc = emit && own_ok ? d : dacc;
    }
    // (an empty resource where the plane is another workgroup's)
    const __amdgpu_buffer_rsrc_t ro = rsrc(out, emit ? a.out_bytes : 0u);
    if (a.stream_out) store_node<kNt>(ro, vout, o, (uint32_t)i * sv);
    else store_node(ro, vout, o, (uint32_t)i * sv);
    if (MODE == kModeResidual && sizeof(T) == 8 && aux) {  // the FP32 copy too
      const float o32[3] = {(float)o[0], (float)o[1], (float)o[2]};
      store_node(rsrc(aux, emit ? a.out_bytes / 2 : 0u), vout / 2, o32, (uint32_t)i * sv / 2);
    }
    load_node(i + 1);
  };

  // planes i0-1 and i0 straight to LDS
  Node ua{}, ub{}, uc{}, pa{}, pb{};
  T Fa[4][3], Fb[4][3];
  load_plane(i0 - 1, pa);
  load_plane(i0, pb);
  load_plane(i0 + 1, s.p);
  s.e = load_modulus(i0 - 1);
  load_node(i0 - 1);
  if (t < 2 * XV) xch[t * N + N - 1] = 0;
  if constexpr (kProl) {  // the coarse planes at and beside plane i0
    const int ic = i0 / 2;
    T ca[3], cb[3], cc[3];
    load_coarse(ic, ca);
    load_coarse(ic + 1, cb);
    load_coarse(ic + 2, cc);
    load_coarse(ic + 3, cz);
    put_coarse(ca);
    __syncthreads();
    get_coarse(Cm);
    __syncthreads();
    put_coarse(cb);
    __syncthreads();
    put_plane(i0 - 1, 0, pa, ua);
    put_plane(i0, 1, pb, ub);
    __syncthreads();
    put_coarse(cc);
  } else {
    put_plane(i0 - 1, 0, pa, ua);
    put_plane(i0, 1, pb, ub);
  }
  __syncthreads();
  get_face(0, Fa, ua);
#pragma unroll
  for (int c = 0; c < 3; c++) {
    pin(s.p.u[c]);
    if (!kApply && !kFirst) pin(s.bb[c]);
    if (MODE == kModeJacobi) pin(s.di[c]);
    if (kProl) pin(cz[c]);
  }
  if (kProl) pin(s.di[0]);
  if constexpr (kFirst) {
    pin(s.p.rs);
    pin(s.p.m);
  }
  pin(s.e);
  __syncthreads();  // plane i0-1 is read: its buffer takes plane i0+1
  // two slabs per turn, so that faces, LDS buffers and node values change
  // places without copies
  for (int i = i0 - 1;;) {
    step(i, std::integral_constant<int, 0>{}, Fa, Fb, ua, ub, uc);
    if (++i > i1) break;
    step(i, std::integral_constant<int, 1>{}, Fb, Fa, ub, uc, ua);
    if (++i > i1) break;
    const Node uz = uc;
    ub = ua;
    ua = uz;
  }
  if constexpr (kX) {  // the rows j > nely + 1 of every (i, k), as k_zero_pad_rows
    const int first = a.nely + 2, npad = a.wy - first;
    const uint32_t n = (uint32_t)a.wx * a.wz * (uint32_t)npad;
    const uint32_t nt = gridDim.x * gridDim.y * blockDim.x;
    for (uint32_t q = (blockIdx.y * gridDim.x + blockIdx.x) * blockDim.x + t; q < n; q += nt) {
      T *po = at32(out, 3u * (q / npad * (uint32_t)a.wy + first + q % npad));
      po[0] = po[1] = po[2] = 0;
    }
  }
  if (MODE != kModeResidual && !kFirst && !kProl && dotp) {  // one partial per workgroup, fixed order
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) dacc += __shfl_down(dacc, off, 64);
    __syncthreads();
    double *red = reinterpret_cast<double *>(smem_raw);
    if ((t & 63) == 0) red[t >> 6] = dacc;
    __syncthreads();
    if (t == 0) {
      double sum = 0.0;
      for (int v = 0; v < (int)(blockDim.x >> 6); v++) sum += red[v];
      dotp[w.dot] = sum;
    }
  }
}

template <typename T, int MODE, bool BCSYM>
__global__ __launch_bounds__(march_threads<T>())
    __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 4 : 3))) void k_fine_march(
    TileArgs a, Blocks<T> B, const T *__restrict__ E, const T *__restrict__ in,
    T *__restrict__ out, const T *__restrict__ b, const T *__restrict__ invD, T omega,
    const uint8_t *__restrict__ fix, const int *__restrict__ fixplane,
    double *__restrict__ dotp, void *__restrict__ aux) {
  fine_march_body<T, MODE, BCSYM>(a, B, E, in, out, b, invD, omega, fix, fixplane, dotp, aux);
}

template <typename T, int MODE, bool BCSYM>
__global__ __launch_bounds__(sizeof(T) == 4 ? 1024 : 512) void k_level1_sweep(
    TileArgs a, K1Vals<T> B, const T *__restrict__ E, const T *__restrict__ in,
    T *__restrict__ out, const T *__restrict__ b, const T *__restrict__ invD, T omega,
    const uint8_t *__restrict__ fix, const int *__restrict__ fixplane) {
  level1_sweep_body<T, MODE, BCSYM>(a, B, E, in, out, b, invD, omega, fix, fixplane);
}

// ---------------------------------------------------------------------------
// host side
struct HostCoef {
  bool done = false, ok0 = false, ok1 = false;
  bool diag0 = false;  // KE_0 has one diagonal value per component
  Blocks<double> b64;
  Blocks<float> b32;
  K1Vals<double> k64;  // the class values of K1
  K1Vals<float> k32;
};
static HostCoef g_coef;

// The 8 values of the blocks; false if an entry of M is not what they give.
static bool fine_blocks(const double M[8][3][3], Blocks<double> &B, Blocks<float> &F) {
  const double a0 = M[0][0][0], b0 = M[0][0][2], p = M[1][1][1], q = M[2][0][2];
  const double r = M[3][0][0], t = M[3][2][2], a7 = M[7][0][0], b7 = M[7][0][2];
  const int sg[3] = {1, -1, 1};
  for (int s = 0; s < 8; s++)
    for (int c = 0; c < 3; c++)
      for (int d = 0; d < 3; d++) {
        const bool in_c = (s >> c) & 1, in_d = (s >> d) & 1;
        const int bits = __builtin_popcount(s);
        double v = 0.0;  // |entry|
        if (bits == 0) v = c == d ? a0 : b0;
        if (bits == 3) v = c == d ? a7 : b7;
        if (bits == 1 && !in_c && !in_d) v = c == d ? p : q;
        if (bits == 2 && in_c && in_d) v = r;
        if (bits == 2 && c == d && !in_c) v = t;
        if (std::fabs(M[s][c][d] - sg[c] * sg[d] * v) > 1e-12 * a0) return false;
      }
  B.d0 = a0 - b0, B.b0 = b0, B.p1 = p, B.q1 = q, B.r2 = r, B.t2 = t, B.d7 = a7 - b7, B.b7 = b7;
  F.d0 = (float)B.d0, F.b0 = (float)B.b0, F.p1 = (float)p, F.q1 = (float)q;
  F.r2 = (float)r, F.t2 = (float)t, F.d7 = (float)B.d7, F.b7 = (float)b7;
  return true;
}

static void init_coef() {
  if (g_coef.done) return;
  g_coef.done = true;
  std::vector<double> KE(576), KE1(8 * 576);
  element_matrices(0.3, 0, KE.data());
  element_matrices(0.3, 1, KE1.data());
  double M[8][3][3];
  g_coef.ok0 = hadamard_blocks(KE.data(), M);
  if (g_coef.ok0) g_coef.ok0 = fine_blocks(M, g_coef.b64, g_coef.b32);
  if (g_coef.ok0) {
    g_coef.diag0 = true;
    for (int c = 0; c < 3; c++) {
      const double d = KE[24 * c + c];
      for (int a = 1; a < 8; a++)
        if (std::fabs(KE[24 * (3 * a + c) + 3 * a + c] - d) > 1e-14 * std::fabs(d))
          g_coef.diag0 = false;
      g_coef.b64.ikd[c] = 1.0 / d;
      g_coef.b32.ikd[c] = (float)(1.0 / d);
    }
  }
  double coef[kK1Nnz];
  g_coef.ok1 = level1_hadamard(KE1.data(), coef);
  if (g_coef.ok1) {
    // class values from each class's first member (which carries sign +),
    // then every non-zero checked against its class
    bool seen[kK1Classes] = {};
    double scale = 0.0;
    for (int q = 0; q < kK1Nnz; q++) {
      const int c = kK1Class[q] & 127;
      if (!seen[c]) g_coef.k64.v[c] = coef[q];
      seen[c] = true;
      scale = std::fmax(scale, std::fabs(coef[q]));
    }
    for (int q = 0; q < kK1Nnz; q++) {
      const double v = g_coef.k64.v[kK1Class[q] & 127];
      if (std::fabs(coef[q] - ((kK1Class[q] & 128) ? -v : v)) > 1e-12 * scale) g_coef.ok1 = false;
    }
    for (int c = 0; c < kK1Classes; c++) g_coef.ok1 = g_coef.ok1 && seen[c];
    for (int c = 0; c < kK1Classes; c++) g_coef.k32.v[c] = (float)g_coef.k64.v[c];
  }
}

bool tile_level1_available() {
  init_coef();
  return g_coef.ok1;
}

bool tile_fine_diag_available() {
  init_coef();
  return g_coef.ok0 && g_coef.diag0;
}

template <typename T>
static Blocks<T> fine_values() {
  if constexpr (sizeof(T) == 8) return g_coef.b64;
  else return g_coef.b32;
}

struct TileShape {
  int TY, TZ, NX, nty, ntz, ntx;
};

// tiles of up to ty x tz element columns
static void set_tiles(TileShape &s, const Level &L, int ty, int tz) {
  s.TY = std::max(2, std::min(L.nely + 1, ty));
  s.TZ = std::max(2, std::min(L.nelz + 1, tz));
  // a tile owns TY-1 node rows, plus the last row of the grid (its upper
  // neighbour element is halo)
  auto tiles = [](int nodes, int T) { return nodes <= T ? 1 : (nodes - T + T - 2) / (T - 1) + 1; };
  s.nty = tiles(L.ny, s.TY);
  s.ntz = tiles(L.nz, s.TZ);
}

static int device_cus() {
  static int ncu[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (!ncu[dev]) {
    int v = 0;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        v <= 0)
      v = 256;
    ncu[dev] = v;
  }
  return ncu[dev];
}

// The x-march length follows from the number of workgroups the device holds at
// once (`slots`): a launch that overflows them by a few workgroups pays a whole
// extra round, so NX is chosen to minimise rounds x (NX + 3), the per-workgroup
// cost in slab steps.  Sets
// the march length of a shape and the launch's cost in slab steps
static int64_t tile_x(TileShape &s, const Level &L, int nx_fixed, int64_t slots) {
  const int64_t yz = (int64_t)s.nty * s.ntz;
  int64_t best_cost = INT64_MAX;
  if (nx_fixed > 0) {
    s.NX = std::min(nx_fixed, L.nx);
  } else {
    int best = L.nx;
    for (int k = 1; k <= 8; k++) {
      const int64_t ntx = std::max<int64_t>(1, std::min<int64_t>(L.nx, k * slots / yz));
      const int nx = (int)((L.nx + ntx - 1) / ntx);
      const int64_t rounds = (((L.nx + nx - 1) / nx) * yz + slots - 1) / slots;
      const int64_t cost = rounds * (nx + 3);
      if (cost < best_cost) {
        best_cost = cost;
        best = nx;
      }
    }
    s.NX = best;
  }
  s.ntx = (L.nx + s.NX - 1) / s.NX;
  return best_cost;
}

// The last shapes that a thread's launches asked for, by the values they follow
// from: a search takes 2-4 us, as long as a small level's launch.
struct ShapeMemo {
  struct Entry {
    int nx = 0, ny = 0, nz = 0, kind = 0;
    int64_t slots = 0;
    TileShape s{};
  } e[8];
  int next = 0;
  template <typename F>
  const TileShape &get(const Level &L, int kind, int64_t slots, F search) {
    for (Entry &v : e)
      if (v.nx == L.nx && v.ny == L.ny && v.nz == L.nz && v.kind == kind && v.slots == slots)
        return v.s;
    Entry &v = e[next];
    next = (next + 1) % 8;
    v = Entry{L.nx, L.ny, L.nz, kind, slots, search()};
    return v.s;
  }
};
static thread_local ShapeMemo t_shapes;

// Level 1: tile of TY x TZ element columns marching over NX node planes.  LDS
// holds two exchange buffers of 9 values per thread (under 80 KiB).  Tuning
// override: TOP3D_TILE_L1=TY,TZ,NX (NX = 0: from the occupancy).
//
// Tiles of up to 256 threads, 4 waves, so that every SIMD has the same share of
// a workgroup, with the cheapest launch; among equals the least work, short rows
// counting for more.  65 x 7 (clipped to the grid) where its launch is cheaper,
// or as cheap with fewer waves on a CU.  Against 65 x 7 for every grid, us per
// sweep of the level below: FP32 512x256x256 84 -> 76.5 (23 x 11), 256x128x128
// 14.1 -> 13.8 (36 x 7), 168x72x104 8.9 -> 7.9 (37 x 6), 200x120x88 10.5 -> 9.3
// (21 x 12); FP64 178 -> 166 (28 x 9), 22.4 -> 22.0, 13.4 -> 10.1 and 15.9 ->
// 14.2; 65 x 7 stays in FP64 for 96x96x96 (9.5 us on 200 CUs; 10.1 with 28 x 9,
// of which 44 CUs have two) and 120x40x40 (5.2 us in 3 waves; 5.5 with 21 x 12).
static TileShape level1_search(const Level &L, int per_cu) {
  TileShape best{};
  const int64_t cus = device_cus();
  auto waves = [](const TileShape &t) { return (t.TY * t.TZ + 63) / 64; };
  // waves of the launch on the CU that has the most
  auto cu_waves = [&](const TileShape &t) {
    return ((int64_t)t.ntx * t.nty * t.ntz + cus - 1) / cus * waves(t);
  };
  int64_t best_cost = INT64_MAX, best_work = INT64_MAX;
  for (int ty = 17; ty <= 42; ty++) {
    TileShape s{};
    set_tiles(s, L, ty, 256 / std::min(ty, std::max(2, L.nely + 1)));
    const int64_t cost = tile_x(s, L, 0, per_cu * cus);
    const int64_t work = (int64_t)s.ntx * s.nty * s.ntz * (s.TY + 6) * 1024 / s.TY;
    if (cost < best_cost || (cost == best_cost && work <= best_work)) {
      best_cost = cost;
      best_work = work;
      best = s;
    }
  }
  TileShape wide{};
  set_tiles(wide, L, 65, 7);
  const int64_t cost = tile_x(wide, L, 0, std::max(1, per_cu / ((waves(wide) + 3) / 4)) * cus);
  if (cost < best_cost || (cost == best_cost && cu_waves(wide) < cu_waves(best))) best = wide;
  return best;
}

// per_cu: workgroups of 4 waves that a CU holds
static TileShape level1_shape(const Level &L, int elem_bytes, int per_cu) {
  const int lds_threads = 80 * 1024 / (18 * elem_bytes);
  // launch bounds: 1024 threads in FP32, 512 in FP64
  const int max_threads = std::min(elem_bytes == 4 ? 1024 : 512, lds_threads);
  const char *env = std::getenv("TOP3D_TILE_L1");
  int oy = 0, oz = 0, ox = 0;
  if (env && std::sscanf(env, "%d,%d,%d", &oy, &oz, &ox) == 3 && oy >= 2 && oz >= 2 && ox >= 0 &&
      oy <= max_threads && oz <= max_threads && oy * oz <= max_threads) {
    TileShape s{};
    set_tiles(s, L, oy, oz);
    // waves in fours: one SIMD holds ceil(waves / 4) of a workgroup
    tile_x(s, L, ox, std::max(1, per_cu / ((s.TY * s.TZ + 255) / 256)) * (int64_t)device_cus());
    return s;
  }
  // (the search asks for the device's CUs too)
  return t_shapes.get(L, 0, (int64_t)per_cu << 32 | device_cus(),
                      [&] { return level1_search(L, per_cu); });
}

// The fine level's shape (k_fine_march): (TY + 1) x (TZ + 1) nodes within the
// workgroup's threads, one of which holds the zeros.  At 257x129x129 nodes, in
// FP64, 23 x 9 columns ran a sweep in 81.6 us, 24 x 9 in 83.8 us, 20 x 11 in
// 85.5 us, 17 x 12 in 84.4 us, 17 x 13 in 87.9 us, 22 x 10, whose 97 tiles
// leave 7 slabs instead of 8, in 93.1 us, 15 x 15 and 26 x 8 likewise in 104
// us and 9 x 23, short rows, in 93.5 us; in FP32 33 x 14 in 32.7, 23 x 20 in
// 33.7, 20 x 23 in 34.2, 45 x 10 in 34.3, 26 x 17 and 38 x 12, which cost a slab
// more, in 36.7 and 37.6 us: rows of 17 to 23 columns, 35 in FP32, with the
// cheapest launch, the longest among equals.  Tuning override:
// TOP3D_TILE_L0 (FP32), TOP3D_TILE_L0_F64=TY,TZ,NX (NX = 0: the march length
// from the occupancy).
static TileShape march_search(const Level &L, int64_t slots, bool f64) {
  const int kNodes = (f64 ? march_threads<double>() : march_threads<float>()) - 1;
  TileShape best{};
  int64_t best_cost = INT64_MAX;
  for (int ty = 17; ty <= (f64 ? 23 : 35); ty++) {
    TileShape s{};
    set_tiles(s, L, ty, kNodes / (std::min(ty, std::max(2, L.nely + 1)) + 1) - 1);
    const int64_t cost = tile_x(s, L, 0, slots);
    if (cost <= best_cost) {
      best_cost = cost;
      best = s;
    }
  }
  return best;
}

static TileShape march_shape(const Level &L, int64_t slots, bool f64) {
  const int kNodes = (f64 ? march_threads<double>() : march_threads<float>()) - 1;
  const char *env = std::getenv(f64 ? "TOP3D_TILE_L0_F64" : "TOP3D_TILE_L0");
  int oy = 0, oz = 0, ox = 0;
  if (env && std::sscanf(env, "%d,%d,%d", &oy, &oz, &ox) == 3 && oy >= 2 && oz >= 2 && ox >= 0 &&
      oy <= kNodes && oz <= kNodes && (oy + 1) * (oz + 1) <= kNodes) {
    TileShape s{};
    set_tiles(s, L, oy, oz);
    tile_x(s, L, ox, slots);
    return s;
  }
  return t_shapes.get(L, f64 ? 2 : 1, slots, [&] { return march_search(L, slots, f64); });
}

// workgroups of `nthr` threads and `shm` bytes of LDS one CU holds at once.
// A workgroup's waves are dealt over the CU's 4 SIMDs, so one SIMD holds
// ceil(waves / 4) of them: two 9-wave workgroups need 6 wave slots on one
// SIMD.  (Measured: an FP32 fine sweep in 9-wave workgroups at 91 VGPRs, 5
// waves per SIMD, held one workgroup per CU and took 21% longer than at 79.)
static int wg_per_cu(const void *kernel, int nthr, size_t shm) {
  hipFuncAttributes at{};
  int per_simd = 4;
  if (hipFuncGetAttributes(&at, kernel) == hipSuccess && at.numRegs > 0)
    per_simd = std::max(1, std::min(8, 512 / ((at.numRegs + 7) / 8 * 8)));
  const int waves = (nthr + 63) / 64;
  const int by_waves = std::min(4 * per_simd / waves, per_simd / ((waves + 3) / 4));
  const int by_lds = (int)((160 * 1024) / std::max<size_t>(shm, 1));
  return std::max(1, std::min(by_waves, by_lds));
}

// checks that a level's offsets fit in 32 bits (the output's byte size also
// bounds the store offset that writes nothing, plus 16) and fills the
// kernels' arguments
template <typename T>
static bool tile_args(const Level &L, int64_t nmod, bool available, TileArgs &a) {
  if (!available) {
    set_error(TOP3D_ERR_ARG, "element matrix lacks the reflection structure");
    return false;
  }
  if ((int64_t)sizeof(T) * 3 * L.nodes() >= (int64_t(1) << 32) - 32 ||
      (int64_t)sizeof(T) * nmod >= (int64_t(1) << 32)) {
    set_error(TOP3D_ERR_ARG, "grid too large for 32-bit offsets (%lld nodes)",
              (long long)L.nodes());
    return false;
  }
  a.nelx = L.nelx;
  a.nely = L.nely;
  a.nelz = L.nelz;
  a.wy = L.wy;
  a.wz = L.wz;
  a.out_bytes = (uint32_t)(sizeof(T) * 3 * L.nodes());
  a.e_bytes = (uint32_t)(sizeof(T) * nmod);
  a.stream_out = 0;
  a.wx = L.wx;
  return true;
}

static void tile_args_shape(const TileShape &s, TileArgs &a) {
  a.TY = s.TY;
  a.TZ = s.TZ;
  a.NX = s.NX;
  a.nty = s.nty;
}

template <typename T>
static int run_fine(const DevGrid &g, int mode, const T *E, const T *in, T *out, const T *b,
                       const T *invD, T omega, int bcsym, double *dotp = nullptr,
                       int dot_cap = 0, void *aux = nullptr) {
  init_coef();
  const Level &L = g.lv[0];
  TileArgs a;
  if (!tile_args<T>(L, g.nelem, g_coef.ok0, a)) return 0;
  a.few = g.ewy;
  a.fez = g.ewz;
  a.E0 = g.E0;
  a.Emin = g.Emin;
  // the diagonal from the moduli needs a KE whose diagonal is one value per
  // component
  if (mode == kModeJacobiDiag && !g_coef.diag0) mode = kModeJacobi;
  const bool diag = mode == kModeJacobiDiag;
  const size_t shm = sizeof(T) * march_lds_values(diag) * (size_t)march_threads<T>();
  size_t coarse_lds = 0;  // the coarse plane of kModeProlong
  // workgroups per CU, [0] sweeps reading invD, [1] forming the diagonal
  static int per_cu[2] = {0, 0};
  if (!per_cu[diag])
    per_cu[diag] = wg_per_cu(diag ? (const void *)k_fine_march<T, kModeJacobiDiag, false>
                                  : (const void *)k_fine_march<T, kModeJacobi, false>,
                             march_threads<T>(), shm);
  const int64_t slots = (int64_t)per_cu[diag] * device_cus();
  TileShape s = march_shape(L, slots, sizeof(T) == 8);
  if (mode == kModeProlong) {  // (marches that start at odd planes)
    s.NX += s.NX & 1;
    s.ntx = (L.nx + s.NX - 1) / s.NX;
    const Level &C = g.lv[1];
    a.c_wx = C.wx;
    a.c_wy = C.wy;
    a.c_wz = C.wz;
    a.c_bytes = (uint32_t)(sizeof(T) * 3 * C.nodes());
    coarse_lds = sizeof(T) * 3 * (size_t)(s.TY / 2 + 3) * (s.TZ / 2 + 3);
  }
  tile_args_shape(s, a);
  // Past the caches where the launch reads no more than the memory-side cache
  // holds (256 MB) and with its output exceeds it: the output would push out
  // what the next launch reads again.  FP64, repeated: sweep of 256x128x128 (238
  // MB read, 341 in all) 79.5 against 84 us, apply of 320x128x128 (171 and 297
  // MB) 65 against 78; where the reads do not fit the store is slower, 113
  // against 110 us per sweep of 320x128x128 (297 and 424 MB), 218 against 200
  // per apply of 384x192x192 (465 and 807), as where all fits, 42.7 against 34.5
  // us per FP32 sweep of 256x128x128 (171 MB in all).
  const int64_t cache = int64_t(256) << 20;
  const int64_t reads = (mode == kModeFirst   ? 4
                         : mode == kModeProlong ? 7
                         : mode == kModeApply || mode == kModeApplyX ? 3
                         : mode == kModeJacobi ? 9
                                               : 6) *
                            (int64_t)a.out_bytes / 3 +
                        a.e_bytes;
  a.stream_out = reads <= cache && reads + a.out_bytes > cache;
  const dim3 grid(s.ntx, s.nty * s.ntz);
  const int bs = ((s.TY + 1) * (s.TZ + 1) + 63) / 64 * 64;
  const int nwg = s.ntx * s.nty * s.ntz;
  if (dotp && nwg > dot_cap) dotp = nullptr;
  const auto B = fine_values<T>();
#define T3D_LAUNCH(M, S)                                                                  \
  hipLaunchKernelGGL((k_fine_march<T, M, S>), grid, dim3(bs), shm + coarse_lds, stream(), a, B, \
                     E, in, out, b, invD, omega, g.fixmask[0], g.fixplane[0], dotp, aux)
  if (bcsym) {
    if (mode == kModeApply) T3D_LAUNCH(kModeApply, true);
    else if (mode == kModeJacobi) T3D_LAUNCH(kModeJacobi, true);
    else if (mode == kModeResidual) T3D_LAUNCH(kModeResidual, true);
    else if (mode == kModeFirst) T3D_LAUNCH(kModeFirst, true);
    else if (mode == kModeJacobiDiag) T3D_LAUNCH(kModeJacobiDiag, true);
    else if constexpr (sizeof(T) == 4) T3D_LAUNCH(kModeProlong, true);
  } else {
    if (mode == kModeApply) T3D_LAUNCH(kModeApply, false);
    else if (mode == kModeJacobi) T3D_LAUNCH(kModeJacobi, false);
    else if (mode == kModeResidual) T3D_LAUNCH(kModeResidual, false);
    else if (mode == kModeFirst) T3D_LAUNCH(kModeFirst, false);
    else if (mode == kModeJacobiDiag) T3D_LAUNCH(kModeJacobiDiag, false);
    else if constexpr (sizeof(T) == 4) T3D_LAUNCH(kModeProlong, false);
    else T3D_LAUNCH(kModeApplyX, false);
  }
#undef T3D_LAUNCH
  return dotp ? nwg : 0;
}

template <typename T>
static void run_level1(const DevGrid &g, int mode, const T *Eh, const T *in, T *out,
                          const T *b, const T *invD, T omega, int bcsym) {
  init_coef();
  const Level &L = g.lv[1];
  TileArgs a;
  if (!tile_args<T>(L, level1_moduli_count(g), g_coef.ok1, a)) return;
  a.few = L.nely + 1;  // the slots of k_level1_moduli
  a.fez = L.nelz + 1;
  if (mode == kModeJacobiDiag) mode = kModeJacobi;
  // workgroups of 4 waves per CU (their LDS, two buffers of 9 values per thread,
  // leaves room for all that the registers do)
  static const int per_cu = wg_per_cu((const void *)k_level1_sweep<T, kModeJacobi, false>, 256,
                                      sizeof(T) * 2 * 9 * 256);
  const TileShape s = level1_shape(L, (int)sizeof(T), per_cu);
  const int nthr = s.TY * s.TZ, bs = (nthr + 63) / 64 * 64;
  const size_t shm = sizeof(T) * 2 * 9 * (size_t)nthr;
  tile_args_shape(s, a);
  const dim3 grid(s.ntx, s.nty * s.ntz);
  K1Vals<T> B;
  if constexpr (sizeof(T) == 8) B = g_coef.k64; else B = g_coef.k32;
#define T3D_LAUNCH(M, S)                                                                    \
  hipLaunchKernelGGL((k_level1_sweep<T, M, S>), grid, dim3(bs), shm, stream(), a, B, Eh, in, \
                     out, b, invD, omega, g.fixmask[1], g.fixplane[1])
  if (bcsym) {
    if (mode == kModeApply) T3D_LAUNCH(kModeApply, true);
    else if (mode == kModeJacobi) T3D_LAUNCH(kModeJacobi, true);
    else T3D_LAUNCH(kModeResidual, true);
  } else {
    if (mode == kModeApply) T3D_LAUNCH(kModeApply, false);
    else if (mode == kModeJacobi) T3D_LAUNCH(kModeJacobi, false);
    else T3D_LAUNCH(kModeResidual, false);
  }
#undef T3D_LAUNCH
}

template <typename T>
void launch_fine_tile(const DevGrid &g, int mode, const T *E, const T *in, T *out,
                      const T *b, const T *invD, T omega, int bcsym) {
  run_fine<T>(g, mode, E, in, out, b, invD, omega, bcsym);
}

// out = K(x) in from the densities x, zero on the padded rows
void launch_fine_tile_apply_x(const DevGrid &g, const double *x, const double *in, double *out) {
  run_fine<double>(g, kModeApplyX, x, in, out, nullptr, nullptr, 0.0, 0);
}

// r = b - K u and its FP32 copy when r32 is given
void launch_fine_tile_residual(const DevGrid &g, const double *E, const double *u, double *r,
                               float *r32, const double *b, int bcsym) {
  run_fine<double>(g, kModeResidual, E, u, r, b, nullptr, 0.0, bcsym, nullptr, 0, r32);
}

int launch_fine_apply_dot(const DevGrid &g, const double *E, const double *p, double *q,
                          int bcsym, double *partials, int cap) {
  return run_fine<double>(g, kModeApply, E, p, q, nullptr, nullptr, 0.0, bcsym, partials,
                                cap);
}

template <typename T>
int launch_fine_tile_sweep_dot(const DevGrid &g, const T *E, const T *in, T *out, const T *b,
                               const T *invD, T omega, int bcsym, double *partials, int cap) {
  return run_fine<T>(g, kModeJacobiDiag, E, in, out, b, invD, omega, bcsym, partials, cap);
}
template int launch_fine_tile_sweep_dot<float>(const DevGrid &, const float *, const float *,
                                               float *, const float *, const float *, float, int,
                                               double *, int);
template int launch_fine_tile_sweep_dot<double>(const DevGrid &, const double *, const double *,
                                                double *, const double *, const double *, double,
                                                int, double *, int);

template <typename T>
void launch_level1_tile(const DevGrid &g, int mode, const T *Eh, const T *in, T *out,
                        const T *b, const T *invD, T omega, int bcsym) {
  run_level1<T>(g, mode, Eh, in, out, b, invD, omega, bcsym);
}

// Per level-1 element slot (i, k, j), i in 0..nelx+1, k in 0..nelz, j in
// 0..nely (y fastest): the 8-point Walsh-Hadamard transform of the moduli
// of its 8 fine elements (sub-cell o: x offset o & 1, y offset (o >> 1) & 1,
// z offset o >> 2), the form in which the level-1 sweep applies them; zero
// for the halo slots.  The moduli are fixed for a solve, so this runs once
// per solve instead of once per element step of every level-1 sweep.
template <typename T>
__global__ __launch_bounds__(256) void k_level1_moduli(int nelx, int nely, int nelz, int few,
                                                       int fez, const T *__restrict__ E,
                                                       T *__restrict__ Eh) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int sy = nely + 1, sz = nelz + 1;
  if (t >= (int64_t)(nelx + 2) * sz * sy) return;
  const int j = (int)(t % sy), k = (int)((t / sy) % sz), i = (int)(t / ((int64_t)sy * sz));
  T Eo[8];
#pragma unroll
  for (int o = 0; o < 8; o++) Eo[o] = 0;
  if (i >= 1 && i <= nelx && j >= 1 && k >= 1) {
#pragma unroll
    for (int o = 0; o < 8; o++) {
      const int64_t fe = ((int64_t)(2 * i - 1 + (o & 1)) * fez + (2 * k - 1 + (o >> 2))) * few +
                         (2 * j - 1 + ((o >> 1) & 1));
      Eo[o] = E[fe];
    }
  }
  T p1[8], p2[8], h[8];
#pragma unroll
  for (int o = 0; o < 8; o += 2) {
    p1[o] = Eo[o] + Eo[o + 1];
    p1[o + 1] = Eo[o] - Eo[o + 1];
  }
#pragma unroll
  for (int o = 0; o < 8; o += 4)
#pragma unroll
    for (int q = 0; q < 2; q++) {
      p2[o + q] = p1[o + q] + p1[o + q + 2];
      p2[o + q + 2] = p1[o + q] - p1[o + q + 2];
    }
#pragma unroll
  for (int q = 0; q < 4; q++) {
    h[q] = p2[q] + p2[q + 4];
    h[q + 4] = p2[q] - p2[q + 4];
  }
  T *pe = Eh + 8 * t;
#pragma unroll
  for (int o = 0; o < 8; o++) pe[o] = h[o];
}

int64_t level1_moduli_count(const DevGrid &g) {
  const Level &L = g.lv[1];
  return g.nl < 2 ? 0 : 8 * (int64_t)(L.nelx + 2) * (L.nely + 1) * (L.nelz + 1);
}

template <typename T>
void launch_level1_moduli(const DevGrid &g, const T *E, T *Eh) {
  const Level &L = g.lv[1];
  const int64_t n = level1_moduli_count(g) / 8;
  if (n <= 0) return;
  hipLaunchKernelGGL((k_level1_moduli<T>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     stream(), L.nelx, L.nely, L.nelz, g.ewy, g.ewz, E, Eh);
}
template void launch_level1_moduli<double>(const DevGrid &, const double *, double *);
template void launch_level1_moduli<float>(const DevGrid &, const float *, float *);

// First pre-smoothing sweep of the fine level from z = 0, with the diagonal
// formed from the moduli as in the kJacobiDiag sweep:
//   out = w b / (KE[c][c] sum of the node's 8 element moduli)  (real nodes),
//   out = w b at fixed DOFs, 0 on every other node.
// One thread per node of a node plane (blockIdx.y = plane).
template <typename TB, typename T>
__global__ __launch_bounds__(256) void k_jacobi_zero_fine(
    int nx, int ny, int nz, int wy, int wz, int few, int fez, const TB *__restrict__ b,
    const T *__restrict__ E, const uint8_t *__restrict__ fix, Blocks<T> B, T omega,
    T *__restrict__ out) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= wy * wz) return;
  const int j = t % wy, k = t / wy, i = blockIdx.y;
  const int64_t node = (int64_t)i * wz * wy + t;
  T *po = out + 3 * node;
  if (!(i >= 1 && i <= nx && j >= 1 && j <= ny && k >= 1 && k <= nz)) {
    po[0] = po[1] = po[2] = T(0);
    return;
  }
  // the node's elements: (i-1..i, j-1..j, k-1..k) in halo element indices
  auto slab = [&](int ie) {
    const int64_t e = ((int64_t)ie * fez + (k - 1)) * few + (j - 1);
    return ((E[e] + E[e + 1]) + E[e + few]) + E[e + few + 1];
  };
  const T rs = T(1) / (slab(i - 1) + slab(i));
  const uint8_t m = fix[node];
  const TB *pb = b + 3 * node;
#pragma unroll
  for (int c = 0; c < 3; c++) {
    const T dd = ((m >> c) & 1) ? T(1) : rs * B.ikd[c];
    po[c] = omega * dd * (T)pb[c];
  }
}

template <typename TB, typename T>
bool launch_fine_jacobi_zero(const DevGrid &g, const TB *b, const T *E, T omega, T *out) {
  if (!tile_fine_diag_available()) return false;
  const Level &L = g.lv[0];
  const Blocks<T> B = fine_values<T>();
  dim3 bs(256), gs((L.wy * L.wz + 255) / 256, L.wx);
  hipLaunchKernelGGL((k_jacobi_zero_fine<TB, T>), gs, bs, 0, stream(), L.nx, L.ny, L.nz, L.wy,
                     L.wz, g.ewy, g.ewz, b, E, g.fixmask[0], B, omega, out);
  return true;
}
// 1 / (sum of the node's 8 element moduli), 0 on nodes beyond the grid
template <typename T>
__global__ __launch_bounds__(256) void k_recip_moduli(int nx, int ny, int nz, int wy, int wz,
                                                      int few, int fez, const T *__restrict__ E,
                                                      T *__restrict__ rs) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= wy * wz) return;
  const int j = t % wy, k = t / wy, i = blockIdx.y;
  T v = 0;
  if (i >= 1 && i <= nx && j >= 1 && j <= ny && k >= 1 && k <= nz) {
    auto slab = [&](int ie) {
      const int64_t e = ((int64_t)ie * fez + (k - 1)) * few + (j - 1);
      return ((E[e] + E[e + 1]) + E[e + few]) + E[e + few + 1];
    };
    v = T(1) / (slab(i - 1) + slab(i));
  }
  rs[(int64_t)i * wz * wy + t] = v;
}

template <typename T>
void launch_recip_moduli(const DevGrid &g, const T *E, T *rs) {
  const Level &L = g.lv[0];
  dim3 bs(256), gs((L.wy * L.wz + 255) / 256, L.wx);
  hipLaunchKernelGGL((k_recip_moduli<T>), gs, bs, 0, stream(), L.nx, L.ny, L.nz, L.wy, L.wz,
                     g.ewy, g.ewz, E, rs);
}
template void launch_recip_moduli<float>(const DevGrid &, const float *, float *);
template void launch_recip_moduli<double>(const DevGrid &, const double *, double *);

// The first two sweeps from zero: x = omega b / diagonal (k_jacobi_zero_fine)
// is formed from b as the nodes are loaded, so that it is neither written nor
// read, and b, which the second sweep needs too, is read once.  In the V-cycle at
// 256x128x128 46 us FP32 and 86 us FP64 against 31 + 41 and 49 + 85 for the two.
template <typename T>
void launch_fine_first_sweeps(const DevGrid &g, const T *E, const T *rs, const T *b, T omega,
                              T *out, int bcsym) {
  run_fine<T>(g, kModeFirst, E, b, out, b, rs, omega, bcsym);
}
template void launch_fine_first_sweeps<float>(const DevGrid &, const float *, const float *,
                                              const float *, float, float *, int);
template void launch_fine_first_sweeps<double>(const DevGrid &, const double *, const double *,
                                               const double *, double, double *, int);

// out = a Jacobi sweep of z + P zc, zc the level-1 vector: the correction of the
// V-cycle is added as the nodes are loaded, the coarse planes interpolated from
// LDS.  In the V-cycle at 256x128x128 48.6 us against 25.6 + 40 for prolongation
// and sweep, at 512x256x256 346 against 189 + 302.  FP32 only: in FP64 it takes
// more than the 168 registers of three workgroups per CU (288 us against
// 62 + 85).
void launch_fine_prolong_sweep(const DevGrid &g, const float *E, const float *rs, const float *z,
                               const float *zc, const float *b, float omega, float *out,
                               int bcsym) {
  run_fine<float>(g, kModeProlong, E, z, out, b, rs, omega, bcsym, nullptr, 0,
                  const_cast<float *>(zc));
}

// Inverse diagonal of the fine operator from the moduli (KE_0's diagonal is
// one value per component): 1 / (KE[c][c] sum of the node's 8 element
// moduli) on real nodes, 1 at fixed DOFs, 0 elsewhere (the values of
// assembleInvertedMatrixDiagonalSubspace_halo, stencil_methods.c:693-773).
template <typename T>
__global__ __launch_bounds__(256) void k_invdiag_fine(int nx, int ny, int nz, int wy, int wz,
                                                      int few, int fez, const T *__restrict__ E,
                                                      const uint8_t *__restrict__ fix,
                                                      Blocks<T> B, T *__restrict__ invD) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= wy * wz) return;
  const int j = t % wy, k = t / wy, i = blockIdx.y;
  const int64_t node = (int64_t)i * wz * wy + t;
  T *po = invD + 3 * node;
  if (!(i >= 1 && i <= nx && j >= 1 && j <= ny && k >= 1 && k <= nz)) {
    po[0] = po[1] = po[2] = T(0);
    return;
  }
  auto slab = [&](int ie) {
    const int64_t e = ((int64_t)ie * fez + (k - 1)) * few + (j - 1);
    return ((E[e] + E[e + 1]) + E[e + few]) + E[e + few + 1];
  };
  const T rs = T(1) / (slab(i - 1) + slab(i));
  const uint8_t m = fix[node];
#pragma unroll
  for (int c = 0; c < 3; c++) po[c] = ((m >> c) & 1) ? T(1) : rs * B.ikd[c];
}

bool launch_fine_invdiag(const DevGrid &g, const double *E, double *invD) {
  if (!tile_fine_diag_available()) return false;
  const Level &L = g.lv[0];
  dim3 bs(256), gs((L.wy * L.wz + 255) / 256, L.wx);
  hipLaunchKernelGGL((k_invdiag_fine<double>), gs, bs, 0, stream(), L.nx, L.ny, L.nz, L.wy,
                     L.wz, g.ewy, g.ewz, E, g.fixmask[0], g_coef.b64, invD);
  return true;
}

template bool launch_fine_jacobi_zero<double, double>(const DevGrid &, const double *,
                                                      const double *, double, double *);
template bool launch_fine_jacobi_zero<float, float>(const DevGrid &, const float *,
                                                    const float *, float, float *);

// rows j > nely+1 of every (i, k) set to zero, as the reference's operator
// does for its padded y nodes (stencil_methods.c:407-418)
__global__ void k_zero_pad_rows(int64_t nrows, int wy, int first, double *__restrict__ out) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int npad = wy - first;
  if (t >= nrows * npad) return;
  const int64_t node = (t / npad) * wy + first + t % npad;
  out[3 * node] = out[3 * node + 1] = out[3 * node + 2] = 0.0;
}

void launch_zero_pad_rows(const DevGrid &g, double *out) {
  const Level &L = g.lv[0];
  const int first = L.nely + 2;
  if (first >= L.wy) return;
  const int64_t n = (int64_t)L.wx * L.wz * (L.wy - first);
  hipLaunchKernelGGL(k_zero_pad_rows, dim3((n + 255) / 256), dim3(256), 0, stream(),
                     (int64_t)L.wx * L.wz, L.wy, first, out);
}

template void launch_fine_tile<double>(const DevGrid &, int, const double *, const double *,
                                       double *, const double *, const double *, double, int);
template void launch_fine_tile<float>(const DevGrid &, int, const float *, const float *,
                                      float *, const float *, const float *, float, int);
template void launch_level1_tile<double>(const DevGrid &, int, const double *, const double *,
                                         double *, const double *, const double *, double, int);
template void launch_level1_tile<float>(const DevGrid &, int, const float *, const float *,
                                        float *, const float *, const float *, float, int);

}  // namespace t3d
