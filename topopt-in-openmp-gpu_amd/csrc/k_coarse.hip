// Assembled coarse levels on the GPU (replacing the host CSR assembly of
// stencil_assembly.c:126-260 and the PCIe round trips of
// stencil_solvers.c:172-250).
//
// Level-l element matrices are built by Galerkin recursion,
//   Ke_l(E) = sum_{children c} Q_c^T Ke_{l-1}(c) Q_c,
// with Q_c the trilinear interpolation from the parent's 8 nodes to child
// c's nodes.  Because the reference's sub-cell matrices at level l use the
// fine elements' own quadrature points (local_matrix.c:268-293), this equals
// its sum_f E_f KE_l[f] exactly in exact arithmetic.  Element matrices are
// then gathered into a 27-point node stencil with symmetric elimination of
// the fixed DOFs (stencil_assembly.c:226-259), which serves the smoother
// levels and the dense coarsest matrix.
#include <mutex>

#include <rocblas/rocblas.h>

#include "t3d_internal.hpp"

namespace t3d {

__host__ __device__ constexpr int cn_x(int n) { return (n == 1 || n == 2 || n == 5 || n == 6) ? 1 : 0; }
__host__ __device__ constexpr int cn_y(int n) { return (n == 0 || n == 1 || n == 4 || n == 5) ? 1 : 0; }
__host__ __device__ constexpr int cn_z(int n) { return n >= 4 ? 1 : 0; }
__host__ __device__ constexpr int cn_of(int ox, int oy, int oz) {
  return oz * 4 + (oy ? (ox ? 1 : 0) : (ox ? 2 : 3));
}

// weight of parent node B at child c's node b (trilinear, per direction)
__device__ __forceinline__ double qweight(int cx, int cy, int cz, int b, int B) {
  const int p[3] = {cx + cn_x(b), cy + cn_y(b), cz + cn_z(b)};  // in half units 0..2
  const int q[3] = {cn_x(B), cn_y(B), cn_z(B)};
  double w = 1.0;
#pragma unroll
  for (int d = 0; d < 3; d++) {
    const double t = 0.5 * p[d];
    w *= q[d] ? t : 1.0 - t;
  }
  return w;
}

// One workgroup (576 threads, one per matrix entry) per parent element.
// SRC = 0: children are level-1 elements built from fine moduli and KE_1;
// SRC = 1: children are stored level-(l-1) element matrices.  The 8 children
// are staged in LDS together and the two products run for all of them
// between two barriers.
template <int SRC>
__global__ __launch_bounds__(576) void k_galerkin(
    int nelx, int nely, int nelz,        // parent level elements
    int cnely, int cnelz,                // child level elements (SRC = 1)
    int few, int fez, const double *__restrict__ KE1, const double *__restrict__ E,
    const double *__restrict__ Kchild, double *__restrict__ Kparent) {
  __shared__ double Kall[8 * 576];  // child matrices
  __shared__ double Tm[8 * 576];    // Kc Q_c per child
  __shared__ double Wq[8 * 64];     // Q_c: weight of parent node B at child node b, [c][b][B]
  const int t = threadIdx.x;
  const int r = t / 24, s = t % 24;
  const int64_t pe = blockIdx.x;  // compact parent index ((I*nelz + K)*nely + J), 0-based
  const int J = (int)(pe % nely);
  const int K = (int)((pe / nely) % nelz);
  const int I = (int)(pe / ((int64_t)nely * nelz));
  {
    double kv[8];
#pragma unroll
    for (int c = 0; c < 8; c++) {
      const int ci = 2 * I + cn_x(c), cj = 2 * J + cn_y(c), ck = 2 * K + cn_z(c);
      if (SRC == 0) {
        double v = 0.0;
        for (int ii = 0; ii < 2; ii++)
          for (int kk = 0; kk < 2; kk++)
            for (int jj = 0; jj < 2; jj++) {
              const int64_t fe = ((int64_t)(2 * ci + ii + 1) * fez + (2 * ck + kk + 1)) * few +
                                 (2 * cj + jj + 1);
              v += E[fe] * KE1[576 * (4 * ii + 2 * kk + jj) + t];
            }
        kv[c] = v;
      } else {
        kv[c] = Kchild[576 * (((int64_t)ci * cnelz + ck) * cnely + cj) + t];
      }
    }
#pragma unroll
    for (int c = 0; c < 8; c++) Kall[576 * c + t] = kv[c];
  }
  if (t < 512) {
    const int c = t >> 6, q = t & 63;
    Wq[t] = qweight(cn_x(c), cn_y(c), cn_z(c), q >> 3, q & 7);
  }
  __syncthreads();
  // Tm_c[a][S] = sum_b Kc[a][3b + cs] Q_c[b][Snode]
  {
    const int a = r, Sn = s / 3, cs = s % 3;
#pragma unroll 1
    for (int c = 0; c < 8; c++) {
      double v = 0.0;
#pragma unroll
      for (int b = 0; b < 8; b++)
        v += Kall[576 * c + 24 * a + 3 * b + cs] * Wq[64 * c + 8 * b + Sn];
      Tm[576 * c + t] = v;
    }
  }
  __syncthreads();
  // P[R][S] = sum_c sum_a Q_c[a][Rnode] Tm_c[3a + cr][S]
  double acc = 0.0;
  {
    const int Rn = r / 3, cr = r % 3;
#pragma unroll 1
    for (int c = 0; c < 8; c++) {
      double v = 0.0;
#pragma unroll
      for (int a = 0; a < 8; a++) v += Wq[64 * c + 8 * a + Rn] * Tm[576 * c + 24 * (3 * a + cr) + s];
      acc += v;
    }
  }
  Kparent[576 * pe + t] = acc;
}

// Level-2 element matrices as one GEMM on FP64 MFMA:
//   Ke2[e][q] = sum_{f<64} E[fine(e, f)] KE_2[f][q],  q < 576,
// with f = 16 ii + 4 kk + jj the reference's sub-cell index
// (local_matrix.c:283).  A workgroup owns kRows level-2 elements: their 64
// moduli are gathered into LDS, and each wave sweeps every 4th of the
// workgroup's 16-column tiles of KE_2 (36 over gridDim.y), holding the tile's
// 64x16 slice in registers while it runs over the 16-element row tiles
// (v_mfma_f64_16x16x4f64, K = 64).
// Few elements leave the device idle: 16 rows per workgroup and the columns
// over 9 or 3 workgroups took 8 us for 1024 elements and 25-28 us for 8192,
// against 71 and 80 us with 128 rows and all columns, and 39 us for 1024 with
// 64 rows.  From 32768 elements on the gather of the moduli, repeated by each
// column group, and the output's bandwidth decide: 64 rows and all columns
// took 1.0-1.2 ms for 524288 elements (2.4 GB) against 1.2-1.8 ms with 128
// rows, 1.5-1.8 with 16 and 3 groups.
// kCols: 576, or the kKeBlocks values of the node-pair blocks (58% of the
// products and of the output).
template <int kRows, int kCols>
__global__ __launch_bounds__(256) void k_elem_level2_mfma(
    int nelx, int nely, int nelz, int few, int fez, const double *__restrict__ KE2,
    const double *__restrict__ E, double *__restrict__ Ke2) {
  __shared__ double As[kRows][65];
  const int64_t nel = (int64_t)nelx * nely * nelz;
  const int64_t e0 = (int64_t)blockIdx.x * kRows;
  const int tid = threadIdx.x;
  for (int q = tid; q < kRows * 64; q += 256) {
    const int r = q >> 6, f = q & 63;
    const int64_t e = e0 + r;
    double v = 0.0;
    if (e < nel) {
      const int J = (int)(e % nely), K = (int)((e / nely) % nelz),
                I = (int)(e / ((int64_t)nely * nelz));
      const int ii = f >> 4, kk = (f >> 2) & 3, jj = f & 3;
      v = E[((int64_t)(4 * I + ii + 1) * fez + (4 * K + kk + 1)) * few + (4 * J + jj + 1)];
    }
    As[r][f] = v;
  }
  __syncthreads();
  const int w = tid >> 6, lane = tid & 63, li = lane & 15, lk = lane >> 4;
  typedef double double4_v __attribute__((ext_vector_type(4)));
  const int ntile = kCols / 16 / gridDim.y, nt1 = (blockIdx.y + 1) * ntile;
  for (int nt = blockIdx.y * ntile + w; nt < nt1; nt += 4) {
    double bfrag[16];
#pragma unroll
    for (int k = 0; k < 16; k++) bfrag[k] = KE2[(4 * k + lk) * kCols + 16 * nt + li];
#pragma unroll 2
    for (int mt = 0; mt < kRows / 16; mt++) {
      double4_v acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int k = 0; k < 16; k++)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(As[16 * mt + li][4 * k + lk], bfrag[k], acc,
                                                   0, 0, 0);
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int64_t e = e0 + 16 * mt + lk + 4 * v;
        if (e < nel) Ke2[e * kCols + 16 * nt + li] = acc[v];
      }
    }
  }
}

template <int kCols>
static void run_elem_level2(const DevGrid &g, const double *KE, const double *E, double *Ke) {
  const Level &L = g.lv[2];
  const int64_t nel = L.elements();
  constexpr int kMany = kCols == 576 ? 9 : 7;  // column groups (of the 36 or 21 tiles)
  if (nel < 32768)
    hipLaunchKernelGGL((k_elem_level2_mfma<16, kCols>),
                       dim3((nel + 15) / 16, nel <= 4096 ? kMany : 3), dim3(256), 0, stream(),
                       L.nelx, L.nely, L.nelz, g.ewy, g.ewz, KE, E, Ke);
  else
    hipLaunchKernelGGL((k_elem_level2_mfma<64, kCols>), dim3((nel + 63) / 64), dim3(256), 0,
                       stream(), L.nelx, L.nely, L.nelz, g.ewy, g.ewz, KE, E, Ke);
}

bool launch_elem_level2_blocks(const DevGrid &g, const double *E, double *Ke2b) {
  if (!g.KE2b) return false;
  run_elem_level2<kKeBlocks>(g, g.KE2b, E, Ke2b);
  return true;
}

void launch_elem_level2(const DevGrid &g, const double *E, double *Ke2) {
  const Level &L = g.lv[2];
  const int64_t nel = L.elements();
  if (g.KE2) {
    run_elem_level2<576>(g, g.KE2, E, Ke2);
    return;
  }
  hipLaunchKernelGGL((k_galerkin<0>), dim3(nel), dim3(576), 0, stream(), L.nelx,
                     L.nely, L.nelz, 0, 0, g.ewy, g.ewz, g.KE[1], E, nullptr, Ke2);
}

// Moduli of the 512 fine elements of each level-3 element, row e (compact
// level-3 element index (I*nelz + K)*nely + J), column f = 64 ii + 8 kk + jj
// (the sub-cell order of getKEsubspace, local_matrix.c:283).  One workgroup
// per kG3Run level-3 elements consecutive in y: it reads the 64 (ii, kk)
// rows of 8 kG3Run fine moduli (contiguous in E), and writes the elements'
// rows of Eg, which are consecutive, as one contiguous run from LDS (rows
// padded to 520 so that the row-wise LDS stores of the reads spread over
// the banks).
constexpr int kG3Run = 4;
constexpr int kG3Ld = 520;

__global__ __launch_bounds__(256) void k_gather_level3(int nelx, int nely, int nelz, int few,
                                                       int fez, const double *__restrict__ E,
                                                       double *__restrict__ Eg) {
  __shared__ double buf[kG3Run * kG3Ld];
  const int nrun = (nely + kG3Run - 1) / kG3Run;
  const int64_t ik = blockIdx.x / nrun;  // I * nelz + K
  const int J0 = kG3Run * (int)(blockIdx.x % nrun);
  const int K = (int)(ik % nelz), I = (int)(ik / nelz);
  const int nj = min(kG3Run, nely - J0);
  for (int q = threadIdx.x; q < 64 * 8 * kG3Run; q += blockDim.x) {
    const int row = q / (8 * kG3Run), c = q % (8 * kG3Run);  // row = 8 ii + kk
    if (c < 8 * nj) {
      const int fi = 8 * I + (row >> 3), fk = 8 * K + (row & 7), fj = 8 * J0 + c;
      buf[(c >> 3) * kG3Ld + 8 * row + (c & 7)] =
          E[((int64_t)(fi + 1) * fez + (fk + 1)) * few + (fj + 1)];
    }
  }
  __syncthreads();
  double *dst = Eg + (ik * nely + J0) * 512;
  for (int q = threadIdx.x; q < 512 * nj; q += blockDim.x)
    dst[q] = buf[(q >> 9) * kG3Ld + (q & 511)];
}

// one rocBLAS handle per device, created on first use
static rocblas_handle blas_handle() {
  static std::mutex mu;
  static rocblas_handle handles[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return nullptr;
  std::lock_guard<std::mutex> lk(mu);
  if (!handles[dev] && rocblas_create_handle(&handles[dev]) != rocblas_status_success)
    handles[dev] = nullptr;
  return handles[dev];
}

bool launch_elem_level3(const DevGrid &g, const double *E, double *Eg, double *Ke3) {
  const Level &L = g.lv[3];
  const int64_t nel = L.elements();
  if (!g.KE3 || nel <= 0 || nel > (int64_t)INT32_MAX / 576) return false;
  rocblas_handle h = blas_handle();
  if (!h || rocblas_set_stream(h, stream()) != rocblas_status_success) return false;
  const int64_t nwg = (int64_t)L.nelx * L.nelz * ((L.nely + kG3Run - 1) / kG3Run);
  hipLaunchKernelGGL(k_gather_level3, dim3((unsigned)nwg), dim3(256), 0, stream(), L.nelx,
                     L.nely, L.nelz, g.ewy, g.ewz, E, Eg);
  // row-major Ke3 [nel x 576] = Eg [nel x 512] KE_3 [512 x 576], i.e. in
  // column-major terms Ke3^T (576 x nel) = KE_3^T (576 x 512) Eg^T (512 x nel)
  const double one = 1.0, zero = 0.0;
  return rocblas_dgemm(h, rocblas_operation_none, rocblas_operation_none, 576, (rocblas_int)nel,
                       512, &one, g.KE3, 576, Eg, 512, &zero, Ke3, 576) ==
         rocblas_status_success;
}

void launch_elem_galerkin(const DevGrid &g, int l, const double *Kchild, double *Kparent) {
  const Level &L = g.lv[l], &C = g.lv[l - 1];
  hipLaunchKernelGGL((k_galerkin<1>), dim3(L.elements()), dim3(576), 0, stream(), L.nelx,
                     L.nely, L.nelz, C.nely, C.nelz, g.ewy, g.ewz, nullptr, nullptr, Kchild,
                     Kparent);
}

// 27-point stencil from element matrices, one thread per (node, neighbour):
// threadIdx.x = neighbour nb, kNsNodes consecutive nodes per workgroup, so
// that the threads of a node read the same three rows of each of its
// element matrices; the workgroup's 243 x kNsNodes values are staged in LDS
// and written as kNsNodes-long runs of each S plane.
// S[(nb*9 + r*3 + c) * nint + n]; symmetric elimination of fixed DOFs.
// bc_symmetric = 0 keeps the columns of fixed DOFs and only replaces fixed
// rows by identity rows (the matrix-free convention, stencil_methods.c:515-518).
constexpr int kNsNodes = 32;

__global__ __launch_bounds__(27 * kNsNodes) void k_node_stencil(
    int nelx, int nely, int nelz, int wy, int wz, const double *__restrict__ Ke,
    const uint8_t *__restrict__ fix, double *__restrict__ S, int bc_symmetric) {
  __shared__ double tile[243 * kNsNodes];
  const int64_t nx = nelx + 1, ny = nely + 1, nz = nelz + 1, nint = nx * ny * nz;
  const int nb = threadIdx.x;
  const int64_t n0 = (int64_t)blockIdx.x * kNsNodes;
  const int64_t n = n0 + threadIdx.y;
  const int nloc = (int)min((int64_t)kNsNodes, nint - n0);
  if (n < nint) {
    const int j = (int)(n % ny), k = (int)((n / ny) % nz), i = (int)(n / (ny * nz));
    const int dx = nb / 9 - 1, dz = (nb / 3) % 3 - 1, dy = nb % 3 - 1;
    const int i2 = i + dx, j2 = j + dy, k2 = k + dz;
    double v[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    const bool nb_in = i2 >= 0 && i2 < nx && j2 >= 0 && j2 < ny && k2 >= 0 && k2 < nz;
    if (nb_in) {
      for (int e = 0; e < 8; e++) {  // elements (0-based) containing node n
        const int ex = (e & 1) ? 0 : -1, ey = (e & 2) ? 0 : -1, ez = (e & 4) ? 0 : -1;
        const int ie = i + ex, je = j + ey, ke = k + ez;
        if (ie < 0 || ie >= nelx || je < 0 || je >= nely || ke < 0 || ke >= nelz) continue;
        const int ox = dx - ex, oy = dy - ey, oz = dz - ez;  // neighbour offset in element
        if (ox < 0 || ox > 1 || oy < 0 || oy > 1 || oz < 0 || oz > 1) continue;
        const int a = cn_of(-ex, -ey, -ez), b = cn_of(ox, oy, oz);
        const double *K = Ke + 576 * (((int64_t)ie * nelz + ke) * nely + je);
#pragma unroll
        for (int r = 0; r < 3; r++)
#pragma unroll
          for (int c = 0; c < 3; c++) v[3 * r + c] += K[24 * (3 * a + r) + 3 * b + c];
      }
      const uint8_t m1 = fix[((int64_t)(i + 1) * wz + (k + 1)) * wy + (j + 1)];
      const uint8_t m2 = fix[((int64_t)(i2 + 1) * wz + (k2 + 1)) * wy + (j2 + 1)];
      for (int r = 0; r < 3; r++)
        for (int c = 0; c < 3; c++) {
          const bool fr = (m1 >> r) & 1, fc = bc_symmetric && ((m2 >> c) & 1);
          if (fr || fc) v[3 * r + c] = (nb == 13 && r == c) ? 1.0 : 0.0;
        }
    }
#pragma unroll
    for (int q = 0; q < 9; q++) tile[(nb * 9 + q) * kNsNodes + threadIdx.y] = v[q];
  }
  __syncthreads();
  const int tid = threadIdx.y * blockDim.x + threadIdx.x;
  for (int e = tid; e < 243 * kNsNodes; e += blockDim.x * kNsNodes) {
    const int q = e / kNsNodes, nn = e % kNsNodes;
    if (nn < nloc) S[(int64_t)q * nint + n0 + nn] = tile[e];
  }
}

void launch_node_stencil(const DevGrid &g, int l, const double *Ke, double *S,
                         int bc_symmetric) {
  const Level &L = g.lv[l];
  const int64_t nint = L.interior_nodes();
  hipLaunchKernelGGL(k_node_stencil, dim3((unsigned)((nint + kNsNodes - 1) / kNsNodes)),
                     dim3(27, kNsNodes), 0, stream(), L.nelx, L.nely, L.nelz, L.wy, L.wz, Ke,
                     g.fixmask[l], S, bc_symmetric);
}

// The symmetric half layout of a matrix with symmetric elimination
// (kHalfPlanes planes): the 13 neighbours nb = 14..26 as full 3x3 blocks at
// planes (nb-14)*9 + 3r + c, the centre's upper triangle r <= c at planes
// 117 + half_centre_index(r, c); with S32 the FP32 form of the V-cycle, and of
// S the centre's diagonal, which the inverse diagonal is formed from.
// A node's 14 blocks are sums over 1 to 8 of its elements, 36 element blocks in
// all, each element block in the sum of one node: that of its first node in the
// order x, z, y, which is the neighbours' order too.  With the element's nodes
// numbered in that order the blocks of a node in one element are a run, so that
// consecutive threads load consecutive values; they meet in LDS, are summed in
// the order of the elements and written, 16 nodes to a plane.  Bound by memory
// (level 2 of 512x256x256, 1.4 GB of blocks and 0.3 GB of stencil, beside the
// first fine sweeps: 1.3-1.7 ms; a thread per element block took 2.9 ms, with
// every load in a line of its own, and a thread per neighbour, which loaded one
// element after the other, 24 bytes at a time, and wrote S in FP64 too, 2.3-2.8).
constexpr int kHsNodes = 16, kHsThreads = 512;
constexpr int kHsValues = 9 * 36, kHsLd = kHsValues + 1;
// x, z, y order of the node at (x, y, z) of an element
__host__ __device__ constexpr int ke_rank(int x, int y, int z) { return 4 * x + 2 * z + y; }

template <bool BLOCKS>
__global__ __launch_bounds__(kHsThreads) void k_node_stencil_half(
    int nelx, int nely, int nelz, int wy, int wz, const double *__restrict__ Ke,
    const uint8_t *__restrict__ fix, double *__restrict__ S, float *__restrict__ S32,
    uint32_t nblk) {
  __shared__ double val[kHsNodes * kHsLd];  // [node][ke_block(rank, .) of its element]
  __shared__ int elem[kHsNodes * 8];        // [node][its rank in the element]; -1: none
  __shared__ uint8_t mask[14 * kHsNodes];   // fixed DOFs of neighbour nb - 13
  // contiguous eighths of the nodes to the XCDs: a plane's line is written by
  // workgroups of one
  const uint32_t xcd = blockIdx.x & 7u;
  const uint32_t blk = xcd * (nblk >> 3) + min(xcd, nblk & 7u) + (blockIdx.x >> 3);
  const uint32_t nx = nelx + 1, ny = nely + 1, nz = nelz + 1, nint = nx * ny * nz;
  const uint32_t n0 = blk * kHsNodes;
  const int nloc = (int)min((uint32_t)kHsNodes, nint - n0);
  const int tid = threadIdx.x;
  {
    const int nn = tid & (kHsNodes - 1), it = tid / kHsNodes;
    const uint32_t n = min(n0 + nn, nint - 1);
    const int j = (int)(n % ny), k = (int)(n / ny % nz), i = (int)(n / (ny * nz));
    if (it < 8) {
      const int ie = i - (it >> 2), ke = k - ((it >> 1) & 1), je = j - (it & 1);
      const bool in = ie >= 0 && ie < nelx && je >= 0 && je < nely && ke >= 0 && ke < nelz;
      elem[nn * 8 + it] = in ? (ie * nelz + ke) * nely + je : -1;
    } else if (it < 8 + 14) {  // (neighbours beyond the grid are nodes of the halo)
      const int nb = 13 + it - 8, dx = nb / 9 - 1, dz = (nb / 3) % 3 - 1, dy = nb % 3 - 1;
      mask[(nb - 13) * kHsNodes + nn] =
          fix[((int64_t)(i + dx + 1) * wz + (k + dz + 1)) * wy + (j + dy + 1)];
    }
  }
  __syncthreads();
#pragma unroll
  for (int t = 0; t < (kHsNodes * kHsValues + kHsThreads - 1) / kHsThreads; t++) {
    const int o = tid + kHsThreads * t, nn = o / kHsValues, q = o - nn * kHsValues;
    if (nn < kHsNodes) {
      const int bq = q / 9;
      int ra = 0;  // the run that holds block bq
#pragma unroll
      for (int r = 1; r < 8; r++) ra += bq >= ke_block(r, r);
      const int e = elem[nn * 8 + ra];
      double v = 0.0;
      if (e >= 0) {
        if constexpr (BLOCKS) {
          v = Ke[(int64_t)kKeBlocks * e + q];
        } else {
          const int rb = bq - ke_block(ra, ra) + ra;
          const int a = cn_of(ra >> 2, ra & 1, (ra >> 1) & 1);
          const int b = cn_of(rb >> 2, rb & 1, (rb >> 1) & 1);
          v = Ke[576 * (int64_t)e + 24 * (3 * a + q % 9 / 3) + 3 * b + q % 3];
        }
      }
      val[nn * kHsLd + q] = v;
    }
  }
  __syncthreads();
  for (int o = tid; o < kHalfPlanes * kHsNodes; o += kHsThreads) {
    const int q = o / kHsNodes, m = o % kHsNodes;
    if (m >= nloc) continue;
    int nb = 13, r, c;
    if (q < 117) {
      nb = 14 + q / 9;
      r = (q % 9) / 3, c = q % 3;
    } else {  // upper triangle of the centre, row by row
      r = q < 120 ? 0 : q < 122 ? 1 : 2;
      c = q - (r == 0 ? 117 : r == 1 ? 119 : 120);
    }
    const int dx = nb / 9 - 1, dz = (nb / 3) % 3 - 1, dy = nb % 3 - 1;
    double v = 0.0;
#pragma unroll
    for (int e = 0; e < 8; e++) {  // the node at (x, y, z) of the element, (7 - e)'s bits
      const int x = 1 - (e & 1), y = 1 - (e >> 1 & 1), z = 1 - (e >> 2);
      const int x2 = x + dx, y2 = y + dy, z2 = z + dz;
      if (((x2 | y2 | z2) & ~1) == 0)  // the neighbour is a node of it
        v += val[m * kHsLd + 9 * ke_block(ke_rank(x, y, z), ke_rank(x2, y2, z2)) + 3 * r + c];
    }
    const bool diag = nb == 13 && r == c;
    if (((mask[m] >> r) | (mask[(nb - 13) * kHsNodes + m] >> c)) & 1) v = diag ? 1.0 : 0.0;
    if (!S32 || diag) S[(int64_t)q * nint + n0 + m] = v;
    if (S32) S32[(int64_t)q * nint + n0 + m] = (float)v;
  }
}

void launch_node_stencil_half(const DevGrid &g, int l, const double *Ke, double *S, float *S32,
                              bool blocks) {
  const Level &L = g.lv[l];
  const uint32_t nblk = (uint32_t)((L.interior_nodes() + kHsNodes - 1) / kHsNodes);
  const dim3 bs(kHsThreads);
  if (blocks)
    hipLaunchKernelGGL(k_node_stencil_half<true>, dim3(nblk), bs, 0, stream(), L.nelx, L.nely,
                       L.nelz, L.wy, L.wz, Ke, g.fixmask[l], S, S32, nblk);
  else
    hipLaunchKernelGGL(k_node_stencil_half<false>, dim3(nblk), bs, 0, stream(), L.nelx, L.nely,
                       L.nelz, L.wy, L.wz, Ke, g.fixmask[l], S, S32, nblk);
}

// the assembled coarsest level into the coarse factor's np x np storage
// (row-major; logical DOF d at storage index pos[d])
__global__ void k_stencil_to_dense(int nx, int ny, int nz, const double *__restrict__ S,
                                   const int *__restrict__ pos, double *__restrict__ A,
                                   int64_t np) {
  const int64_t nint = (int64_t)nx * ny * nz;
  const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (tid >= 27 * nint) return;
  const int nb = (int)(tid / nint);
  const int64_t p = tid % nint;
  const int j = (int)(p % ny), k = (int)((p / ny) % nz), i = (int)(p / ((int64_t)ny * nz));
  const int i2 = i + nb / 9 - 1, k2 = k + (nb / 3) % 3 - 1, j2 = j + nb % 3 - 1;
  if (i2 < 0 || i2 >= nx || j2 < 0 || j2 >= ny || k2 < 0 || k2 >= nz) return;
  const int64_t q = ((int64_t)i2 * nz + k2) * ny + j2;
  for (int r = 0; r < 3; r++)
    for (int c = 0; c < 3; c++)
      A[(int64_t)pos[3 * p + r] * np + pos[3 * q + c]] =
          S[(int64_t)(nb * 9 + 3 * r + c) * nint + p];
}

void launch_stencil_to_dense(const DevGrid &g, int l, const double *S, CoarseFactor &cf) {
  const Level &L = g.lv[l];
  cf.begin_assembly();
  const int64_t nthreads = 27 * L.interior_nodes();
  const int bs = 256;
  hipLaunchKernelGGL(k_stencil_to_dense, dim3((nthreads + bs - 1) / bs), dim3(bs), 0,
                     stream(), L.nx, L.ny, L.nz, S, cf.pos, cf.A, (int64_t)cf.np);
}

}  // namespace t3d
