// Design-loop kernels: compliance and sensitivity, the density filter and
// its transpose, volume, change and the optimality-criteria update.
#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>

#include "t3d_internal.hpp"

namespace t3d {

constexpr int kBS = 256;
constexpr int kPartials = 1024;

__host__ __device__ constexpr int dn_x(int n) { return (n == 1 || n == 2 || n == 5 || n == 6) ? 1 : 0; }
__host__ __device__ constexpr int dn_y(int n) { return (n == 0 || n == 1 || n == 4 || n == 5) ? 1 : 0; }
__host__ __device__ constexpr int dn_z(int n) { return n >= 4 ? 1 : 0; }

__device__ __forceinline__ double blk_sum(double v) {
  __shared__ double sm[kBS / 64];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0;
  if (threadIdx.x == 0)
    for (int i = 0; i < kBS / 64; i++) s += sm[i];
  __syncthreads();
  return s;
}

__device__ __forceinline__ double blk_max(double v) {
  __shared__ double sm[kBS / 64];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_down(v, off, 64));
  if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0;
  if (threadIdx.x == 0)
    for (int i = 0; i < kBS / 64; i++) s = fmax(s, sm[i]);
  __syncthreads();
  return s;
}

__global__ void k_reduce_final(const double *__restrict__ partials, int n, int op,
                               double *__restrict__ out) {
  double s = 0;
  for (int i = threadIdx.x; i < n; i += blockDim.x)
    s = op ? fmax(s, partials[i]) : s + partials[i];
  s = op ? blk_max(s) : blk_sum(s);
  if (threadIdx.x == 0) *out = s;
}

// ---- compliance and sensitivity (stencil_methods.c:808-862) ---------------
// ce = u_e^T KE u_e; c = sum E(x_e) ce; dc_e = -3 (E0-Emin) x_e^2 ce.
__global__ __launch_bounds__(kBS) void k_sensitivity(
    int nelx, int nely, int nelz, int wy, int wz, int few, int fez, double E0, double Emin,
    const double *__restrict__ KE, const double *__restrict__ x,
    const double *__restrict__ u, double *__restrict__ dc, double *__restrict__ partials) {
  const int64_t ne = (int64_t)nelx * nely * nelz;
  double csum = 0.0;
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < ne;
       t += (int64_t)gridDim.x * blockDim.x) {
    const int j = (int)(t % nely) + 1, k = (int)((t / nely) % nelz) + 1,
              i = (int)(t / ((int64_t)nely * nelz)) + 1;
    double ue[24];
#pragma unroll
    for (int n = 0; n < 8; n++) {
      const int64_t nd = 3 * (((int64_t)(i + dn_x(n)) * wz + (k + dn_z(n))) * wy + (j + dn_y(n)));
      ue[3 * n] = u[nd];
      ue[3 * n + 1] = u[nd + 1];
      ue[3 * n + 2] = u[nd + 2];
    }
    double ce = 0.0;
#pragma unroll 4
    for (int r = 0; r < 24; r++) {
      double tr = 0.0;
#pragma unroll
      for (int c = 0; c < 24; c++) tr += KE[24 * r + c] * ue[c];
      ce += ue[r] * tr;
    }
    const int64_t e = ((int64_t)i * fez + k) * few + j;
    const double xe = x[e];
    csum += ce * (Emin + xe * xe * xe * (E0 - Emin));
    dc[e] = ce * (-3.0 * (E0 - Emin) * xe * xe);
  }
  csum = blk_sum(csum);
  if (threadIdx.x == 0) partials[blockIdx.x] = csum;
}

// The same quantities with u_e^T KE u_e = h^T (T KE T^T / 64) h, h = T u_e the
// per-component 8-point Walsh-Hadamard transform of the element's nodal
// values: 72 additions and 8 3x3 blocks instead of 576 multiply-adds with KE
// read per element.  Element coordinates in 32-bit arithmetic (ne < 2^31).
struct WhBlocks {
  double m[8][3][3];
};

__global__ __launch_bounds__(kBS) void k_sensitivity_wh(
    int nelx, int nely, int nelz, int wy, int wz, int few, int fez, double E0, double Emin,
    const WhBlocks B, const double *__restrict__ x, const double *__restrict__ u,
    double *__restrict__ dc, double *__restrict__ partials) {
  const uint32_t ne = (uint32_t)nelx * nely * nelz;
  double csum = 0.0;
  for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < ne; t += gridDim.x * blockDim.x) {
    const uint32_t ty = t / (uint32_t)nely, tz = ty / (uint32_t)nelz;
    const int j = (int)(t - ty * nely) + 1, k = (int)(ty - tz * nelz) + 1, i = (int)tz + 1;
    double h[8][3];  // [p][c], p = px | py << 1 | pz << 2
#pragma unroll
    for (int p = 0; p < 8; p++) {
      const int64_t nd =
          3 * (((int64_t)(i + (p & 1)) * wz + (k + (p >> 2))) * wy + (j + ((p >> 1) & 1)));
      h[p][0] = u[nd];
      h[p][1] = u[nd + 1];
      h[p][2] = u[nd + 2];
    }
#pragma unroll
    for (int bit = 1; bit < 8; bit <<= 1)
#pragma unroll
      for (int p = 0; p < 8; p++)
        if (!(p & bit))
#pragma unroll
          for (int c = 0; c < 3; c++) {
            const double a = h[p][c], b = h[p | bit][c];
            h[p][c] = a + b;
            h[p | bit][c] = a - b;
          }
    double ce = 0.0;
#pragma unroll
    for (int s = 0; s < 8; s++) {
      const double hs[3] = {h[s ^ 1][0], h[s ^ 2][1], h[s ^ 4][2]};
#pragma unroll
      for (int c = 0; c < 3; c++) {
        double tr = 0.0;
#pragma unroll
        for (int d = 0; d < 3; d++) tr += B.m[s][c][d] * hs[d];
        ce += hs[c] * tr;
      }
    }
    const int64_t e = ((int64_t)i * fez + k) * few + j;
    const double xe = x[e];
    csum += ce * (Emin + xe * xe * xe * (E0 - Emin));
    dc[e] = ce * (-3.0 * (E0 - Emin) * xe * xe);
  }
  csum = blk_sum(csum);
  if (threadIdx.x == 0) partials[blockIdx.x] = csum;
}

void launch_sensitivity(const DevGrid &g, const double *x, const double *u, double *dc,
                        double *partials, double *c) {
  const Level &L = g.lv[0];
  if (g.wh0 && (int64_t)L.nelx * L.nely * L.nelz < (int64_t)INT32_MAX) {
    WhBlocks B;
    std::memcpy(B.m, g.M0, sizeof(B.m));
    hipLaunchKernelGGL(k_sensitivity_wh, dim3(kPartials), dim3(kBS), 0, stream(), L.nelx,
                       L.nely, L.nelz, L.wy, L.wz, g.ewy, g.ewz, g.E0, g.Emin, B, x, u, dc,
                       partials);
  } else {
    hipLaunchKernelGGL(k_sensitivity, dim3(kPartials), dim3(kBS), 0, stream(), L.nelx, L.nely,
                       L.nelz, L.wy, L.wz, g.ewy, g.ewz, g.E0, g.Emin, g.KE[0], x, u, dc,
                       partials);
  }
  hipLaunchKernelGGL(k_reduce_final, dim3(1), dim3(kBS), 0, stream(), partials, kPartials, 0,
                     c);
}

// ---- density filter (stencil_optimization.c:228-395) ----------------------
// neighbourhood i2 in [i1-(ceil(r)-1), i1+ceil(r)] clipped to [1, nel],
// weight max(0, r - dist).
struct FilterWin {
  int lo, hi;
};
__device__ __forceinline__ FilterWin fwin(int i1, int cr, int nel) {
  return FilterWin{max(i1 - (cr - 1), 1), min(i1 + cr + 1, nel + 1)};
}

// MODE 0: out = (H rho)/Hs; MODE 1: out = v / Hs; MODE 2: out = H v
template <int MODE>
__global__ __launch_bounds__(kBS) void k_filter(int nelx, int nely, int nelz, int few,
                                                int fez, double rmin, int cr,
                                                const double *__restrict__ in,
                                                double *__restrict__ out) {
  const int64_t ne = (int64_t)nelx * nely * nelz;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= ne) return;
  const int j1 = (int)(t % nely) + 1, k1 = (int)((t / nely) % nelz) + 1,
            i1 = (int)(t / ((int64_t)nely * nelz)) + 1;
  const FilterWin wi = fwin(i1, cr, nelx), wk = fwin(k1, cr, nelz), wj = fwin(j1, cr, nely);
  double acc = 0.0, ws = 0.0;
  for (int i2 = wi.lo; i2 < wi.hi; i2++)
    for (int k2 = wk.lo; k2 < wk.hi; k2++)
      for (int j2 = wj.lo; j2 < wj.hi; j2++) {
        const int d2 = (i1 - i2) * (i1 - i2) + (j1 - j2) * (j1 - j2) + (k1 - k2) * (k1 - k2);
        const double w = fmax(0.0, rmin - sqrt((double)d2));
        if (MODE != 1) acc += w * in[((int64_t)i2 * fez + k2) * few + j2];
        ws += w;
      }
  const int64_t e1 = ((int64_t)i1 * fez + k1) * few + j1;
  if (MODE == 0) out[e1] = acc / ws;
  if (MODE == 1) out[e1] = in[e1] / ws;
  if (MODE == 2) out[e1] = acc;
}

// Radii up to 7: tiles in LDS.  The window's non-zero weights are those of
// the offsets with |d| < rmin, so |di|, |dk|, |dj| <= R = ceil(rmin) - 1, and
// a weight depends on the squared distance only (the expression above).  The
// elements outside the grid are staged as zeros; a weight that is zero is
// never applied.
constexpr int kFilterMaxR = 6;
constexpr int kFTK = 8, kFTJ = 32;  // tile in z and y, one thread per column
// what the filter does with the elements outside the grid
enum { kHaloKeep = 0, kHaloZero = 1, kHaloCopy = 2 };

// The workgroups at the grid's faces also write the halo elements beside
// their elements [i0, i1] x kFTK x kFTJ.
__device__ __forceinline__ void filter_write_halo(int i0, int i1, int k0, int j0, int nelx,
                                                  int nely, int nelz, int few, int fez, int halo,
                                                  const double *__restrict__ in,
                                                  double *__restrict__ out) {
  const int il = i0 == 1 ? 0 : i0, ih = i1 >= nelx ? nelx + 1 : i1;
  const int kl = k0 == 1 ? 0 : k0, kh = k0 + kFTK > nelz ? nelz + 1 : k0 + kFTK - 1;
  const int jl = j0 == 1 ? 0 : j0, jh = j0 + kFTJ > nely ? nely + 1 : j0 + kFTJ - 1;
  if (!(il == 0 || ih > nelx || kl == 0 || kh > nelz || jl == 0 || jh > nely)) return;
  const int nj = jh - jl + 1, nk = kh - kl + 1, ni = ih - il + 1;
  for (int q = threadIdx.x; q < ni * nk * nj; q += kFTK * kFTJ) {
    const int jj = jl + q % nj, kk = kl + (q / nj) % nk, ii = il + q / (nj * nk);
    if (ii >= 1 && ii <= nelx && kk >= 1 && kk <= nelz && jj >= 1 && jj <= nely) continue;
    const int64_t e = ((int64_t)ii * fez + kk) * few + jj;
    out[e] = halo == kHaloCopy ? in[e] : 0.0;
  }
}

// R = 1 (rmin <= 2, weights w0..w3 at squared distance 0..3).  A workgroup
// marches along x over ni element planes of its 32 x 8 columns, with the next
// plane's loads in flight and one barrier per plane.  Per plane a thread sums
// its 9 neighbours by in-plane distance,
//   A0 the element, A1 the 4 beside it, A2 the 4 corners,
// and an element's sum takes those of three planes,
//   w0 A0 + w1 (A1 + A0- + A0+) + w2 (A2 + A1- + A1+) + w3 (A2- + A2+).
// The sum of the weights Hs follows from the same counts of elements inside
// the grid (C1 of 4, C2 of 4, n of 2 planes).
// TR = false: out = (H in) / Hs; TR = true: out = H (in / Hs).
// Bound by the step of each plane (wait, barrier, nine LDS reads) rather than
// by its 16 bytes per element: 29 us (filter) and 30 us (transpose) at
// 256x128x128, where one thread per element with its window's loads and
// range checks took 43 us, and 20 us for the division and 41 us for the sums
// of the transpose, with a fill and two copies around them.
template <bool TR>
__global__ __launch_bounds__(kFTJ *kFTK) void k_filter_march(
    int nelx, int nely, int nelz, int few, int fez, int ni, double w0, double w1, double w2,
    double w3, const double *__restrict__ in, double *__restrict__ out, int halo) {
  constexpr int LJ = kFTJ + 2, LK = kFTK + 2, NS = LJ * LK, NT = kFTJ * kFTK;
  __shared__ double tile[2][NS];
  const int t = threadIdx.x;
  const int j0 = 1 + kFTJ * blockIdx.x, k0 = 1 + kFTK * blockIdx.y, i0 = 1 + ni * blockIdx.z;
  const int i1 = min(i0 + ni - 1, nelx);
  // Hs = base + n * slope at a column, n of the planes beside it in the grid
  auto column = [&](int k, int j, double &base, double &slope) {
    const double cj = (j > 1) + (j < nely), ck = (k > 1) + (k < nelz);
    const double c1 = cj + ck, c2 = cj * ck;
    base = w0 + (w1 * c1 + w2 * c2);
    slope = w1 + (w2 * c1 + w3 * c2);
  };
  auto planes = [&](int i) { return (double)((i > 1) + (i < nelx)); };
  // the one or two elements of a plane that this thread stages
  bool ok[2];
  int64_t off[2];
  double sb[2], ss[2], v[2];
#pragma unroll
  for (int e = 0; e < 2; e++) {
    const int q = t + e * NT;
    const int j = j0 - 1 + q % LJ, k = k0 - 1 + q / LJ;
    ok[e] = q < NS && k >= 1 && k <= nelz && j >= 1 && j <= nely;
    off[e] = ok[e] ? (int64_t)k * few + j : 0;
    if (TR) column(k, j, sb[e], ss[e]);
  }
  const int64_t plane = (int64_t)fez * few;
  auto load = [&](int i) {  // (planes 0 and nelx + 1 exist, and count as zero)
#pragma unroll
    for (int e = 0; e < 2; e++) v[e] = in[i * plane + off[e]];
  };
  const int tj = t % kFTJ, tk = t / kFTJ, j = j0 + tj, k = k0 + tk;
  const bool own = j <= nely && k <= nelz;
  double base, slope;
  column(k, j, base, slope);
  double am[3] = {0, 0, 0}, a0[3] = {0, 0, 0}, ap[3];
  load(i0 - 1);
  for (int p = i0 - 1; p <= i1 + 1; p++) {
    double *buf = tile[p & 1];
    const bool pin = p >= 1 && p <= nelx;
#pragma unroll
    for (int e = 0; e < 2; e++) {
      double x = ok[e] && pin ? v[e] : 0.0;
      if (TR) x /= ss[e] * planes(p) + sb[e];
      if (t + e * NT < NS) buf[t + e * NT] = x;
    }
    load(min(p + 1, i1 + 1));
    __syncthreads();
    const double *c = buf + (tk + 1) * LJ + tj + 1;
    ap[0] = c[0];
    ap[1] = (c[-1] + c[1]) + (c[-LJ] + c[LJ]);
    ap[2] = (c[-LJ - 1] + c[-LJ + 1]) + (c[LJ - 1] + c[LJ + 1]);
    const int i = p - 1;
    if (own && i >= i0 && i <= i1) {
      double acc = w0 * a0[0];
      if (w1 != 0.0) acc += w1 * (a0[1] + (am[0] + ap[0]));
      if (w2 != 0.0) acc += w2 * (a0[2] + (am[1] + ap[1]));
      if (w3 != 0.0) acc += w3 * (am[2] + ap[2]);
      out[i * plane + (int64_t)k * few + j] = TR ? acc : acc / (slope * planes(i) + base);
    }
#pragma unroll
    for (int q = 0; q < 3; q++) {
      am[q] = a0[q];
      a0[q] = ap[q];
    }
  }
  if (halo != kHaloKeep)
    filter_write_halo(i0, i1, k0, j0, nelx, nely, nelz, few, fez, halo, in, out);
}

// R >= 2.  A workgroup stages its kFTI x 8 x 32 elements (x, z, y) and R more
// on every side, and each thread sums the kFTI elements of one column along
// x.  The offsets (dk, dj) of one in-plane distance m share their weights, so
// their columns are added first (one LDS read and one addition per value) and
// the weights are applied once per m, to a column whose half length is the
// largest |di| with a weight.  The LDS reads bound it (rmin 3.5: 86 per
// element for 179 weights).  At 168x72x104, rmin 3.5: 54 us (filter) and 60
// us (transpose); a list of taps with the address arithmetic and the range
// check per tap took 1.05 ms, and 0.67 + 1.03 ms.
constexpr int kFTI = 8;
struct FilterClasses {
  double w2[3 * kFilterMaxR * kFilterMaxR + 1];  // weight at squared distance
  int16_t first[2 * kFilterMaxR * kFilterMaxR + 2];  // offsets of class n: first[n]..first[n+1]
  int8_t m[2 * kFilterMaxR * kFilterMaxR + 1], h[2 * kFilterMaxR * kFilterMaxR + 1];
  int8_t dk[(2 * kFilterMaxR + 1) * (2 * kFilterMaxR + 1)];
  int8_t dj[(2 * kFilterMaxR + 1) * (2 * kFilterMaxR + 1)];
  int count;
};

// The sum of the weights Hs depends only on how the window is clipped, per
// axis one of 2R + 1 classes of positions: the class of position p in 1..nel
// and a position of class c.
__device__ __forceinline__ int filter_class(int p, int nel, int R) {
  if (nel <= 2 * R + 1 || p - 1 < R) return p - 1;
  return nel - p < R ? 2 * R - (nel - p) : R;
}
__device__ __forceinline__ int filter_class_pos(int c, int nel, int R) {
  return (nel <= 2 * R + 1 || c <= R) ? c + 1 : nel - (2 * R - c);
}

// Hs of every class triple, one wavefront each
__global__ __launch_bounds__(64) void k_filter_sums(int R, int nelx, int nely, int nelz,
                                                    const FilterClasses W,
                                                    double *__restrict__ hs) {
  const int nc = 2 * R + 1, q = blockIdx.x;
  const int j1 = filter_class_pos(q % nc, nely, R), k1 = filter_class_pos((q / nc) % nc, nelz, R),
            i1 = filter_class_pos(q / (nc * nc), nelx, R);
  double ws = 0.0;
  for (int e = threadIdx.x; e < nc * nc * nc; e += 64) {
    const int dj = e % nc - R, dk = (e / nc) % nc - R, di = e / (nc * nc) - R;
    const bool in_grid = i1 + di >= 1 && i1 + di <= nelx && k1 + dk >= 1 && k1 + dk <= nelz &&
                         j1 + dj >= 1 && j1 + dj <= nely;
    if (in_grid) ws += W.w2[di * di + dk * dk + dj * dj];
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) ws += __shfl_down(ws, off, 64);
  // (a class beyond a narrow grid has no element)
  if (threadIdx.x == 0) hs[q] = i1 <= nelx && k1 <= nelz && j1 <= nely ? ws : 1.0;
}

// the offsets of one class, half length H
template <int H, int LD, int LJ>
__device__ __forceinline__ void filter_class_columns(const double *base, const FilterClasses &W,
                                                     int n, double (&acc)[kFTI]) {
  double w[H + 1], u[kFTI + 2 * H];
  const int m = W.m[n], q1 = W.first[n + 1];
#pragma unroll
  for (int d = 0; d <= H; d++) w[d] = W.w2[m + d * d];
#pragma unroll
  for (int p = 0; p < kFTI + 2 * H; p++) u[p] = 0.0;
#pragma unroll 2
  for (int q = W.first[n]; q < q1; q++) {
    const double *col = base + W.dk[q] * LJ + W.dj[q];
#pragma unroll
    for (int p = 0; p < kFTI + 2 * H; p++) u[p] += col[(p - H) * LD];
  }
#pragma unroll
  for (int p = 0; p < kFTI + 2 * H; p++)
#pragma unroll
    for (int o = 0; o < kFTI; o++) {
      const int d = p - H > o ? p - H - o : o - (p - H);
      if (d <= H) acc[o] += w[d] * u[p];
    }
}

// TR as in k_filter_march
template <bool TR, int R>
__global__ __launch_bounds__(kFTJ *kFTK) void k_filter_tile(
    int nelx, int nely, int nelz, int few, int fez, const FilterClasses W,
    const double *__restrict__ hs, const double *__restrict__ in, double *__restrict__ out,
    int halo) {
  constexpr int LI = kFTI + 2 * R, LK = kFTK + 2 * R, LJ = kFTJ + 2 * R;
  constexpr int NT = kFTJ * kFTK, NC = 2 * R + 1, LD = LK * LJ;
  __shared__ double tile[LI * LK * LJ];
  const int t = threadIdx.x;
  const int j0 = 1 + kFTJ * blockIdx.x, k0 = 1 + kFTK * blockIdx.y, i0 = 1 + kFTI * blockIdx.z;
  auto hsum = [&](int i, int k, int j) {
    return hs[(filter_class(i, nelx, R) * NC + filter_class(k, nelz, R)) * NC +
              filter_class(j, nely, R)];
  };
#pragma unroll 4
  for (int q = t; q < LI * LK * LJ; q += NT) {
    const int j = j0 - R + q % LJ, k = k0 - R + (q / LJ) % LK, i = i0 - R + q / LD;
    double v = 0.0;
    if (i >= 1 && i <= nelx && k >= 1 && k <= nelz && j >= 1 && j <= nely) {
      v = in[((int64_t)i * fez + k) * few + j];
      if (TR) v /= hsum(i, k, j);
    }
    tile[q] = v;
  }
  __syncthreads();
  const int tj = t % kFTJ, tk = t / kFTJ;
  double acc[kFTI];
#pragma unroll
  for (int o = 0; o < kFTI; o++) acc[o] = 0.0;
  const double *base = tile + (R * LK + tk + R) * LJ + tj + R;
#pragma unroll 1
  for (int n = 0; n < W.count; n++) {
    const int h = W.h[n];
    if (h == 0) filter_class_columns<0, LD, LJ>(base, W, n, acc);
    if (h == 1) filter_class_columns<1, LD, LJ>(base, W, n, acc);
    if (h == 2) filter_class_columns<2, LD, LJ>(base, W, n, acc);
    if constexpr (R >= 3)
      if (h == 3) filter_class_columns<3, LD, LJ>(base, W, n, acc);
    if constexpr (R >= 4)
      if (h == 4) filter_class_columns<4, LD, LJ>(base, W, n, acc);
    if constexpr (R >= 5)
      if (h == 5) filter_class_columns<5, LD, LJ>(base, W, n, acc);
    if constexpr (R >= 6)
      if (h == 6) filter_class_columns<6, LD, LJ>(base, W, n, acc);
  }
  const int j = j0 + tj, k = k0 + tk;
  if (j <= nely && k <= nelz) {
#pragma unroll
    for (int o = 0; o < kFTI; o++) {
      const int i = i0 + o;
      if (i <= nelx)
        out[((int64_t)i * fez + k) * few + j] = TR ? acc[o] : acc[o] / hsum(i, k, j);
    }
  }
  if (halo != kHaloKeep)
    filter_write_halo(i0, i0 + kFTI - 1, k0, j0, nelx, nely, nelz, few, fez, halo, in, out);
}

template <bool TR, int R>
static void filter_tile(const DevGrid &g, const FilterClasses &W, const double *hs,
                        const double *in, double *out, int halo) {
  const Level &L = g.lv[0];
  const dim3 grid((L.nely + kFTJ - 1) / kFTJ, (L.nelz + kFTK - 1) / kFTK,
                  (L.nelx + kFTI - 1) / kFTI);
  hipLaunchKernelGGL((k_filter_tile<TR, R>), grid, dim3(kFTJ * kFTK), 0, stream(), L.nelx,
                     L.nely, L.nelz, g.ewy, g.ewz, W, hs, in, out, halo);
}

static FilterClasses filter_classes(double rmin, int R) {
  FilterClasses W{};
  for (int d2 = 0; d2 <= 3 * R * R; d2++) W.w2[d2] = std::fmax(0.0, rmin - std::sqrt((double)d2));
  int q = 0;
  for (int m = 0; m <= 2 * R * R; m++) {
    int h = -1;
    while (h < R && W.w2[m + (h + 1) * (h + 1)] > 0.0) h++;
    if (h < 0) continue;
    const int q0 = q;
    for (int dk = -R; dk <= R; dk++)
      for (int dj = -R; dj <= R; dj++)
        if (dk * dk + dj * dj == m) {
          W.dk[q] = (int8_t)dk;
          W.dj[q++] = (int8_t)dj;
        }
    if (q == q0) continue;
    W.m[W.count] = (int8_t)m;
    W.h[W.count] = (int8_t)h;
    W.first[W.count++] = (int16_t)q0;
  }
  W.first[W.count] = (int16_t)q;
  return W;
}

// false where the loop over the window runs: no weight at all (rmin <= 0), a
// tile beyond the LDS (rmin > 7), a grid beyond the launch limits, or no memory
// for the sums of weights (the loop needs none).
template <bool TR>
static bool filter_tiles(DevGrid &g, double rmin, const double *in, double *out, int halo,
                         ScratchBlock &sums) {
  const Level &L = g.lv[0];
  if (!(rmin > 0.0) || rmin > kFilterMaxR + 1 || L.nelz > kFTK * 65535 || L.nelx > 65535)
    return false;
  const int R = std::max(1, (int)std::ceil(rmin) - 1);
  if (R == 1) {
    double w[4];
    for (int d2 = 0; d2 < 4; d2++) w[d2] = std::fmax(0.0, rmin - std::sqrt((double)d2));
    const int nty = (L.nely + kFTJ - 1) / kFTJ, ntz = (L.nelz + kFTK - 1) / kFTK;
    // planes per workgroup: four workgroups per CU, between 2 and 32 planes
    // (each march stages two planes more than it writes)
    const int ni = (int)std::max<int64_t>(
        2, std::min<int64_t>(32, (int64_t)nty * ntz * L.nelx / 1024));
    hipLaunchKernelGGL((k_filter_march<TR>), dim3(nty, ntz, (L.nelx + ni - 1) / ni),
                       dim3(kFTJ * kFTK), 0, stream(), L.nelx, L.nely, L.nelz, g.ewy, g.ewz, ni,
                       w[0], w[1], w[2], w[3], in, out, halo);
    return true;
  }
  const FilterClasses W = filter_classes(rmin, R);
  const int nc = 2 * R + 1, n = nc * nc * nc;
  static_assert((2 * kFilterMaxR + 1) * (2 * kFilterMaxR + 1) * (2 * kFilterMaxR + 1) <=
                    kOcScratchDoubles, "sums of weights");
  double *hs = sums.get();
  if (!hs) return false;
  hipLaunchKernelGGL(k_filter_sums, dim3(n), dim3(64), 0, stream(), R, L.nelx, L.nely, L.nelz, W,
                     hs);
  switch (R) {
    case 2: filter_tile<TR, 2>(g, W, hs, in, out, halo); break;
    case 3: filter_tile<TR, 3>(g, W, hs, in, out, halo); break;
    case 4: filter_tile<TR, 4>(g, W, hs, in, out, halo); break;
    case 5: filter_tile<TR, 5>(g, W, hs, in, out, halo); break;
    default: filter_tile<TR, 6>(g, W, hs, in, out, halo); break;
  }
  return true;
}

template <int MODE>
static void filter_window(const DevGrid &g, double rmin, const double *in, double *out) {
  const Level &L = g.lv[0];
  const dim3 grid((L.elements() + kBS - 1) / kBS);
  hipLaunchKernelGGL((k_filter<MODE>), grid, dim3(kBS), 0, stream(), L.nelx, L.nely, L.nelz,
                     g.ewy, g.ewz, rmin, (int)std::ceil(rmin), in, out);
}

// the halo elements of out before a window pass that leaves them
static void filter_halo(const DevGrid &g, const double *in, double *out, int halo) {
  if (halo == kHaloZero) launch_fill<double>(g.nelem, out, 0.0);
  if (halo == kHaloCopy)
    hipMemcpyAsync(out, in, sizeof(double) * g.nelem, hipMemcpyDeviceToDevice, stream());
}

void launch_filter(DevGrid &g, double rmin, const double *rho, double *out, int halo,
                   ScratchBlock &sums) {
  if (filter_tiles<false>(g, rmin, rho, out, halo, sums)) return;
  filter_halo(g, rho, out, halo);
  filter_window<0>(g, rmin, rho, out);
}

bool launch_filter_grad(DevGrid &g, double rmin, const double *v, double *out, int halo,
                        ScratchBlock &sums) {
  if (filter_tiles<true>(g, rmin, v, out, halo, sums)) return true;
  double *tmp = (double *)g.work(kSlotFilterTmp, sizeof(double) * g.nelem);
  if (!tmp) return false;
  launch_fill<double>(g.nelem, tmp, 0.0);
  filter_window<1>(g, rmin, v, tmp);
  filter_halo(g, v, out, halo);
  filter_window<2>(g, rmin, tmp, out);
  return true;
}

// ---- volume (gpu_definitions.c:94-110) ------------------------------------
__global__ __launch_bounds__(kBS) void k_volume(int nelx, int nely, int nelz, int few, int fez,
                                                const double *__restrict__ x,
                                                double *__restrict__ partials) {
  const int64_t ne = (int64_t)nelx * nely * nelz;
  double s = 0;
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < ne;
       t += (int64_t)gridDim.x * blockDim.x) {
    const int j = (int)(t % nely) + 1, k = (int)((t / nely) % nelz) + 1,
              i = (int)(t / ((int64_t)nely * nelz)) + 1;
    s += x[((int64_t)i * fez + k) * few + j];
  }
  s = blk_sum(s);
  if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

void launch_volume(const DevGrid &g, const double *x, double *partials, double *result) {
  const Level &L = g.lv[0];
  hipLaunchKernelGGL(k_volume, dim3(kPartials), dim3(kBS), 0, stream(), L.nelx, L.nely,
                     L.nelz, g.ewy, g.ewz, x, partials);
  hipLaunchKernelGGL(k_reduce_final, dim3(1), dim3(kBS), 0, stream(), partials, kPartials, 0,
                     result);
}

// ---- change = max |x - xnew|, then x = xnew (gpu_definitions.c:112-125) ----
__global__ __launch_bounds__(kBS) void k_change(int64_t n, double *__restrict__ x,
                                                const double *__restrict__ xnew,
                                                double *__restrict__ partials) {
  double m = 0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    m = fmax(m, fabs(x[i] - xnew[i]));
    x[i] = xnew[i];
  }
  m = blk_max(m);
  if (threadIdx.x == 0) partials[blockIdx.x] = m;
}

void launch_change(int64_t n, double *x, const double *xnew, double *partials, double *result) {
  hipLaunchKernelGGL(k_change, dim3(kPartials), dim3(kBS), 0, stream(), n, x, xnew, partials);
  hipLaunchKernelGGL(k_reduce_final, dim3(1), dim3(kBS), 0, stream(), partials, kPartials, 1,
                     result);
}

// ---- optimality criteria (gpu_definitions.c:127-157) ----------------------
// The bisection of gpu_definitions.c:127-157 evaluates one multiplier per
// pass over the elements.  Here a pass evaluates kOcCand = 31 multipliers that
// the loop would visit next, and the walk over their sums visits exactly the
// multipliers of the step-by-step loop:
//   l1 = 0 (no upward step yet): the 31 next halvings of l2, of which the
//     walk takes all up to the first upward step, so that one or two passes
//     replace the 30 to 60 steps from 1e9 down to the root's binade;
//   l1 > 0: the five levels of the bisection tree below [l1, l2].
// About 20 tree steps remain once l1 > 0, so an update takes 5 or 6 passes.
// (x_e sqrt(-dc_e / (dv_e lmid)) is formed as x_e sqrt(-dc_e / dv_e) times
// 1 / sqrt(lmid): one division and square root per element and pass.)
//
// A pass reads 24 bytes per element and spends 4 FP64 instructions per
// multiplier and element; at 31 multipliers the instructions bound it (35 us
// at 256x128x128, 18 of them the reads').  An update of that grid takes 6
// passes, 0.24 ms with the final write, against 0.66 ms for the 20 passes of 7
// multipliers (20.6 us each, and a one-workgroup walk of 6.6 us after each)
// that it replaced.  Fewer multipliers per pass come out even: a pass costs
// about 20 us more than 0.5 us per multiplier.  The walk over a pass's sums is done redundantly by every
// workgroup of the next kernel (kOcCand x kOcBlocks partial sums, 63 KB from
// the L2) instead of by a one-workgroup kernel in between.
constexpr int kOcDepth = 5;
constexpr int kOcCand = (1 << kOcDepth) - 1;
constexpr int kOcBS = 1024;     // threads: 16 waves, one workgroup per CU
constexpr int kOcBlocks = 256;
constexpr int kOcPasses = 6;    // passes between host checks
static_assert(kOcScratchDoubles >= 2 * (8 + kOcCand * kOcBlocks), "OC scratch size");

// xnew_e for a multiplier with rl = 1 / sqrt(lmid), a = x_e sqrt(-dc_e / dv_e):
// move limit 0.2, bounds [0, 1].
__device__ __forceinline__ double oc_x(double xi, double a, double rl) {
  const double move = 0.2;
  return fmax(0.0, fmax(xi - move, fmin(1.0, fmin(xi + move, a * rl))));
}

// The bisection state.  pending: the partial sums of the candidates of
// [l1, l2] are waiting to be walked.
struct OcState {
  double l1, l2, done, gval, lmid, steps, pending, unused;
};

// Candidates of [l1, l2]: for l1 = 0 candidate c is l2 halved c + 1 times;
// else heap order, node n with the lower half as child 2n+1 and the upper
// half as child 2n+2 (the path from the root is spelt by the bits of n + 1).
__device__ __forceinline__ double oc_candidate(double l1, double l2, int c) {
  if (l1 == 0.0) {
    double mid = 0.5 * (l2 + l1);
    for (int q = 0; q < c; q++) mid = 0.5 * (mid + l1);
    return mid;
  }
  double lo = l1, hi = l2, mid = 0.5 * (hi + lo);
  const int depth = 31 - __clz(c + 1);
  for (int d = depth - 1; d >= 0; d--) {
    if (((c + 1) >> d) & 1) lo = mid; else hi = mid;
    mid = 0.5 * (hi + lo);
  }
  return mid;
}

// The state after walking the pending sums (np partial sums per candidate),
// in LDS for every thread; S: kOcCand doubles of LDS.
__device__ __forceinline__ OcState oc_walk(const OcState *__restrict__ in,
                                           const double *__restrict__ partials, int np,
                                           double *S, OcState *st) {
  const OcState old = *in;
  if (old.done == 0.0 && old.pending != 0.0) {
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int c = w; c < kOcCand; c += kOcBS / 64) {
      double s = 0.0;
      for (int i = lane; i < np; i += 64) s += partials[c * np + i];
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
      if (lane == 0) S[c] = s;
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    OcState n = old;
    if (old.done == 0.0 && old.pending != 0.0) {
      const bool spine = old.l1 == 0.0;
      n.pending = 0.0;
      int node = 0;
      for (int d = 0; d < (spine ? kOcCand : kOcDepth); d++) {
        const double lmid = 0.5 * (n.l2 + n.l1);
        const bool up = S[node] + n.gval > 0;
        n.lmid = lmid;
        n.steps += 1.0;
        if (up) n.l1 = lmid; else n.l2 = lmid;
        node = spine ? node + 1 : 2 * node + (up ? 2 : 1);
        if (spine && !up && n.l2 > 0.0) continue;  // l1 = 0: the ratio is 1
        if (!((n.l2 - n.l1) / (n.l1 + n.l2) > 1e-6)) {
          n.done = 1.0;
          break;
        }
        if (spine && up) break;
      }
    }
    *st = n;
  }
  __syncthreads();
  return *st;
}

// One pass: walks the sums of the previous one, then leaves the partial sums
// of the new candidates.  state, partials: the two buffers of each, of which
// [cur] is read and [cur ^ 1] written (every workgroup reads the old ones).
// first: the state is [0, 1e9] with this gval.  A: where xnew overlaps none of
// the inputs, the first pass leaves x_e sqrt(-dc_e / dv_e) in xnew for the
// passes after it (57 of their some 180 instructions per element), which the
// final write replaces.
template <bool FIRST, bool A>
__global__ __launch_bounds__(kOcBS) void k_oc_pass(int64_t n, const double *x, const double *dv,
                                                   const double *dc, double *xnew,
                                                   double gval, OcState *state,
                                                   double *partials, int cur) {
  __shared__ double S[kOcCand + 1];
  __shared__ OcState sst;
  __shared__ double red[kOcBS / 64][kOcCand + 1];
  const int t = threadIdx.x, np = gridDim.x;
  OcState st;
  if (FIRST) {
    st = OcState{0.0, 1e9, 0.0, gval, 0.0, 0.0, 0.0, 0.0};
  } else {
    st = oc_walk(state + cur, partials + cur * kOcCand * kOcBlocks, np, S, &sst);
  }
  if (st.done == 0.0) st.pending = 1.0;
  if (blockIdx.x == 0 && t == 0) state[cur ^ 1] = st;
  if (st.done != 0.0) return;  // (uniform)
  __syncthreads();
  if (t < kOcCand) S[t] = 1.0 / sqrt(oc_candidate(st.l1, st.l2, t));
  __syncthreads();
  double rl[kOcCand], s[kOcCand + 1];  // (slot kOcCand: zero)
#pragma unroll
  for (int c = 0; c < kOcCand; c++) {
    // one value for the workgroup: kept in scalar registers
    const uint64_t b = __double_as_longlong(S[c]);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)b);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(b >> 32));
    rl[c] = __longlong_as_double(((uint64_t)hi << 32) | lo);
    s[c] = 0.0;
  }
  s[kOcCand] = 0.0;
  const double move = 0.2;
  const int64_t stride = (int64_t)gridDim.x * kOcBS;
  // two elements per step; past the end element i again, with weight 0
  for (int64_t i = (int64_t)blockIdx.x * kOcBS + t; i < n; i += 2 * stride) {
    double xe[2], ve[2], ae[2];
#pragma unroll
    for (int e = 0; e < 2; e++) {
      const int64_t j = e == 0 || i + stride < n ? i + e * stride : i;
      xe[e] = x[j];
      ve[e] = dv[j];
      ae[e] = A && !FIRST ? xnew[j] : dc[j];
    }
#pragma unroll
    for (int e = 0; e < 2; e++) {
      const bool in = e == 0 || i + stride < n;
      const double a = A && !FIRST ? ae[e] : xe[e] * sqrt(-ae[e] / ve[e]);
      if (A && FIRST && in) xnew[i + e * stride] = a;
      const double w = in ? ve[e] : 0.0;
      // oc_x less x_e: the bounds less x_e, and the multiply-add rounds once.
      // (Sums of dv xnew and dv x apart would lose an element's difference
      // beside the large dv x of elements that do not move.)
      const double hi = fmin(1.0, xe[e] + move) - xe[e], lo = fmax(0.0, xe[e] - move) - xe[e];
#pragma unroll
      for (int c = 0; c < kOcCand; c++)
        s[c] = fma(w, fmax(lo, fmin(hi, fma(a, rl[c], -xe[e]))), s[c]);
    }
  }
  // Wave sums of the 32 values by halving: at each step a lane keeps half of
  // its values and adds its partner's copies of them (32 exchanges instead of
  // 6 per value); lane l ends with the sum of value brev5(l & 31), over its
  // half of the wave, and the last exchange adds the other half.
  const int lane = t & 63;
#pragma unroll
  for (int h = 16; h > 0; h >>= 1) {
    const int bit = 16 / h;  // lane bits 1, 2, 4, 8, 16
    const bool upper = (lane & bit) != 0;
#pragma unroll
    for (int c = 0; c < h; c++) {
      const double give = upper ? s[c] : s[c + h], keep = upper ? s[c + h] : s[c];
      s[c] = keep + __shfl_xor(give, bit, 64);
    }
  }
  s[0] += __shfl_xor(s[0], 32, 64);
  if (lane < 32) red[t >> 6][__brev((unsigned)lane) >> 27] = s[0];
  __syncthreads();
  if (t < kOcCand) {
    double v = 0.0;
    for (int w = 0; w < kOcBS / 64; w++) v += red[w][t];
    partials[((cur ^ 1) * kOcCand) * kOcBlocks + (int64_t)t * np + blockIdx.x] = v;
  }
}

// xnew for the last multiplier the walk visited; the state for the host.
__global__ __launch_bounds__(kOcBS) void k_oc_write(int64_t n, const double *x, double *xnew,
                                                    const double *dv, const double *dc,
                                                    OcState *state, const double *partials,
                                                    int cur) {
  __shared__ double S[kOcCand + 1];
  __shared__ OcState sst;
  const OcState st =
      oc_walk(state + cur, partials + cur * kOcCand * kOcBlocks, gridDim.x, S, &sst);
  if (blockIdx.x == 0 && threadIdx.x == 0) state[cur ^ 1] = st;
  const double rl = 1.0 / sqrt(st.lmid);
  for (int64_t i = (int64_t)blockIdx.x * kOcBS + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kOcBS) {
    const double xi = x[i];
    xnew[i] = oc_x(xi, xi * sqrt(-dc[i] / dv[i]), rl);
  }
}

// Runs the bisection, checking on the host every kOcPasses passes (passes
// after convergence return at once).  xnew is written after each chunk for
// the last multiplier, so a converged chunk needs no further launch.
// scratch (kOcScratchDoubles doubles of device memory): its previous contents
// do not matter.  Returns the number of bisection steps or -1.
int oc_update(const double *x, double *xnew, const double *dv, const double *dc,
              int64_t nelem, double gval, double *scratch) {
  OcState *state = (OcState *)scratch;  // 2 of 8 doubles
  double *partials = scratch + 16;      // 2 x kOcCand x kOcBlocks
  const dim3 grid((unsigned)std::max<int64_t>(
      1, std::min<int64_t>(kOcBlocks, (nelem + kOcBS - 1) / kOcBS)));
  int cur = 0;
  OcState h{};
  auto apart = [&](const double *p) { return p + nelem <= xnew || xnew + nelem <= p; };
  // the first chunk only: the write after it replaces what a pass left there
  bool a = apart(x) && apart(dv) && apart(dc);
  for (int pass = 0; h.steps < 4096.0; a = false) {
    for (int q = 0; q < kOcPasses; q++, pass++, cur ^= 1) {
      auto *k = pass == 0 ? (a ? k_oc_pass<true, true> : k_oc_pass<true, false>)
                          : (a ? k_oc_pass<false, true> : k_oc_pass<false, false>);
      hipLaunchKernelGGL(k, grid, dim3(kOcBS), 0, stream(), nelem, x, dv, dc, xnew, gval, state,
                         partials, cur);
    }
    hipLaunchKernelGGL(k_oc_write, grid, dim3(kOcBS), 0, stream(), nelem, x, xnew, dv, dc, state,
                       partials, cur);
    cur ^= 1;
    if (!T3D_HIP(hipGetLastError()) ||
        !T3D_HIP(hipMemcpyAsync(&h, state + cur, sizeof(h), hipMemcpyDeviceToHost, stream())) ||
        !T3D_HIP(hipStreamSynchronize(stream())))
      return -1;
    if (h.done != 0.0) return (int)h.steps;
  }
  set_error(TOP3D_ERR_NO_CONVERGE, "update_solution: OC bisection did not converge in 4096 steps");
  return -1;
}

}  // namespace t3d
