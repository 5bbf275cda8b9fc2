// mfm_sync.hip -- coarse-fine synchronisation of a level pair on the device:
// the flux register of the coarse-fine interface (increments from the coarse
// and fine face fluxes, reflux into the coarse cells next to the fine
// region) and the average of the fine level down onto the coarse cells it
// covers.  FP64, no FMA contraction.
#include "mfm_fill.hpp"

namespace mfm {
namespace {
constexpr int kSB = 256;
// Components per thread: blockIdx.y takes a chunk of them.  An interface has
// only some ten thousand faces, too few threads to fill the chip with one
// thread walking every component of a face, one after the other.
// Two levels of 343 boxes of 16^3 cells, 23 components (zero, coarse and two
// fine increments, reflux, average down): 340 -> 183 us.
constexpr int kSyncComps = 4;

__device__ __forceinline__ long off3(const FillFab& F, int i, int j, int k) {
  return (long)(i - F.lo[0]) +
         (long)F.n[0] * ((long)(j - F.lo[1]) + (long)F.n[1] * (long)(k - F.lo[2]));
}

// Register values are stored component-major: reg[c * ne + e].
__global__ __launch_bounds__(kSB) void k_reg_zero(double* reg, long n) {
  const long t = (long)blockIdx.x * kSB + threadIdx.x;
  if (t < n) reg[t] = 0.0;
}

// reg -= scale * F_coarse at the face (the coarse side of the register)
__global__ __launch_bounds__(kSB) void k_reg_coarse(const RegFace* __restrict__ E, long ne,
                                                   const FillFab* __restrict__ F, int dims,
                                                   double* __restrict__ reg, int nc,
                                                   double scale) {
  const long t = (long)blockIdx.x * kSB + threadIdx.x;
  if (t >= ne) return;
  const RegFace e = E[t];
  const FillFab f = F[e.cb * dims + e.d];
  int fc[3] = {e.c[0], e.c[1], e.c[2]};
  if (e.sigma > 0) fc[e.d] += 1;
  const double* p = f.p + off3(f, fc[0], fc[1], fc[2]);
  const int c0 = (int)blockIdx.y * kSyncComps, c1 = min(c0 + kSyncComps, nc);
  for (int c = c0; c < c1; ++c) {
    const double x = scale * p[c * f.cs];
    reg[c * ne + t] = reg[c * ne + t] - x;
  }
}

// reg += (scale / r^(dims-1)) * F_fine over the fine faces covering the
// coarse face, the first transverse direction fastest.
__global__ __launch_bounds__(kSB) void k_reg_fine(const RegFace* __restrict__ E, long ne,
                                                 const FillFab* __restrict__ F, int dims,
                                                 int r, double* __restrict__ reg, int nc,
                                                 double scale) {
  const long t = (long)blockIdx.x * kSB + threadIdx.x;
  if (t >= ne) return;
  const RegFace e = E[t];
  const FillFab f = F[e.fb * dims + e.d];
  int tr[2] = {-1, -1}, nt = 0;
  for (int d = 0; d < dims; ++d)
    if (d != e.d) tr[nt++] = d;
  double denom = 1.0;
  for (int q = 0; q < dims - 1; ++q) denom *= r;
  const double sc = scale / denom;
  const int n2 = nt > 1 ? r : 1;
  const int c0 = (int)blockIdx.y * kSyncComps, c1 = min(c0 + kSyncComps, nc);
  for (int c = c0; c < c1; ++c) {
    double acc = reg[c * ne + t];
    for (int q2 = 0; q2 < n2; ++q2)
      for (int q1 = 0; q1 < r; ++q1) {
        int fi[3] = {e.f0[0], e.f0[1], e.f0[2]};
        fi[tr[0]] += q1;
        if (nt > 1) fi[tr[1]] += q2;
        const double x = sc * f.p[off3(f, fi[0], fi[1], fi[2]) + c * f.cs];
        acc = acc + x;
      }
    reg[c * ne + t] = acc;
  }
}

// U += (scale * sigma * invvol) * reg for each register face of the cell,
// in the face list order (direction, then low face before high face).
__global__ __launch_bounds__(kSB) void k_reflux(const RegCell* __restrict__ C, long ncell,
                                               const RegFace* __restrict__ E, long ne,
                                               const FillFab* __restrict__ U,
                                               const double* __restrict__ reg, int nc,
                                               double scale, double invvol) {
  const long t = (long)blockIdx.x * kSB + threadIdx.x;
  if (t >= ncell) return;
  const RegCell g = C[t];
  const RegFace e0 = E[g.e0];
  const FillFab u = U[e0.cb];
  double* p = u.p + off3(u, e0.c[0], e0.c[1], e0.c[2]);
  const int c0 = (int)blockIdx.y * kSyncComps, c1 = min(c0 + kSyncComps, nc);
  for (int c = c0; c < c1; ++c) {
    double v = p[c * u.cs];
    for (int e = g.e0; e < g.e1; ++e) {
      const double f = scale * (double)E[e].sigma * invvol;
      v = v + f * reg[c * ne + e];
    }
    p[c * u.cs] = v;
  }
}

// averagewithvolumes (src/CoarseAverageExtF.ChF:10-50) into the coarse cell.
// RR: the refinement ratio when it is 2 (the children's loads then leave
// together), 0: any.
template <int RR, int DIMS>
__global__ __launch_bounds__(kSB) void k_average_down(const AvgRect* __restrict__ R, int nr,
                                                     const FillFab* __restrict__ Uc,
                                                     const FillFab* __restrict__ Uf, int nc,
                                                     int ratio, double vol) {
  const int bx = blockIdx.x;
  int lo = 0, hi = nr - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (R[mid].blk0 <= bx) lo = mid; else hi = mid - 1;
  }
  const AvgRect a = R[lo];
  const unsigned t = (unsigned)(bx - a.blk0) * kSB + threadIdx.x;
  const unsigned n01 = (unsigned)a.n[0] * a.n[1];
  if (t >= n01 * a.n[2]) return;
  const int k = (int)(t / n01);
  const unsigned rem = t - (unsigned)k * n01;
  const int j = (int)(rem / (unsigned)a.n[0]);
  const int i = (int)(rem - (unsigned)j * a.n[0]);
  const int ic[3] = {a.lo[0] + i, a.lo[1] + j, a.lo[2] + k};
  const FillFab uc = Uc[a.cb], uf = Uf[a.fb];
  const int r = RR > 0 ? RR : ratio;
  const int rz = DIMS == 3 ? r : 1;
  const int fz0 = DIMS == 3 ? ic[2] * r : ic[2];
  const double* f0 = uf.p + off3(uf, ic[0] * r, ic[1] * r, fz0);
  double* d0 = uc.p + off3(uc, ic[0], ic[1], ic[2]);
  const long sy = uf.n[0], sz = (long)uf.n[0] * uf.n[1];
  const int c0 = (int)blockIdx.y * kSyncComps, c1 = min(c0 + kSyncComps, nc);
  if constexpr (RR == 2) {
    constexpr int NZ = DIMS == 3 ? 2 : 1;
    double v[kSyncComps][NZ][2][2];
#pragma unroll
    for (int q = 0; q < kSyncComps; ++q) {
      const double* p = f0 + min(c0 + q, nc - 1) * uf.cs;
#pragma unroll
      for (int kk = 0; kk < NZ; ++kk)
#pragma unroll
        for (int jj = 0; jj < 2; ++jj)
#pragma unroll
          for (int ii = 0; ii < 2; ++ii) v[q][kk][jj][ii] = p[ii + jj * sy + kk * sz];
    }
#pragma unroll
    for (int q = 0; q < kSyncComps; ++q) {
      double sum = 0.0, volc = 0.0;
#pragma unroll
      for (int kk = 0; kk < NZ; ++kk)
#pragma unroll
        for (int jj = 0; jj < 2; ++jj)
#pragma unroll
          for (int ii = 0; ii < 2; ++ii) {
            const double x = vol * v[q][kk][jj][ii];
            sum = sum + x;
            volc = volc + vol;
          }
      if (c0 + q < nc) d0[(c0 + q) * uc.cs] = sum / volc;
    }
    return;
  }
  for (int c = c0; c < c1; ++c) {
    double sum = 0.0, volc = 0.0;
    for (int kk = 0; kk < rz; ++kk)
      for (int jj = 0; jj < r; ++jj)
        for (int ii = 0; ii < r; ++ii) {
          const double x = vol * f0[ii + jj * sy + kk * sz + c * uf.cs];
          sum = sum + x;
          volc = volc + vol;
        }
    d0[c * uc.cs] = sum / volc;
  }
}

unsigned comp_blocks(int nc) { return (unsigned)((nc + kSyncComps - 1) / kSyncComps); }
}  // namespace

hipError_t launch_reg_zero(double* reg, long n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_reg_zero, dim3((unsigned)((n + kSB - 1) / kSB)), dim3(kSB), 0, s, reg, n);
  return hipGetLastError();
}

hipError_t launch_reg_coarse(const RegFace* E, long ne, const FillFab* F, int dims,
                             double* reg, int nc, double scale, hipStream_t s) {
  if (ne <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_reg_coarse, dim3((unsigned)((ne + kSB - 1) / kSB), comp_blocks(nc)),
                     dim3(kSB), 0, s, E, ne, F, dims, reg, nc, scale);
  return hipGetLastError();
}

hipError_t launch_reg_fine(const RegFace* E, long ne, const FillFab* F, int dims, int r,
                           double* reg, int nc, double scale, hipStream_t s) {
  if (ne <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_reg_fine, dim3((unsigned)((ne + kSB - 1) / kSB), comp_blocks(nc)),
                     dim3(kSB), 0, s, E, ne, F, dims, r, reg, nc, scale);
  return hipGetLastError();
}

hipError_t launch_reflux(const RegCell* C, long ncell, const RegFace* E, long ne,
                         const FillFab* U, const double* reg, int nc, double scale,
                         double invvol, hipStream_t s) {
  if (ncell <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_reflux, dim3((unsigned)((ncell + kSB - 1) / kSB), comp_blocks(nc)),
                     dim3(kSB), 0, s, C, ncell, E, ne, U, reg, nc, scale, invvol);
  return hipGetLastError();
}

hipError_t launch_average_down(const AvgRect* R, int nr, int nblk, const FillFab* Uc,
                               const FillFab* Uf, int nc, int dims, int r, double vol,
                               hipStream_t s) {
  if (nr <= 0 || nblk <= 0) return hipSuccess;
  const dim3 grid((unsigned)nblk, comp_blocks(nc)), block(kSB);
  if (dims == 3) {
    if (r == 2) hipLaunchKernelGGL((k_average_down<2, 3>), grid, block, 0, s, R, nr, Uc, Uf, nc, r, vol);
    else hipLaunchKernelGGL((k_average_down<0, 3>), grid, block, 0, s, R, nr, Uc, Uf, nc, r, vol);
  } else if (r == 2) {
    hipLaunchKernelGGL((k_average_down<2, 2>), grid, block, 0, s, R, nr, Uc, Uf, nc, r, vol);
  } else {
    hipLaunchKernelGGL((k_average_down<0, 2>), grid, block, 0, s, R, nr, Uc, Uf, nc, r, vol);
  }
  return hipGetLastError();
}

}  // namespace mfm
