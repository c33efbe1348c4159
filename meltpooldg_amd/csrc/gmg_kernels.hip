// Setup kernels of the multigrid preconditioner: the dense coarse-grid matrix
// assembled on the device from element matrices, and its in-place Gauss-Jordan
// inverse (the matrix is symmetric positive definite: no pivoting), blocked so
// that most of the work is a rank-32 update with the panels staged in LDS.
#include "blas.hpp"

namespace mpdg {

struct CoarseTables {
  double S[kMaxN1][kMaxN1], G[kMaxN1][kMaxN1], w[kMaxN1];
};

__device__ __forceinline__ bool constrained(long g, int nd0, int nd1, int nd2, int m) {
  const int ix = g % nd0, iy = (g / nd0) % nd1, iz = g / ((long)nd0 * nd1);
  return ((m & 1) && ix == 0) || ((m & 2) && ix == nd0 - 1) || ((m & 4) && iy == 0) ||
         ((m & 8) && iy == nd1 - 1) || ((m & 16) && iz == 0) || ((m & 32) && iz == nd2 - 1);
}

// One thread per (cell, I, J) entry of the element matrix
//   A_e[I][J] = sum_q m_q phi_I phi_J + k_cell grad phi_I . G_q grad phi_J,
// Cartesian cells: m_q = c_m vol W_q, G_q = diag(vol/h_d^2) W_q; mapped cells: m_q = c_m JxW_q,
// G_q = JxW_q B B^T, stored per cell in E[cell][I][J]; coarse_gather_kernel sums them into the
// dense row-major matrix A in a fixed order (no atomics); rows and columns of constrained DoFs
// are left out (their identity diagonal is set separately).
template <typename T>
__global__ __launch_bounds__(256) void coarse_matrix_kernel(CoarseTables t, int n1, int nc0, int nc1, long ncells,
                                                            int nd0, int nd1, int nd2, int dmask, double cm,
                                                            double ks0, double ks1, double ks2, double c_mass,
                                                            const double *__restrict__ kc, double kconst,
                                                            const T *__restrict__ metric, double *__restrict__ E) {
  const int nloc = n1 * n1 * n1, K = n1 - 1;
  const long gid = (long)blockIdx.x * 256 + threadIdx.x;
  if (gid >= ncells * nloc * nloc) return;
  const long cell = gid / ((long)nloc * nloc);
  const int e = (int)(gid - cell * nloc * nloc), I = e / nloc, J = e - I * nloc;
  const int cx = cell % nc0, cy = (cell / nc0) % nc1, cz = cell / ((long)nc0 * nc1);
  const int i0 = I % n1, i1 = (I / n1) % n1, i2 = I / (n1 * n1);
  const int j0 = J % n1, j1 = (J / n1) % n1, j2 = J / (n1 * n1);
  const double kap = kc ? kc[cell] : kconst;
  double acc = 0.0;
  for (int qz = 0; qz < n1; ++qz)
    for (int qy = 0; qy < n1; ++qy)
      for (int qx = 0; qx < n1; ++qx) {
        const double pI = t.S[qx][i0] * t.S[qy][i1] * t.S[qz][i2], pJ = t.S[qx][j0] * t.S[qy][j1] * t.S[qz][j2];
        const double a[3] = {t.G[qx][i0] * t.S[qy][i1] * t.S[qz][i2], t.S[qx][i0] * t.G[qy][i1] * t.S[qz][i2],
                             t.S[qx][i0] * t.S[qy][i1] * t.G[qz][i2]};
        const double b[3] = {t.G[qx][j0] * t.S[qy][j1] * t.S[qz][j2], t.S[qx][j0] * t.G[qy][j1] * t.S[qz][j2],
                             t.S[qx][j0] * t.S[qy][j1] * t.G[qz][j2]};
        if (metric) {
          auto M = [&](int comp) -> double { return metric[metric_at(n1, nc0, ncells, cell, comp, qx, qy, qz)]; };
          const double g00 = M(1), g01 = M(2), g11 = M(3), g02 = M(4), g12 = M(5), g22 = M(6);
          const double gg = a[0] * (g00 * b[0] + g01 * b[1] + g02 * b[2]) +
                            a[1] * (g01 * b[0] + g11 * b[1] + g12 * b[2]) +
                            a[2] * (g02 * b[0] + g12 * b[1] + g22 * b[2]);
          acc += c_mass * M(0) * pI * pJ + kap * gg;
        } else {
          const double W = t.w[qx] * t.w[qy] * t.w[qz];
          acc += W * (cm * pI * pJ + kap * (ks0 * a[0] * b[0] + ks1 * a[1] * b[1] + ks2 * a[2] * b[2]));
        }
      }
  E[gid] = acc;
}

// A[I][J] = sum over the cells holding both DoFs (z, y, x order) of E[cell][I_loc][J_loc];
// along each direction the cells holding node index x are c with K c <= x <= K c + K
__global__ __launch_bounds__(256) void coarse_gather_kernel(const double *__restrict__ E, int n1, int nc0, int nc1,
                                                            int nc2, int nd0, int nd1, int nd2, int dmask,
                                                            double *__restrict__ A) {
  const int K = n1 - 1, nloc = n1 * n1 * n1;
  const long n = (long)nd0 * nd1 * nd2;
  const long gid = (long)blockIdx.x * 256 + threadIdx.x;
  if (gid >= n * n) return;
  const long gI = gid / n, gJ = gid - gI * n;
  double acc = 0.0;
  if (!(dmask && (constrained(gI, nd0, nd1, nd2, dmask) || constrained(gJ, nd0, nd1, nd2, dmask)))) {
    const int ii[3] = {(int)(gI % nd0), (int)((gI / nd0) % nd1), (int)(gI / ((long)nd0 * nd1))};
    const int jj[3] = {(int)(gJ % nd0), (int)((gJ / nd0) % nd1), (int)(gJ / ((long)nd0 * nd1))};
    const int nc[3] = {nc0, nc1, nc2};
    int lo[3], hi[3];
    bool empty = false;
    for (int d = 0; d < 3; ++d) {
      const int mx = max(ii[d], jj[d]), mn = min(ii[d], jj[d]);
      lo[d] = max(0, (mx + K - 1) / K - 1);
      hi[d] = min(nc[d] - 1, mn / K);
      empty = empty || lo[d] > hi[d];
    }
    if (!empty)
      for (int cz = lo[2]; cz <= hi[2]; ++cz)
        for (int cy = lo[1]; cy <= hi[1]; ++cy)
          for (int cx = lo[0]; cx <= hi[0]; ++cx) {
            const long cell = cx + (long)nc0 * (cy + (long)nc1 * cz);
            const int I = (ii[0] - K * cx) + n1 * ((ii[1] - K * cy) + n1 * (ii[2] - K * cz));
            const int J = (jj[0] - K * cx) + n1 * ((jj[1] - K * cy) + n1 * (jj[2] - K * cz));
            acc += E[(cell * nloc + I) * nloc + J];
          }
  }
  A[gid] = acc;
}

__global__ __launch_bounds__(256) void coarse_dirichlet_kernel(double *A, long n, int nd0, int nd1, int nd2,
                                                               int dmask) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i < n && constrained(i, nd0, nd1, nd2, dmask)) A[i * n + i] = 1.0;
}

template <typename T>
int launch_coarse_matrix(const OperatorData<T> &od, double c_mass, const double *kc, double kconst, double *A,
                         double *E, hipStream_t s) {
  const FE1D &fe = fe1d(od.degree);
  CoarseTables t{};
  for (int a = 0; a < fe.n1; ++a) {
    t.w[a] = fe.qw[a];
    for (int b = 0; b < fe.n1; ++b) {
      t.S[a][b] = fe.S[a][b];
      t.G[a][b] = fe.G[a][b];
    }
  }
  const long n = od.n_dofs, nloc = (long)fe.n1 * fe.n1 * fe.n1, work = od.n_cells * nloc * nloc;
  const double vol = od.h[0] * od.h[1] * od.h[2];
  hipLaunchKernelGGL(coarse_matrix_kernel<T>, dim3((work + 255) / 256), dim3(256), 0, s, t, fe.n1, od.nc[0],
                     od.nc[1], od.n_cells, od.nd[0], od.nd[1], od.nd[2], od.dmask, c_mass * vol,
                     vol / (od.h[0] * od.h[0]), vol / (od.h[1] * od.h[1]), vol / (od.h[2] * od.h[2]), c_mass, kc,
                     kconst, od.metric, E);
  hipLaunchKernelGGL(coarse_gather_kernel, dim3((n * n + 255) / 256), dim3(256), 0, s, E, fe.n1, od.nc[0], od.nc[1],
                     od.nc[2], od.nd[0], od.nd[1], od.nd[2], od.dmask, A);
  if (od.dmask)
    hipLaunchKernelGGL(coarse_dirichlet_kernel, dim3((n + 255) / 256), dim3(256), 0, s, A, n, od.nd[0], od.nd[1],
                       od.nd[2], od.dmask);
  return hipGetLastError() == hipSuccess ? MPDG_OK : MPDG_ERR_DEVICE;
}

// Blocked in-place Gauss-Jordan inversion. For the diagonal block [k0, k0 + nb) of the current
// matrix [[A11, A12], [A21, A22]] one step writes
//   A11 <- A11^-1,  A12 <- A11^-1 A12,  A22 <- A22 - A21 A11^-1 A12,  A21 <- -A21 A11^-1
// (the scalar step with 1x1 blocks is the textbook in-place Gauss-Jordan); after the last block
// the array holds A^-1. Two launches per block: both panels (the old column panel is kept in old_col), and the
// rank-nb update of everything outside the block's rows and columns, whose workgroup with the next
// diagonal block inverts that too. What bounds it: the chain of launches, each a few microseconds of
// latencies on a few workgroups. n = 729: 23 blocks in 0.74 ms; four launches per block, with the panels by
// one thread per row or column and the diagonal block by a workgroup with two barriers per pivot, took
// 2.0 ms and were the longest part of a multigrid update.
constexpr int kGJB = 32;    // block width
constexpr int kGJTile = 64;  // update tile (64 x 64 per workgroup, 4 x 4 per thread)

// Inverse of the nb x nb block in D (padded with the identity) into A, by the first wavefront: lane = 32 (half of
// the columns) + row, 16 values in registers; the pivot row goes through LDS
__device__ __forceinline__ void gjb_invert_block(double (&D)[kGJB][kGJB + 1], double (&R)[kGJB], double *A, int n, int k0, int nb) {
  const int lane = threadIdx.x, i = lane & 31, h = lane >> 5;
  if (lane >= 64) return;
  double a[16];
#pragma unroll
  for (int m = 0; m < 16; ++m) a[m] = i < nb && 16 * h + m < nb ? D[i][16 * h + m] : (i == 16 * h + m ? 1.0 : 0.0);
#pragma unroll
  for (int k = 0; k < kGJB; ++k) {
    if (i == k) {
#pragma unroll
      for (int m = 0; m < 16; ++m) R[16 * h + m] = a[m];
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const double piv = 1.0 / R[k], mine = a[k % 16], other = __shfl_xor(mine, 32);
    const double f = (h == k / 16 ? mine : other) * piv, scale = i == k ? piv : 1.0, g = i == k ? 0.0 : f;
#pragma unroll
    for (int m = 0; m < 16; ++m) a[m] = fma(-g, R[16 * h + m], a[m] * scale);
    if (h == k / 16) a[k % 16] = i == k ? piv : -f;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
#pragma unroll
  for (int m = 0; m < 16; ++m)
    if (i < nb && 16 * h + m < nb) A[(long)(k0 + i) * n + k0 + 16 * h + m] = a[m];
}

__global__ __launch_bounds__(256) void gjb_diag_kernel(double *A, int n, int nb) {
  __shared__ double D[kGJB][kGJB + 1], R[kGJB];
  for (int e = threadIdx.x; e < nb * nb; e += 256) {
    const int i = e / nb, j = e - i * nb;
    D[i][j] = A[(long)i * n + j];
  }
  __syncthreads();
  gjb_invert_block(D, R, A, n, 0, nb);
}

// A12 <- A11^-1 A12 (workgroups 0 .. tiles - 1, 32 columns each) and A21 <- -A21 A11^-1 with the old A21 to old_col
// (n x 32; the other workgroups, 32 rows each)
__global__ __launch_bounds__(256) void gjb_panel_kernel(double *A, double *old_col, int n, int k0, int nb, int tiles) {
  __shared__ double D[kGJB][kGJB + 1], X[kGJB][kGJB + 1];
  const bool rows = (int)blockIdx.x < tiles;  // the row panel
  const int t0 = kGJB * (rows ? blockIdx.x : blockIdx.x - tiles), c = threadIdx.x & 31, g = threadIdx.x >> 5;
  if (t0 == k0) return;
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const int r = g + 8 * m;
    D[r][c] = r < nb && c < nb ? A[(long)(k0 + r) * n + k0 + c] : 0.0;
    if (rows) {
      X[r][c] = r < nb && t0 + c < n ? A[(long)(k0 + r) * n + t0 + c] : 0.0;
    } else {
      X[r][c] = t0 + r < n && c < nb ? A[(long)(t0 + r) * n + k0 + c] : 0.0;
      if (t0 + r < n) old_col[(long)(t0 + r) * kGJB + c] = X[r][c];
    }
  }
  __syncthreads();
  double s[4] = {};
#pragma unroll 8
  for (int q = 0; q < kGJB; ++q)
#pragma unroll
    for (int m = 0; m < 4; ++m) s[m] += rows ? D[g + 8 * m][q] * X[q][c] : X[g + 8 * m][q] * D[q][c];
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const int r = g + 8 * m;
    if (rows) {
      if (r < nb && t0 + c < n) A[(long)(k0 + r) * n + t0 + c] = s[m];
    } else {
      if (t0 + r < n && c < nb) A[(long)(t0 + r) * n + k0 + c] = -s[m];
    }
  }
}

// A22 <- A22 - (old A21) A12 for rows and columns outside the block (A12 already updated); then the next block's
// inverse
__global__ __launch_bounds__(256) void gjb_update_kernel(double *A, const double *old_col, int n, int k0, int nb) {
  __shared__ double Ct[kGJB][kGJTile + 1], Rt[kGJB][kGJTile + 1], D[kGJB][kGJB + 1], R[kGJB];
  const int i0 = blockIdx.y * kGJTile, j0 = blockIdx.x * kGJTile;
  for (int e = threadIdx.x; e < kGJTile * kGJB; e += 256) {
    const int ii = e / kGJB, c = e - ii * kGJB, i = i0 + ii;
    Ct[c][ii] = i < n && c < nb && !(i >= k0 && i < k0 + nb) ? old_col[(long)i * kGJB + c] : 0.0;
  }
  for (int e = threadIdx.x; e < kGJTile * kGJB; e += 256) {
    const int c = e / kGJTile, jj = e - c * kGJTile;
    Rt[c][jj] = (j0 + jj < n && c < nb) ? A[(long)(k0 + c) * n + j0 + jj] : 0.0;
  }
  const int ty = threadIdx.x / 16, tx = threadIdx.x - ty * 16;
  auto outside = [&](int i, int j) {
    return i < n && j < n && !(i >= k0 && i < k0 + nb) && !(j >= k0 && j < k0 + nb);
  };
  double v[4][4];
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int i = i0 + ty + 16 * m, j = j0 + tx + 16 * p;
      v[m][p] = outside(i, j) ? A[(long)i * n + j] : 0.0;
    }
  __syncthreads();
  double acc[4][4] = {};
#pragma unroll 8
  for (int c = 0; c < kGJB; ++c) {
    double a[4], b[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      a[m] = Ct[c][ty + 16 * m];
      b[m] = Rt[c][tx + 16 * m];
    }
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int p = 0; p < 4; ++p) acc[m][p] = fma(a[m], b[p], acc[m][p]);
  }
  const int k1 = k0 + kGJB, nb1 = min(kGJB, n - k1);
  const bool next = i0 == j0 && k1 < n && k1 >= i0 && k1 < i0 + kGJTile;  // (blocks do not straddle tiles)
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int i = i0 + ty + 16 * m, j = j0 + tx + 16 * p;
      const double x = v[m][p] - acc[m][p];
      if (next && i >= k1 && i < k1 + nb1 && j >= k1 && j < k1 + nb1) D[i - k1][j - k1] = x;
      else if (outside(i, j)) A[(long)i * n + j] = x;
    }
  if (next) {  // (uniform)
    __syncthreads();
    gjb_invert_block(D, R, A, n, k1, nb1);
  }
}

size_t gauss_jordan_scratch(int n) { return (size_t)n * kGJB; }
int launch_gauss_jordan_inverse(double *A, double *scratch, int n, hipStream_t s) {
  const int tiles = (n + kGJB - 1) / kGJB, bt = (n + kGJTile - 1) / kGJTile;
  hipLaunchKernelGGL(gjb_diag_kernel, dim3(1), dim3(256), 0, s, A, n, std::min(kGJB, n));
  for (int k0 = 0; k0 < n && tiles > 1; k0 += kGJB) {
    const int nb = std::min(kGJB, n - k0);
    hipLaunchKernelGGL(gjb_panel_kernel, dim3(2 * tiles), dim3(256), 0, s, A, scratch, n, k0, nb, tiles);
    hipLaunchKernelGGL(gjb_update_kernel, dim3(bt, bt), dim3(256), 0, s, A, scratch, n, k0, nb);
  }
  return hipGetLastError() == hipSuccess ? MPDG_OK : MPDG_ERR_DEVICE;
}

template int launch_coarse_matrix<double>(const OperatorData<double> &, double, const double *, double, double *,
                                          double *, hipStream_t);
template int launch_coarse_matrix<float>(const OperatorData<float> &, double, const double *, double, double *,
                                         double *, hipStream_t);

}  // namespace mpdg
