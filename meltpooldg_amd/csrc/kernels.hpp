// Shared declarations of the HIP kernels and their host launchers.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "../../include/mpdg_heat.h"
#include "fe1d.hpp"

namespace mpdg {

enum KappaMode { KAPPA_CONST = MPDG_KAPPA_CONST, KAPPA_QP = MPDG_KAPPA_QP, KAPPA_CELL = MPDG_KAPPA_CELL, KAPPA_LAW = MPDG_KAPPA_LAW };
enum LawId { LAW_TANH = MPDG_LAW_TANH, LAW_MUSHY = MPDG_LAW_MUSHY };

// tanh |x| = -E / (E + 2) with E = e^y - 1 = 2^n (e^r - 1) + (2^n - 1), y = -2 |x|, r = y - n ln 2 (ln 2 in two
// parts after Cody and Waite, e^r - 1 by its Taylor series on |r| <= ln 2 / 2): small x keep their relative accuracy, and the
// rounding errors of e^r - 1, E and E + 2 are carried into the quotient's correction. Largest error over 4M
// arguments |x| <= 25, in units of 2^-53 (2^-24) of the result: 1.16 (FP32 1.4), the device library's 1.34
// (2.33). The law is evaluated at every point of every apply, and the library's tanh and the division by
// the width took a third to a half of it: Q2 64^3 FP64 92 -> 63 us, Q3 64^3 178 -> 131 us, FP32 unchanged.
template <typename Number> struct TanhSeries;
template <> struct TanhSeries<double> {
  static constexpr int N = 12;
  static constexpr double c[N] = {1.0 / 6227020800.0, 1.0 / 479001600.0, 1.0 / 39916800.0, 1.0 / 3628800.0,
                                  1.0 / 362880.0,     1.0 / 40320.0,     1.0 / 5040.0,     1.0 / 720.0,
                                  1.0 / 120.0,        1.0 / 24.0,        1.0 / 6.0,        0.5};
  static constexpr double log2e = 1.4426950408889634, ln2_hi = 0x1.62e42fefa3800p-1, ln2_lo = 0x1.ef35793c76730p-45;
};
template <> struct TanhSeries<float> {
  static constexpr int N = 7;
  static constexpr float c[N] = {1.0f / 40320.0f, 1.0f / 5040.0f, 1.0f / 720.0f, 1.0f / 120.0f, 1.0f / 24.0f, 1.0f / 6.0f, 0.5f};
  static constexpr float log2e = 1.44269504f, ln2_hi = 0x1.62e400p-1f, ln2_lo = 0x1.7f7d1cp-20f;
};
__device__ __forceinline__ double reciprocal_estimate(double d) {
  const double v = __builtin_amdgcn_rcp(d);
  return fma(fma(-d, v, 1.0), v, v);
}
__device__ __forceinline__ float reciprocal_estimate(float d) { return __builtin_amdgcn_rcpf(d); }
template <typename Number> __device__ __forceinline__ Number law_tanh(Number x) {
  using C = TanhSeries<Number>;
  constexpr bool carry = sizeof(Number) == 8;
  const Number one = 1, y = -2 * fabs(x), n = rint(y * C::log2e);
  const Number a = fma(n, -C::ln2_hi, y), r = fma(n, -C::ln2_lo, a), r2 = r * r;
  Number q = C::c[0];
#pragma unroll
  for (int i = 1; i < C::N; ++i) q = fma(q, r, C::c[i]);
  const Number p = fma(r2, q, r), p_lo = carry ? fma(r2, q, r - p) + fma(n, -C::ln2_lo, a - r) : Number(0);
  const Number s = ldexp(one, (int)n), h = s - one, h_lo = s - (h + one);
  const Number e = fma(s, p, h), e_lo = fma(s, p_lo, fma(s, p, h - e)) + h_lo;
  const Number d = e + 2, d_lo = e - (d - 2), v = reciprocal_estimate(d), t = e * v;
  const Number u = fma(fma(-(d_lo + e_lo), t, fma(-d, t, e)) + e_lo, v, t);
  return copysign(y < -40 ? one : u, x);
}

template <typename Number>
__device__ __forceinline__ Number law_kappa(int law, const Number *p, Number T) {
  if (law == LAW_TANH) {
    const Number inv = Number(1) / p[3];
    return p[0] * (Number(1) + p[1] * law_tanh((T - p[2]) * inv));
  }
  // mushy zone (liquid_solid): p = {k_liquid, k_solid, T_solidus, T_liquidus}
  const Number inv = Number(1) / (p[3] - p[2]);
  Number fs = (p[3] - T) * inv;
  fs = fs < Number(0) ? Number(0) : (fs > Number(1) ? Number(1) : fs);
  return p[0] + (p[1] - p[0]) * (Number(3) - Number(2) * fs) * fs * fs;
}

// A brick of the Q1..Q3 apply is cells[0] x cells[1] x cells[2] cells: pencils of cells side by side along x,
// done one after the other, steps along y, pencils along z. Shared-plane classes: bit 0 upper x plane, bit 1
// upper y plane, bit 2 upper z plane.
struct BrickGrid {
  int nb[3];       // bricks
  int cells[3];    // cells of a full brick
  long off[8];     // scratch offset of each class (off[0] unused)
  long total;      // scratch entries
};
// n / d for n < 2^31 by a multiplication: m = floor(2^(31 + s) / d) + 1 with 2^s >= d exceeds 2^(31 + s) / d by at
// most 1, so that n m / 2^(31 + s) exceeds n / d by less than 1 / 2^s <= 1 / d
struct FixedDivisor {
  unsigned long m = 1;
  int d = 1, shift = 0;
  FixedDivisor() = default;
  explicit FixedDivisor(int divisor) : d(divisor) {
    int s = 0;
    while ((1l << s) < d) ++s;
    shift = 31 + s;
    m = (1ul << shift) / d + 1;
  }
  __host__ __device__ __forceinline__ unsigned quotient(unsigned n) const { return (unsigned)((n * m) >> shift); }
};
// The classes an apply left to its reader: v + brick_sum is what the apply's own pass over the shared planes
// would have stored, in the same order of summation
template <typename Number> struct BrickSums {
  const Number *scratch = nullptr;
  BrickGrid g{};
  FixedDivisor nd0, nd1, plane[3];  // grid sizes, DoFs between shared planes
  int nd2 = 1;
  bool active = false;
  BrickSums() = default;
  BrickSums(const Number *scratch_, const BrickGrid &g_, int K, const int *nd)
      : scratch(scratch_), g(g_), nd0(nd[0]), nd1(nd[1]), nd2(nd[2]), active(true) {
    for (int d = 0; d < 3; ++d) plane[d] = FixedDivisor(K * g.cells[d]);
  }
};
#ifdef __HIPCC__
template <typename Number> __device__ __forceinline__ Number brick_sum(const BrickSums<Number> &B, Number v, unsigned i) {
  const unsigned row = B.nd0.quotient(i), iz = B.nd1.quotient(row);
  const int at[3] = {(int)(i - row * B.nd0.d), (int)(row - iz * B.nd1.d), (int)iz};
  int h[3];  // the shared plane a coordinate lies on (-1: none)
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const int q = (int)B.plane[d].quotient(at[d]);
    h[d] = q * B.plane[d].d == at[d] && q < B.g.nb[d] ? q - 1 : -1;
  }
  if (h[0] < 0 && h[1] < 0 && h[2] < 0) return v;
  const long ny1 = B.g.nb[1] - 1, nz1 = B.g.nb[2] - 1;
  double s = (double)v;
  if (h[0] >= 0) s += (double)B.scratch[B.g.off[1] + ((long)h[0] * B.nd2 + at[2]) * B.nd1.d + at[1]];
  if (h[1] >= 0) s += (double)B.scratch[B.g.off[2] + (h[1] + ny1 * at[2]) * B.nd0.d + at[0]];
  if (h[0] >= 0 && h[1] >= 0) s += (double)B.scratch[B.g.off[3] + (h[0] * ny1 + h[1]) * B.nd2 + at[2]];
  if (h[2] >= 0) s += (double)B.scratch[B.g.off[4] + ((long)h[2] * B.nd1.d + at[1]) * B.nd0.d + at[0]];
  if (h[0] >= 0 && h[2] >= 0) s += (double)B.scratch[B.g.off[5] + (h[0] * nz1 + h[2]) * B.nd1.d + at[1]];
  if (h[1] >= 0 && h[2] >= 0) s += (double)B.scratch[B.g.off[6] + (h[1] + ny1 * h[2]) * B.nd0.d + at[0]];
  if (h[0] >= 0 && h[1] >= 0 && h[2] >= 0) s += (double)B.scratch[B.g.off[7] + (h[0] * ny1 + h[1]) * nz1 + h[2]];
  return (Number)s;
}
#endif

// the bricks of a Q1..Q3 mesh (heat_brick.hip): {pencils along x, steps along y}, and those of the kernel with
// one cell per lane
void choose_brick(int degree, const int *n_cells, int *brick, int *brick_cells);

// Everything a level operator needs on the device (pointers are device memory).
template <typename Number>
struct OperatorData {
  int degree = 1;
  int nc[3] = {1, 1, 1};
  int nd[3] = {2, 2, 2};
  double L[3] = {1, 1, 1};
  double h[3] = {1, 1, 1};
  long n_dofs = 0, n_cells = 0;
  double c_mass = 1.0;
  int kappa_mode = KAPPA_CONST;
  double kappa = 1.0;
  const Number *kappa_arr = nullptr;
  int law = 0;
  double law_p[4] = {0, 0, 0, 1};
  const Number *T = nullptr;
  int dmask = 0;
  int robin_mask = 0;
  double alpha = 0, emissivity = 0, T_inf_conv = 0, T_inf_rad = 0;
  const double *T_robin = nullptr;  // temperature for the radiation linearisation (FP64)
  // mapped geometry, 7 values per quadrature point (placed by metric_at): JxW, then G = JxW J^-1 J^-T as
  // (00, 01, 11, 02, 12, 22)
  const Number *metric = nullptr;
  // metric with the conductivity folded in (kappa_q G), used for per-qp / k(T) conductivity on mapped meshes
  const Number *metric_k = nullptr;
  const double *coords = nullptr;   // mapping node coordinates (X block, Y block, Z block), FP64
  // apply scratch (apply_edge_elems Number entries): contributions to DoFs that workgroups share, summed
  // into dst after the cell kernel so that vmult is bitwise reproducible. Q4: the rows where four
  // columns meet, all zero between applies; Q1..Q3: the bricks' upper planes, written by every apply
  Number *edge = nullptr;
  size_t edge_elems = 0;
  int brick[2] = {1, 1}, brick_cells[3] = {1, 1, 16};  // Q1..Q3: choose_brick
  void set_mesh(int k, const int *ncells, const double *ext) {
    degree = k;
    for (int d = 0; d < 3; ++d) {
      nc[d] = ncells[d];
      nd[d] = k * ncells[d] + 1;
      L[d] = ext[d];
      h[d] = ext[d] / ncells[d];
    }
    n_dofs = (long)nd[0] * nd[1] * nd[2];
    n_cells = (long)nc[0] * nc[1] * nc[2];
    choose_brick(degree, nc, brick, brick_cells);
  }
};

// The per-point arrays the library makes itself (the metric, the tangent's coefficients). Q1..Q3: blocks of 16
// cells, [comp][qy][qx][qz][cell of the block], so that each load of the apply's wavefront (lane = 16 qz + cell) is
// contiguous (mapped Q3 96^3 FP64 apply: 0.82 ms; 2.4 ms with [cell][comp][q], where every lane reads its
// own line). A block is a pencil of 16 cells along x; the cells that a row has beyond its full pencils follow, row
// after row, in blocks of their own, so that no more than one block has room left (a pencil padded to 16
// cells per row takes 16 times the memory for one cell along x and 1.9 times for 17). Q4, whose kernels give a
// lane consecutive qx: [cell][comp][q].
// Block and place in it of cell cx of a row (row = cy + nc1 cz, of rows)
__host__ __device__ __forceinline__ long point_block(int nc0, long row, long rows, int cx, int &place) {
  const int full = nc0 / 16, rest = nc0 % 16;
  if (cx < 16 * full) {
    place = cx % 16;
    return row * full + cx / 16;
  }
  const long t = row * rest + cx - 16 * full;
  place = (int)(t % 16);
  return rows * full + t / 16;
}
// Where component comp (of ncomp) of quadrature point q = (qx, qy, qz) of a cell (of n_cells) lies
__host__ __device__ __forceinline__ long point_data_at(int n1, int nc0, long n_cells, long cell, int ncomp, int comp, int qx, int qy,
                                                       int qz) {
  const int nq = n1 * n1 * n1;
  if (n1 == 5) return (cell * ncomp + comp) * nq + qx + n1 * (qy + n1 * qz);
  const long row = cell / nc0;
  int place;
  const long block = point_block(nc0, row, n_cells / nc0, (int)(cell - row * nc0), place);
  return ((block * ncomp + comp) * nq + (qy * n1 + qx) * n1 + qz) * 16 + place;
}
inline size_t point_data_elems(int n1, const int *nc, int ncomp) {
  const size_t cells = (size_t)nc[0] * nc[1] * nc[2];
  return (n1 == 5 ? cells : (cells + 15) / 16 * 16) * ncomp * n1 * n1 * n1;
}
constexpr int kMetricComps = 7;
__host__ __device__ __forceinline__ long metric_at(int n1, int nc0, long n_cells, long cell, int comp, int qx, int qy, int qz) {
  return point_data_at(n1, nc0, n_cells, cell, kMetricComps, comp, qx, qy, qz);
}
inline size_t metric_elems(int n1, const int *nc) { return point_data_elems(n1, nc, kMetricComps); }

// A 1D N1 x N1 table stored by its symmetry about the cell centre (Gauss-Lobatto nodes and
// Gauss points are symmetric): T[N1-1-q][N1-1-i] = T[q][i] (ANTI = false, shape values) or
// -T[q][i] (ANTI = true, derivatives); only rows q < (N1+1)/2 are kept. Halving the tables
// halves the scalar registers the kernels hold them in. Indices are compile-time constants
// after unrolling, so the mirrored half costs at most a sign modifier.
template <typename Number, int N1, bool ANTI>
struct Half1D {
  Number h[(N1 + 1) / 2][N1];
  __host__ __device__ __forceinline__ Number operator()(int q, int i) const {
    return (2 * q < N1) ? h[q][i] : (ANTI ? -h[N1 - 1 - q][N1 - 1 - i] : h[N1 - 1 - q][N1 - 1 - i]);
  }
  void set(const double (&full)[kMaxN1][kMaxN1]) {
    for (int q = 0; 2 * q < N1; ++q)
      for (int i = 0; i < N1; ++i) h[q][i] = (Number)full[q][i];
  }
};

template <typename Number, int N1>
struct ApplyArgs {
  Half1D<Number, N1, false> S;  // shape values at the Gauss points
  Half1D<Number, N1, true> D;   // collocation derivative on the Gauss points
  Number w[N1];      // Gauss weights
  int nc[3], nd[3], ncol[2];
  int dmask, xcd_cols, law;
  Number cm;         // c_mass * hx hy hz
  Number ks[3];      // hx hy hz / h_d^2
  Number kappa;
  Number law_p[4];
  const Number *kappa_arr;
  const Number *T;
  const Number *metric;
  Number *edge;      // rows shared by four columns: the upper layer's contributions
};

template <typename Number, int N1>
void fill_apply_args(const OperatorData<Number> &op, ApplyArgs<Number, N1> &A) {
  const FE1D &fe = fe1d(N1 - 1);
  for (int a = 0; a < N1; ++a) A.w[a] = (Number)fe.qw[a];
  A.S.set(fe.S);
  A.D.set(fe.D);
  for (int d = 0; d < 3; ++d) {
    A.nc[d] = op.nc[d];
    A.nd[d] = op.nd[d];
  }
  const double vol = op.metric ? 1.0 : op.h[0] * op.h[1] * op.h[2];
  A.metric = op.metric;
  A.cm = (Number)(op.c_mass * vol);
  for (int d = 0; d < 3; ++d) A.ks[d] = (Number)(vol / (op.h[d] * op.h[d]));
  A.dmask = op.dmask;
  A.kappa = (Number)op.kappa;
  A.kappa_arr = op.kappa_arr;
  A.T = op.T;
  A.law = op.law;
  for (int i = 0; i < 4; ++i) A.law_p[i] = (Number)op.law_p[i];
  A.xcd_cols = 0;
  A.ncol[0] = A.ncol[1] = 1;
  A.edge = op.edge;
}

// heat_apply.hip; `kernel_start` and `kernel_end`, when given, are recorded on the stream
// right before and after the cell kernel (between the face-row pre-pass and the edge fix-up)
// so that the event pair times that kernel alone
// sums (Q1..Q3): where given, dst may be left without the classes of the planes that workgroups share; if so
// *sums is active and the next reader adds them (brick_sum), before another apply uses op.edge
template <typename Number>
int launch_apply(const OperatorData<Number> &op, const Number *src, Number *dst, hipStream_t stream,
                 hipEvent_t kernel_start = nullptr, hipEvent_t kernel_end = nullptr, BrickSums<Number> *sums = nullptr);
// entries of OperatorData::edge the apply of a mesh of degree k and n_cells cells needs
template <typename Number> size_t apply_edge_elems(const OperatorData<Number> &op);

// heat_brick.hip: the apply for Q1..Q3 and the scratch entries (OperatorData::edge) it needs
template <typename Number>
int launch_brick(const OperatorData<Number> &op, const Number *src, Number *dst, hipStream_t stream,
                 hipEvent_t kernel_start, hipEvent_t kernel_end, BrickSums<Number> *sums = nullptr);
size_t brick_scratch_elems(int degree, const int *n_cells, const int *brick, const int *brick_cells);
// Q1..Q3, Cartesian cells: dst -= c_m M (a T + b T_old + c q) + K_k T in one pass (T_old is not read when
// b = 0, q when null); constrained DoFs count as zero and are left alone, a conductivity law is evaluated at
// T as given. dst must not overlap the inputs.
int launch_brick_residual(const OperatorData<double> &op, const double *T, const double *T_old, const double *q, double a,
                          double b, double c, double *dst, hipStream_t stream);

// heat_aux.hip: diagonal, boundary faces, residual, norms, conductivity
// diag = the operator's diagonal (cells only; constrained rows 1); scratch: 2 n_cells (k+1)^3 values
template <typename Number>
int launch_diagonal(const OperatorData<Number> &op, Number *diag, Number *scratch, hipStream_t stream);
// boundary faces: mode 0 Robin tangent on src, 1 its diagonal, 2 boundary residual (+ surface flux)
int launch_boundary(const OperatorData<double> &op, int mode, const double *flux, double *dst,
                    const double *src, const double *T, hipStream_t stream);
struct FluxNodes {
  double nodes[kMaxN1];
  double p[6];
};
// The operator the kernels see: on mapped meshes with per-qp or k(T) conductivity the
// conductivity sits in metric_k and the kernels run with a constant unit conductivity.
template <typename Number>
OperatorData<Number> kernel_view(const OperatorData<Number> &op) {
  OperatorData<Number> v = op;
  if (op.metric && (op.kappa_mode == KAPPA_QP || op.kappa_mode == KAPPA_LAW)) {
    v.metric = op.metric_k;
    v.kappa_mode = KAPPA_CONST;
    v.kappa = 1.0;
  }
  return v;
}
template <typename Number>
int launch_scale_metric(const OperatorData<Number> &op, const Number *kq, Number *metric_k, hipStream_t s);
template <typename Number>
int launch_metric(const OperatorData<Number> &op, const double *coords, Number *metric, hipStream_t s);
int launch_surface_flux_field(const OperatorData<double> &op, const double *p6, double *out, hipStream_t s);
template <typename Number>
int launch_kappa_qp(const OperatorData<Number> &op, Number *kq, hipStream_t stream);
// quadrature-weighted cell averages sum_q w_q k_q of the conductivity (any mode)
template <typename Number>
int launch_cell_average(const OperatorData<Number> &op, Number *kcell, hipStream_t stream);
template <typename Number>
int launch_coarsen_cells(const int *nc_fine, const Number *kf, Number *kc, hipStream_t stream);

}  // namespace mpdg
