// Matrix-free apply of the implicit heat operator J = c_m M + K_kappa for Q1..Q3 on CDNA4
// (gfx950): HeatDiffuseMultiPhaseOperator::tangent_cell_loop / tangent_local_cell_operation
// (source/heat/heat_diffuse_operator.cpp:201-241, :957-1086). Q4 runs the column kernel of
// heat_apply.hip (its five z planes do not fit the four lane rows used here).
//
// Work decomposition
//   * A workgroup of four wavefronts owns a brick of 16 x SEG x ZC cells (ZC = 4, Q1: 8). A
//     wavefront holds one pencil of 16 cells along x per step and marches along y.
//   * Lane = 16 (z plane of the cell) + (cell along x); the lane's registers hold the plane's
//     N1 x N1 DoFs [y][x]. Q1 puts two cells' planes into the four lane rows, Q2 leaves one row
//     idle.
//   * Sum factorisation without a change of layout: x and y sweeps are register-local; the z
//     sweeps contract over the lane rows. In FP64 that is v_mfma_f64_4x4x4_4b (B and D share the
//     layout lane = 16 k + column, so a z sweep is one MFMA per register with the 1D table as A; it
//     runs at the rate of v_fma_f64 and saves the LDS transposes around a sweep on the VALU); in FP32
//     the forward pair of sweeps is one v_mfma_f32_16x16x4 per register whose rows 4 g + r hold row g
//     of table r, and the backward pair transposes y registers against lane rows with
//     v_permlane32/16_swap. Conductivity per point: twelve sweeps (collocated gradients on the Gauss
//     points). One conductivity per Cartesian cell: seven sweeps with 1D mass and stiffness matrices.
//   * Sums over a brick's cells, in FP64 at every precision and in a fixed order: along y the top row
//     of a cell goes through LDS to the next step; along x the last column moves one lane up (DPP
//     row_shr:1), and through LDS to the next pencil; along z the top plane goes through LDS to the next
//     pencil (one workgroup barrier per step). A brick's sums are rounded to the operator's type where they
//     are stored: in FP32 a DoF that bricks share (a corner: eight of them) is a sum of rounded parts.
//   * A brick stores its DoFs except its upper x, y, z planes; those are shared with the next
//     brick, which owns them, and go to a scratch array per class (planes, edges, corners).
//     brick_fixup_kernel adds the classes to dst in a fixed order: no atomics and no zeroed
//     rows, and vmult is bitwise repeatable.
//
// What bounds it: at Q3 FP64 with k per point, the latency of its loads at two wavefronts per SIMD (Q3 128^3:
// 1.66 GB read and 0.56 GB written, which streams of their own take 0.39 ms for, in 0.52 to 0.56 ms; VALU 39 %
// busy, 863 VALU instructions per 64 lanes and step) -- whole vmult: 0.663 ms for the column kernel with LDS
// transposes, scatter and atomics it replaces, 0.566 ms here; elsewhere the VALU (Q3 128^3, constant k: FP64
// 0.62 -> 0.43 ms, FP32 0.42 -> 0.28 ms; Q3 75 x 62 x 49 FP32 83.8 -> 45.4 us). Mapped Q3 96^3 FP64: 1.08 -> 0.78
// ms, near what reading the stored metric takes (0.60 ms with the vectors). Q1 and Q2 on Cartesian cells run
// heat_cells_kernel below, one lane per cell; here they run mapped, as residual and as the full tangent.
#include "tangent.hpp"

namespace mpdg {

namespace {

constexpr int kNX = 16;  // cells of a pencil along x (lanes of a DPP row)
constexpr int kNW = 4;   // wavefronts of a workgroup

template <int N1> struct BrickShape {
  static constexpr int K = N1 - 1;
  static constexpr int ZPW = N1 == 2 ? 2 : 1;  // cells along z per wavefront
  static constexpr int ZC = kNW * ZPW;         // cells along z per brick
};

constexpr int kMaxSteps = 16, kMaxPencils = 2;

constexpr int zc_of(int k) { return k == 1 ? BrickShape<2>::ZC : BrickShape<3>::ZC; }
// brick: {pencils along x, steps along y, cells of a pencil}, the last for the kernel with one cell per lane
BrickGrid brick_grid(int k, const int *nc, const int *brick, bool cells) {
  BrickGrid g;
  const int lx = cells ? brick[2] : kNX, zc = cells ? 64 / lx : zc_of(k), px = (nc[0] + lx - 1) / lx;
  g.cells[0] = lx * brick[0];
  g.cells[1] = brick[1];
  g.cells[2] = zc;
  g.nb[0] = (px + brick[0] - 1) / brick[0];
  g.nb[1] = (nc[1] + brick[1] - 1) / brick[1];
  g.nb[2] = (nc[2] + zc - 1) / zc;
  const long nd[3] = {(long)k * nc[0] + 1, (long)k * nc[1] + 1, (long)k * nc[2] + 1};
  long o = 0;
  g.off[0] = 0;
  for (int c = 1; c < 8; ++c) {
    g.off[c] = o;
    long n = 1;
    for (int d = 0; d < 3; ++d) n *= (c >> d & 1) ? g.nb[d] - 1 : nd[d];
    o += n;
  }
  g.total = o;
  return g;
}

template <typename Number, int N1>
struct BrickArgs {
  Half1D<Number, N1, false> S;            // shape values at the Gauss points
  Half1D<Number, N1, true> D, Dy, G;      // collocation derivative (Dy: times ky/kx), basis derivative
  Half1D<Number, N1, true> Gz;            // basis derivative times kz/kx
  Half1D<Number, N1, false> M1, K1;       // 1D mass and stiffness matrices of the unit cell
  Number w[(N1 + 1) / 2];  // Gauss weights (symmetric)
  int nc[3], nd[3];
  long n_cells;
  BrickGrid g;
  int dmask, law;
  Number cm, kx, ky, kz, kappa;  // V c_m, k_d = V/h_d^2 (mapped cells: 1)
  Number law_p[4];
  const Number *kappa_arr, *T, *metric;
  Number *scratch;
  // residual: the mass term acts on fa src + fb T_old + fc q
  Number fa, fb, fc;
  const Number *T_old, *q;
  // the full Newton tangent: whether it has the solidification terms; convection: 0 none, 1 with the constant
  // velocity vh (over the cell sizes), 2 with a velocity field
  int conv, solid;
  Number vh[3];
};

// x sweep (second index): out[j][q] = sum_i M(q, i) in[j][i]; y sweep (first index) likewise
template <int N1, bool TR, bool ADD, typename Number, typename Mat>
__device__ __forceinline__ void sweep_x(const Mat &M, const Number (&in)[N1][N1], Number (&out)[N1][N1]) {
#pragma unroll
  for (int j = 0; j < N1; ++j)
#pragma unroll
    for (int q = 0; q < N1; ++q) {
      Number a = ADD ? out[j][q] : Number(0);
#pragma unroll
      for (int i = 0; i < N1; ++i) a = fma(TR ? M(i, q) : M(q, i), in[j][i], a);
      out[j][q] = a;
    }
}
template <int N1, bool TR, bool ADD, typename Number, typename Mat>
__device__ __forceinline__ void sweep_y(const Mat &M, const Number (&in)[N1][N1], Number (&out)[N1][N1]) {
#pragma unroll
  for (int i = 0; i < N1; ++i)
#pragma unroll
    for (int q = 0; q < N1; ++q) {
      Number a = ADD ? out[q][i] : Number(0);
#pragma unroll
      for (int j = 0; j < N1; ++j) a = fma(TR ? M(j, q) : M(q, j), in[j][i], a);
      out[q][i] = a;
    }
}

using f32x4 = float __attribute__((ext_vector_type(4)));

// entry (row, col) of a table for a lane-dependent place; 0 outside (Q2's idle row)
template <int N1, typename Number, typename Mat>
__device__ __forceinline__ Number table_entry(const Mat &M, int row, int col) {
  Number v = 0;
#pragma unroll
  for (int a = 0; a < N1; ++a)
#pragma unroll
    for (int b = 0; b < N1; ++b) v = (row == a && col == b) ? M(a, b) : v;
  return v;
}

__device__ __forceinline__ void swap32(float &a, float &b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  const unsigned x = r[0], y = r[1];  // (a bit cast of a subscript would read element 0)
  a = __uint_as_float(x);
  b = __uint_as_float(y);
}
__device__ __forceinline__ void swap16(float &a, float &b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  const unsigned x = r[0], y = r[1];
  a = __uint_as_float(x);
  b = __uint_as_float(y);
}
__device__ __forceinline__ void swap16(double &a, double &b) {
  float al = __uint_as_float((unsigned)__double2loint(a)), ah = __uint_as_float((unsigned)__double2hiint(a));
  float bl = __uint_as_float((unsigned)__double2loint(b)), bh = __uint_as_float((unsigned)__double2hiint(b));
  swap16(al, bl);
  swap16(ah, bh);
  a = __hiloint2double((int)__float_as_uint(ah), (int)__float_as_uint(al));
  b = __hiloint2double((int)__float_as_uint(bh), (int)__float_as_uint(bl));
}
// registers <-> lane rows: afterwards register j of lane row r holds what register r of lane row
// j held (Q1: within each pair of lane rows)
template <int N1, typename Number> __device__ __forceinline__ void row_transpose(Number (&r)[4]) {
  if constexpr (N1 == 2) {
    swap16(r[0], r[1]);
  } else {
    swap32(r[0], r[2]);
    swap32(r[1], r[3]);
    swap16(r[0], r[1]);
    swap16(r[2], r[3]);
  }
}

// The lane's entries of the A operands of the z sweeps (see the file's head): forward tables F0 and
// F1 (values and derivative, or mass and stiffness), backward ones S^T and G_z^T.
template <int N1, typename Number> struct ZTables {  // Q1: transposed sweeps only
  template <typename Args, typename T0, typename T1>
  __device__ __forceinline__ ZTables(const Args &, const T0 &, const T1 &, int) {}
};
template <int N1> struct ZTablesF64 {
  double f0, f1, st, gt;
  template <typename Args, typename T0, typename T1>
  __device__ __forceinline__ ZTablesF64(const Args &P, const T0 &F0, const T1 &F1, int lane) {
    const int i = lane & 3, k = lane >> 4;  // A[i][k]
    f0 = table_entry<N1, double>(F0, i, k);
    f1 = table_entry<N1, double>(F1, i, k);
    st = table_entry<N1, double>(P.S, k, i);
    gt = table_entry<N1, double>(P.Gz, k, i);
  }
};
template <int N1> struct ZTablesF32 {
  float f01;
  template <typename Args, typename T0, typename T1>
  __device__ __forceinline__ ZTablesF32(const Args &, const T0 &F0, const T1 &F1, int lane) {
    const int row = (lane & 15) >> 2, r = lane & 3, k = lane >> 4;  // A[4 row + r][k] = table r, entry (row, k)
    const float a = table_entry<N1, float>(F0, row, k), b = table_entry<N1, float>(F1, row, k);
    f01 = r > 1 ? 0.0f : (r == 0 ? a : b);
  }
};
template <> struct ZTables<3, double> : ZTablesF64<3> { using ZTablesF64<3>::ZTablesF64; };
template <> struct ZTables<4, double> : ZTablesF64<4> { using ZTablesF64<4>::ZTablesF64; };
template <> struct ZTables<3, float> : ZTablesF32<3> { using ZTablesF32<3>::ZTablesF32; };
template <> struct ZTables<4, float> : ZTablesF32<4> { using ZTablesF32<4>::ZTablesF32; };

// v = F0 t along z, and g = F1 t when SECOND
template <int N1, bool SECOND, typename Number, typename T0, typename T1>
__device__ __forceinline__ void z_forward(const T0 &F0, const T1 &F1, const ZTables<N1, Number> &z, const Number (&t)[N1][N1],
                                          Number (&v)[N1][N1], Number (&g)[N1][N1]) {
  if constexpr (N1 == 2) {
    // pairs of lane rows hold different cells: sweeps on the transposed pairs, so that nothing of one
    // cell is multiplied into another
#pragma unroll
    for (int i = 0; i < N1; ++i) {
      Number a[4] = {t[0][i], t[1][i], 0, 0}, s[4] = {0, 0, 0, 0}, d[4] = {0, 0, 0, 0};
      row_transpose<N1>(a);
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        s[q] = fma(F0(q, 0), a[0], F0(q, 1) * a[1]);
        d[q] = fma(F1(q, 0), a[0], F1(q, 1) * a[1]);
      }
      row_transpose<N1>(s);
      if (SECOND) row_transpose<N1>(d);
#pragma unroll
      for (int j = 0; j < N1; ++j) {
        v[j][i] = s[j];
        if (SECOND) g[j][i] = d[j];
      }
    }
  } else if constexpr (sizeof(Number) == 8) {
#pragma unroll
    for (int j = 0; j < N1; ++j)
#pragma unroll
      for (int i = 0; i < N1; ++i) {
        const double x = t[j][i];
        v[j][i] = __builtin_amdgcn_mfma_f64_4x4x4f64(z.f0, x, 0.0, 0, 0, 0);
        if (SECOND) g[j][i] = __builtin_amdgcn_mfma_f64_4x4x4f64(z.f1, x, 0.0, 0, 0, 0);
      }
  } else {
#pragma unroll
    for (int j = 0; j < N1; ++j)
#pragma unroll
      for (int i = 0; i < N1; ++i) {
        const f32x4 r = __builtin_amdgcn_mfma_f32_16x16x4f32(z.f01, t[j][i], f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
        v[j][i] = r[0];
        if (SECOND) g[j][i] = r[1];
      }
  }
}

// out = S_z^T e + G_z^T f (the z table of the way back carries the direction's factor)
template <int N1, typename Args, typename Number>
__device__ __forceinline__ void z_backward(const Args &P, const ZTables<N1, Number> &z, const Number (&e)[N1][N1],
                                           const Number (&f)[N1][N1], Number (&out)[N1][N1]) {
  if constexpr (N1 > 2 && sizeof(Number) == 8) {
#pragma unroll
    for (int j = 0; j < N1; ++j)
#pragma unroll
      for (int i = 0; i < N1; ++i) {
        const double a = __builtin_amdgcn_mfma_f64_4x4x4f64(z.gt, f[j][i], 0.0, 0, 0, 0);
        out[j][i] = __builtin_amdgcn_mfma_f64_4x4x4f64(z.st, e[j][i], a, 0, 0, 0);
      }
  } else {
#pragma unroll
    for (int i = 0; i < N1; ++i) {
      Number a[4] = {0, 0, 0, 0}, b[4] = {0, 0, 0, 0}, o[4] = {0, 0, 0, 0};
#pragma unroll
      for (int j = 0; j < N1; ++j) {
        a[j] = e[j][i];
        b[j] = f[j][i];
      }
      row_transpose<N1>(a);
      row_transpose<N1>(b);
#pragma unroll
      for (int q = 0; q < N1; ++q) {
        Number s = 0;
#pragma unroll
        for (int k = 0; k < N1; ++k) s = fma(P.Gz(k, q), b[k], s);
#pragma unroll
        for (int k = 0; k < N1; ++k) s = fma(P.S(k, q), a[k], s);
        o[q] = s;
      }
      row_transpose<N1>(o);
#pragma unroll
      for (int j = 0; j < N1; ++j) out[j][i] = o[j];
    }
  }
}

// value of the previous lane in the row of 16; the first lane gets `first`
__device__ __forceinline__ double from_previous_cell(double x, double first) {
  const int lo = __builtin_amdgcn_update_dpp(__double2loint(first), __double2loint(x), 0x111, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(__double2hiint(first), __double2hiint(x), 0x111, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}

// orders the LDS accesses of a wavefront's lanes
__device__ __forceinline__ void lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

constexpr int KAPPA_TANGENT = 4;   // the full Newton tangent's coefficients instead of a conductivity
constexpr int TANGENT_DIAGONAL = 5;  // ... and its diagonal: no source is read

// Wavefronts per SIMD the register allocation targets: as many as fit with few or no spilled VGPRs (Q3 FP64:
// 228 VGPRs with per-point conductivity; 168 with one per cell, 6 to 11 of them spilled, in the residual too; Q2's
// residual with a law 16 spilled at three; mapped cells hold three fluxes: Q3 FP64 215, FP32 123). Fewer
// wavefronts were slower even where the next step's source was loaded ahead, and with three or four the
// loads need no such registers. The 1D tables and sizes exceed the scalar registers: Q2 and Q3 keep 50 to 126
// of them in VGPR lanes.
template <int N1, typename Number, bool MAPPED, int KMODE> struct BrickOccupancy { static constexpr int W = 4; };
template <bool M, int KM> struct BrickOccupancy<3, double, M, KM> { static constexpr int W = 3; };
template <bool M, int KM> struct BrickOccupancy<4, double, M, KM> { static constexpr int W = 2; };
template <> struct BrickOccupancy<4, double, false, KAPPA_CONST> { static constexpr int W = 3; };
template <> struct BrickOccupancy<4, double, false, KAPPA_CELL> { static constexpr int W = 3; };
// (more loads of its eight coefficients in flight: Q3 50 x 40 x 30 142 -> 124 us)
template <> struct BrickOccupancy<4, double, false, KAPPA_TANGENT> { static constexpr int W = 1; };
template <int KM> struct BrickOccupancy<4, float, true, KM> { static constexpr int W = 3; };
template <> struct BrickOccupancy<4, float, false, KAPPA_QP> { static constexpr int W = 3; };

// what a lane is, in one register (tested where it is needed: as loop invariants the tests would
// occupy two scalar registers each, and the 1D tables need those)
constexpr int F_TOP = 1;     // its lane row holds its cell's upper z plane
constexpr int F_LOW = 2;     // ... the lowest z plane, with a pencil below in the brick
constexpr int F_STORE = 4;   // ... a plane of the mesh that this wavefront stores
constexpr int F_HZ = 8;      // ... the brick's upper z plane, owned by the next brick
constexpr int F_LAST = 16;   // the last lane of its row
__device__ __forceinline__ int opaque(int f) {
  asm volatile("" : "+v"(f));
  return f;
}

// The kernel's arguments read anew where they are used: kept in scalar registers over the whole
// loop, the mesh's sizes and offsets push the 1D tables out of them (150 v_readlane per step)
template <typename Args> __device__ __forceinline__ const __attribute__((address_space(4))) Args &fresh_args() {
  auto p = (const __attribute__((address_space(4))) Args *)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *p;
}


// RES: dst -= the residual's cell part (see launch_brick_residual) instead of dst = J src
template <int N1, typename Number, int KMODE, bool MAPPED, bool RES = false>
__global__ __launch_bounds__(64 * kNW) __attribute__((amdgpu_waves_per_eu(BrickOccupancy<N1, Number, MAPPED, KMODE>::W)))
void heat_brick_kernel(const BrickArgs<Number, N1> P, const Number *__restrict__ src, Number *__restrict__ dst) {
  using B = BrickShape<N1>;
  constexpr int K = B::K, NQ = N1 * N1 * N1, W = K * kNX;
  // Q3: per-point conductivities go through LDS. 16 cells' values are contiguous in memory and are
  // loaded 1 KB per instruction; read in place, a lane's own N1^2 values would cost one L1 line per
  // lane and load (0.12 ms of the Q3 128^3 apply)
  constexpr bool STAGE = KMODE == KAPPA_QP && N1 == 4 && !MAPPED;
  constexpr int NV = 16 / (int)sizeof(Number), CH = N1 * N1 / NV, PER = 4 * CH, NLD = STAGE ? kNX * PER / 64 : 1;
  __shared__ double top[2][B::ZC][K][N1][kNX];      // top planes of the pencils' cells, by step parity
  __shared__ double yrow[kNW][kMaxPencils][N1][64]; // top rows of the previous y step's cells
  __shared__ Number srow[kNW][kMaxPencils][N1][64]; // their source rows, the next step's lowest
  __shared__ double xcol[kNW][N1][4];               // last x column of the previous pencil
  // per wavefront: staged conductivities, then the rows of results, to be stored with consecutive
  // lanes on consecutive addresses
  constexpr int STAGE_N = STAGE ? NQ * kNX : 0, TILE_N = K > 1 ? 4 * (64 / W) * W : 1;
  __shared__ __attribute__((aligned(16))) Number buf[kNW][STAGE_N > TILE_N ? STAGE_N : TILE_N];

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), row = lane >> 4, c = lane & 15;
  const int l = N1 == 2 ? row & 1 : row;                  // z plane of the cell
  const int zc = N1 == 2 ? 2 * wave + (row >> 1) : wave;  // cell along z in the brick
  // consecutive workgroups run on different XCDs; give each XCD a contiguous range of bricks
  const int nbr = gridDim.x, xcd = blockIdx.x & 7;
  int b = xcd * (nbr >> 3) + min(xcd, nbr & 7) + (blockIdx.x >> 3);
  const int bx = b % P.g.nb[0];
  b /= P.g.nb[0];
  const int by = b % P.g.nb[1], bz = b / P.g.nb[1];
  const int cz = bz * B::ZC + zc, cy0 = by * P.g.cells[1], cx0 = bx * P.g.cells[0];
  const int cy_end = min(cy0 + P.g.cells[1], P.nc[1]), cx_end = min(cx0 + P.g.cells[0], P.nc[0]);
  const int iz = K * cz + l;
  const long sy = P.nd[0], sz = (long)P.nd[0] * P.nd[1];
  // a conductivity that is constant on a Cartesian cell: the cell's operator is a sum of products of
  // 1D mass and stiffness matrices, seven sweeps instead of twelve
  constexpr bool TENSOR = !MAPPED && (KMODE == KAPPA_CONST || KMODE == KAPPA_CELL);
  const ZTables<N1, Number> zt = [&] {
    if constexpr (TENSOR) return ZTables<N1, Number>(P, P.M1, P.K1, lane);
    else return ZTables<N1, Number>(P, P.S, P.G, lane);
  }();
  Number wz = 0;
#pragma unroll
  for (int a = 0; a < N1; ++a) wz = l == a ? P.w[a < N1 - 1 - a ? a : N1 - 1 - a] : wz;
  int flags = 0;
  {
    const bool on = cz < P.nc[2] && l <= K, last_z = cz == P.nc[2] - 1;
    if (l == K) flags |= F_TOP;
    if (l == 0 && zc > 0) flags |= F_LOW;
    if (on && (l < K || zc == B::ZC - 1 || last_z)) flags |= F_STORE;
    if (l == K && !last_z) flags |= F_HZ;
    if (c == kNX - 1) flags |= F_LAST;
  }
  // Lanes without a cell work on the mesh's last cell in their direction: in bounds, and nothing of
  // theirs reaches another lane's cell (sums pass upwards in x and z only). Q2's idle lane row
  // holds zeros.
  const long zoff = sz * (K * min(cz, P.nc[2] - 1) + min(l, K));

  // constrained planes that touch the brick (a z plane would otherwise be tested for in every step of every
  // brick: residual of Q1 128^3 with k per point 88 -> 79 us, Q3 48^3 64 -> 61 us, Q3 75 x 62 x 49 FP32 apply
  // 46.0 -> 44.4 us)
  int bmask = P.dmask;
  if (cx0 > 0) bmask &= ~1;
  if (cx_end < P.nc[0]) bmask &= ~2;
  if (cy0 > 0) bmask &= ~4;
  if (cy_end < P.nc[1]) bmask &= ~8;
  if (bz > 0) bmask &= ~16;
  if (bz + 1 < P.g.nb[2]) bmask &= ~32;
  // ... that touch the pencil at (cxb, cy): zero the DoFs on them
  auto constrain = [&](int cxb, int cy, auto &u) {
    int m = bmask;
    if (m) {
      if (cxb > 0) m &= ~1;
      if (cxb + kNX < fresh_args<BrickArgs<Number, N1>>().nc[0]) m &= ~2;
      if (cy > 0) m &= ~4;
      if (cy + 1 < fresh_args<BrickArgs<Number, N1>>().nc[1]) m &= ~8;
    }
    if (m) {
      const int cx = cxb + opaque(c), z = opaque(iz);
      const auto &A = fresh_args<BrickArgs<Number, N1>>();
      const bool con_z = ((m & 16) && z == 0) || ((m & 32) && z == A.nd[2] - 1);
#pragma unroll
      for (int j = 0; j < N1; ++j)
#pragma unroll
        for (int i = 0; i < N1; ++i)
          if (con_z || ((m & 4) && j == 0) || ((m & 8) && j == K) || ((m & 1) && i == 0 && cx == 0) ||
              ((m & 2) && i == K && cx == A.nc[0] - 1))
            u[j][i] = 0;
    }
  };
  // the plane's rows of the pencil's cells
  auto load_rows = [&](const Number *field, int cxb, int cy, bool lowest, Number (&u)[N1][N1]) {
    const Number *p = field + (zoff + K * min(cxb + c, P.nc[0] - 1)) + sy * ((long)K * cy);
#pragma unroll
    for (int i = 0; i < N1; ++i) u[0][i] = lowest ? p[i] : Number(0);
#pragma unroll
    for (int j = 1; j < N1; ++j)
#pragma unroll
      for (int i = 0; i < N1; ++i) u[j][i] = p[i + sy * j];
    if (N1 == 3) {
#pragma unroll
      for (int j = 0; j < N1; ++j)
#pragma unroll
        for (int i = 0; i < N1; ++i) u[j][i] = row < 3 ? u[j][i] : Number(0);
    }
  };
  // the lane's first point in the arrays with ncomp values per point (point_data_at)
  auto point_data = [&](const auto &A, int ncomp, int cxb, int cy) {
    const long row = cy + (long)A.nc[1] * min(cz, A.nc[2] - 1);
    const int full = (unsigned)A.nc[0] / kNX;
    long block = row * full + (unsigned)cxb / kNX;
    int at = min(l, K) * kNX + c;
    if (cxb + kNX > A.nc[0]) {
      const long t = row * ((unsigned)A.nc[0] % kNX);
      const int place = (int)(t % kNX) + min(c, A.nc[0] - 1 - cxb);
      block = (long)A.nc[1] * A.nc[2] * full + t / kNX;
      at = (place / kNX * ncomp * NQ + min(l, K)) * kNX + place % kNX;
    }
    return A.metric + block * (ncomp * NQ * kNX) + at;
  };
  int parity = 0;
  for (int cy = cy0; cy < cy_end; ++cy) {
    const bool last = cy + 1 == cy_end;  // the brick's top row is complete too
    int pen = 0;
    for (int cxb = cx0; cxb < cx_end; cxb += kNX, ++pen, parity ^= 1) {
      const long cell = min(cxb + c, P.nc[0] - 1) + (long)P.nc[0] * (cy + (long)P.nc[1] * min(cz, P.nc[2] - 1));
      constexpr bool DIAGONAL = KMODE == TANGENT_DIAGONAL;
      Number u[N1][N1];
      if constexpr (!DIAGONAL) load_rows(src, cxb, cy, cy == cy0, u);
      if (!DIAGONAL && cy > cy0) {
#pragma unroll
        for (int i = 0; i < N1; ++i) u[0][i] = srow[wave][pen][i][lane];
      }
      if (!DIAGONAL && !last) {
#pragma unroll
        for (int i = 0; i < N1; ++i) srow[wave][pen][i][lane] = u[K][i];
      }
      // ---- conductivity at the points of this lane's plane qz = l ----
      const auto &A = fresh_args<BrickArgs<Number, N1>>();
      Number w[N1][N1];  // RES: what the mass term is applied to
      if constexpr (RES) {
        Number t[N1][N1];
#pragma unroll
        for (int j = 0; j < N1; ++j)
#pragma unroll
          for (int i = 0; i < N1; ++i) w[j][i] = A.fa * u[j][i];
        if (A.fb != Number(0)) {
          load_rows(A.T_old, cxb, cy, true, t);
#pragma unroll
          for (int j = 0; j < N1; ++j)
#pragma unroll
            for (int i = 0; i < N1; ++i) w[j][i] = fma(A.fb, t[j][i], w[j][i]);
        }
        if (A.q) {
          load_rows(A.q, cxb, cy, true, t);
#pragma unroll
          for (int j = 0; j < N1; ++j)
#pragma unroll
            for (int i = 0; i < N1; ++i) w[j][i] = fma(A.fc, t[j][i], w[j][i]);
        }
        constrain(cxb, cy, w);
      }
      // the law is evaluated at the source as it is; interpolated below, before the constraints
      constexpr bool LAW_OF_SRC = RES && KMODE == KAPPA_LAW;
      if constexpr (!LAW_OF_SRC && !DIAGONAL) constrain(cxb, cy, u);

      using Vec = Number __attribute__((ext_vector_type(NV)));
      Number kq[N1][N1];
      Vec kraw[NLD];
      Number kc = P.kappa;
      if (KMODE == KAPPA_CELL) kc = A.kappa_arr[cell];
      if constexpr (STAGE) {
        const long first = cxb + (long)A.nc[0] * (cy + (long)A.nc[1] * min(bz * B::ZC + wave, A.nc[2] - 1));
        const Vec *p = reinterpret_cast<const Vec *>(A.kappa_arr) + first * (NQ / NV);
        // (a ragged row's last pencil reads into the next row's cells; the array's end is clamped)
        const long left = (A.n_cells - first) * (NQ / NV);
        if (left >= 64 * NLD) {
#pragma unroll
          for (int m = 0; m < NLD; ++m) kraw[m] = __builtin_nontemporal_load(p + 64 * m + lane);
        } else {
#pragma unroll
          for (int m = 0; m < NLD; ++m) kraw[m] = p[min((long)(64 * m + lane), left - 1)];
        }
      } else if (KMODE == KAPPA_QP) {
        // (Q1 past the caches: residual of 160 x 170 x 150, whose k exceeds them, 134 -> 127 us; of 128^3, whose
        // k a repeated call finds there, 72 -> 80 us)
        const Number *p = A.kappa_arr + cell * NQ + N1 * N1 * min(l, K);
#pragma unroll
        for (int j = 0; j < N1; ++j)
#pragma unroll
          for (int i = 0; i < N1; ++i) kq[j][i] = N1 == 2 ? __builtin_nontemporal_load(p + N1 * j + i) : p[N1 * j + i];
      }
      if constexpr (KMODE == KAPPA_LAW && !LAW_OF_SRC) {
        Number a[N1][N1], t[N1][N1];
        load_rows(A.T, cxb, cy, true, a);
        sweep_x<N1, false, false>(P.S, a, t);
        sweep_y<N1, false, false>(P.S, t, a);
        z_forward<N1, false>(P.S, P.G, zt, a, t, t);
#pragma unroll
        for (int j = 0; j < N1; ++j)
#pragma unroll
          for (int i = 0; i < N1; ++i) kq[j][i] = law_kappa<Number>(P.law, P.law_p, t[j][i]);
      }
      Number v[N1][N1];
      if constexpr (TENSOR) {
        // J u = M_x [M_y (c_m M_z + k k_z K_z) + k k_y K_y M_z] u + k k_x K_x M_y M_z u
        Number mz[N1][N1], p[N1][N1];
        z_forward<N1, true>(P.M1, P.K1, zt, u, mz, p);
        if constexpr (RES) z_forward<N1, false>(P.M1, P.K1, zt, w, w, w);
        if (N1 == 3 && KMODE == KAPPA_CELL) kc = row < 3 ? kc : Number(0);
        const Number kx = kc * P.kx, ky = kc * P.ky, kz = kc * P.kz;
#pragma unroll
        for (int j = 0; j < N1; ++j)
#pragma unroll
          for (int i = 0; i < N1; ++i) p[j][i] = fma(P.cm, RES ? w[j][i] : mz[j][i], kz * p[j][i]);
        Number s[N1][N1];
        sweep_y<N1, false, false>(P.M1, mz, u);
        sweep_y<N1, false, false>(P.M1, p, s);
#pragma unroll
        for (int j = 0; j < N1; ++j)
#pragma unroll
          for (int i = 0; i < N1; ++i) {
            mz[j][i] *= ky;
            u[j][i] *= kx;
          }
        sweep_y<N1, false, true>(P.K1, mz, s);
        sweep_x<N1, false, false>(P.M1, s, v);
        sweep_x<N1, false, true>(P.K1, u, v);
      } else if constexpr (DIAGONAL) {
        // sum_q t0 phi^2 + sum_d a_d phi d_d phi + t1 / h_d^2 (d_d phi)^2 with 1D tables S: phi^2, G: phi phi',
        // M1: phi'^2 of the points (columns) at the DoFs (rows)
        const Number *M = point_data(A, kTangentCoeffs, cxb, cy);
        constexpr int C1 = NQ * kNX;
        const bool idle = N1 == 3 && row == 3;
        auto coefficients = [&](Number (&t)[N1][N1], auto value) {
#pragma unroll
          for (int j = 0; j < N1; ++j)
#pragma unroll
            for (int i = 0; i < N1; ++i) t[j][i] = idle ? Number(0) : value(M + (N1 * j + i) * N1 * kNX);
        };
        auto first_order = [&](Number (&t)[N1][N1], int d) {
          coefficients(t, [&](const Number *m) {
            Number a = 0;
            if (A.conv == 1) a = m[2 * C1] * A.vh[d];
            if (A.conv == 2) a = m[(2 + d) * C1];
            if (A.solid) a += m[(5 + d) * C1];
            return a;
          });
        };
        const ZTables<N1, Number> zt2(P, P.M1, P.G, lane);
        Number t[N1][N1], e[N1][N1], k[N1][N1], h[N1][N1], x[N1][N1];
        coefficients(t, [&](const Number *m) { return m[0]; });
        z_forward<N1, false>(P.S, P.G, zt, t, e, e);
        coefficients(t, [&](const Number *m) { return m[C1]; });
        z_forward<N1, false>(P.S, P.G, zt, t, k, k);
        z_forward<N1, false>(P.M1, P.G, zt2, t, t, t);
#pragma unroll
        for (int j = 0; j < N1; ++j)
#pragma unroll
          for (int i = 0; i < N1; ++i) e[j][i] = fma(P.kz, t[j][i], e[j][i]);
        const bool first = A.conv || A.solid;
        if (first) {
          first_order(t, 2);
          z_forward<N1, true>(P.S, P.G, zt, t, h, x);
#pragma unroll
          for (int j = 0; j < N1; ++j)
#pragma unroll
            for (int i = 0; i < N1; ++i) e[j][i] += x[j][i];
        }
        sweep_y<N1, false, false>(P.S, e, h);
        sweep_y<N1, false, false>(P.S, k, x);
#pragma unroll
        for (int j = 0; j < N1; ++j)
#pragma unroll
          for (int i = 0; i < N1; ++i) {
            k[j][i] *= P.ky;
            x[j][i] *= P.kx;
          }
        sweep_y<N1, false, true>(P.M1, k, h);
        if (first) {
          first_order(t, 1);
          z_forward<N1, false>(P.S, P.G, zt, t, k, k);
          sweep_y<N1, false, true>(P.G, k, h);
        }
        sweep_x<N1, false, false>(P.S, h, v);
        sweep_x<N1, false, true>(P.M1, x, v);
        if (first) {
          first_order(t, 0);
          z_forward<N1, false>(P.S, P.G, zt, t, k, k);
          sweep_y<N1, false, false>(P.S, k, e);
          sweep_x<N1, false, true>(P.G, e, v);
        }
      } else {
        // ---- to the points: v = values, gz = z derivative ----
        Number gz[N1][N1], e[N1][N1];
        auto to_points = [&](Number (&x)[N1][N1]) {
          Number t[N1][N1];
          sweep_x<N1, false, false>(P.S, x, t);
          sweep_y<N1, false, false>(P.S, t, x);
        };
        to_points(u);
        z_forward<N1, true>(P.S, P.G, zt, u, v, gz);
        if constexpr (LAW_OF_SRC) {
#pragma unroll
          for (int j = 0; j < N1; ++j)
#pragma unroll
            for (int i = 0; i < N1; ++i) kq[j][i] = law_kappa<Number>(P.law, P.law_p, v[j][i]);
          if (bmask) {
            load_rows(src, cxb, cy, true, u);
            constrain(cxb, cy, u);
            to_points(u);
            z_forward<N1, true>(P.S, P.G, zt, u, v, gz);
          }
        }
        if constexpr (RES) {
          to_points(w);
          z_forward<N1, false>(P.S, P.G, zt, w, w, w);
        }
        // ---- at the points (heat_diffuse_operator.cpp:1029-1077): e = c_m W v + D_x^T f_x + D_y^T f_y,
        //      gz becomes f_z ----
        if constexpr (KMODE == KAPPA_TANGENT) {
          // val = t0 u + t2..t4 . grad u, flux = t1 / h^2 grad u + t5..t7 u (tangent.hip); t2 alone for a
          // constant velocity
          Number gx[N1][N1], gy[N1][N1];
          sweep_x<N1, false, false>(P.D, v, gx);
          sweep_y<N1, false, false>(P.D, v, gy);
          const Number *M = point_data(A, kTangentCoeffs, cxb, cy);
          const bool idle = N1 == 3 && row == 3;
#pragma unroll
          for (int j = 0; j < N1; ++j)
#pragma unroll
            for (int i = 0; i < N1; ++i) {
              const Number *m = M + (N1 * j + i) * N1 * kNX;
              constexpr int C1 = NQ * kNX;
              const Number x = gx[j][i], y = gy[j][i], z = gz[j][i], uq = v[j][i], k = m[C1];
              Number val = m[0] * uq;
              if (A.conv == 1) val += m[2 * C1] * (A.vh[0] * x + A.vh[1] * y + A.vh[2] * z);
              if (A.conv == 2) val += m[2 * C1] * x + m[3 * C1] * y + m[4 * C1] * z;
              gx[j][i] = k * P.kx * x;
              gy[j][i] = k * P.ky * y;
              gz[j][i] = k * P.kz * z;
              if (A.solid) {
                gx[j][i] += m[5 * C1] * uq;
                gy[j][i] += m[6 * C1] * uq;
                gz[j][i] += m[7 * C1] * uq;
              }
              e[j][i] = val;
              if (idle) e[j][i] = gx[j][i] = gy[j][i] = gz[j][i] = Number(0);
            }
          sweep_x<N1, true, true>(P.D, gx, e);
          sweep_y<N1, true, true>(P.Dy, gy, e);
        } else if constexpr (MAPPED) {
          Number gx[N1][N1], gy[N1][N1];
          sweep_x<N1, false, false>(P.D, v, gx);
          sweep_y<N1, false, false>(P.D, v, gy);
          const Number *M = point_data(A, kMetricComps, cxb, cy);
          const bool idle = N1 == 3 && row == 3;
#pragma unroll
          for (int j = 0; j < N1; ++j)
#pragma unroll
            for (int i = 0; i < N1; ++i) {
              const Number *m = M + (N1 * j + i) * N1 * kNX;
              constexpr int C1 = NQ * kNX;
              const Number g00 = m[C1], g01 = m[2 * C1], g11 = m[3 * C1], g02 = m[4 * C1], g12 = m[5 * C1], g22 = m[6 * C1];
              const Number x = gx[j][i], y = gy[j][i], z = gz[j][i];
              e[j][i] = P.cm * m[0] * v[j][i];
              gx[j][i] = kc * (g00 * x + g01 * y + g02 * z);
              gy[j][i] = kc * (g01 * x + g11 * y + g12 * z);
              gz[j][i] = kc * (g02 * x + g12 * y + g22 * z);
              if (idle) e[j][i] = gx[j][i] = gy[j][i] = gz[j][i] = Number(0);
            }
          sweep_x<N1, true, true>(P.D, gx, e);
          sweep_y<N1, true, true>(P.Dy, gy, e);
        } else {
          if constexpr (STAGE) {
            // the 16-byte chunks of a 128-byte line are permuted by the cell's index, so that all lanes'
            // reads of chunk p spread over the banks
            Number *kb = buf[wave];
#pragma unroll
            for (int m = 0; m < NLD; ++m) {
              const int slot = 64 * m + lane, cc = slot / PER, ch = slot % PER;
              *reinterpret_cast<Vec *>(kb + (PER * cc + (ch ^ (cc & 7))) * NV) = kraw[m];
            }
            lds_fence();
#pragma unroll
            for (int p = 0; p < CH; ++p) {
              const Vec t = *reinterpret_cast<const Vec *>(kb + (PER * c + ((CH * row + p) ^ (c & 7))) * NV);
#pragma unroll
              for (int a = 0; a < NV; ++a) kq[(p * NV + a) / N1][(p * NV + a) % N1] = t[a];
            }
            lds_fence();
          }
          // weights of the lane's points: products of the few distinct 1D weights
          constexpr int H = (N1 + 1) / 2;
          const Number wk = wz * P.kx;
          const Number wm = wz * P.cm;
          Number wks[H][H], wms[H][H];
#pragma unroll
          for (int a = 0; a < H; ++a)
#pragma unroll
            for (int d = 0; d <= a; ++d) {
              wks[a][d] = wks[d][a] = (P.w[a] * P.w[d]) * wk;
              wms[a][d] = wms[d][a] = (P.w[a] * P.w[d]) * wm;
            }
          auto half = [](int i) { return i < N1 - 1 - i ? i : N1 - 1 - i; };
#pragma unroll
          for (int j = 0; j < N1; ++j)
#pragma unroll
            for (int i = 0; i < N1; ++i) {
              const Number w = wks[half(j)][half(i)];
              kq[j][i] = w * kq[j][i];
              if (N1 == 3 && row == 3) kq[j][i] = Number(0);
              gz[j][i] *= kq[j][i];
            }
          // x derivative and flux row by row, with the mass term
#pragma unroll
          for (int j = 0; j < N1; ++j) {
            Number f[N1];
#pragma unroll
            for (int q = 0; q < N1; ++q) {
              Number g = 0;
#pragma unroll
              for (int i = 0; i < N1; ++i) g = fma(P.D(q, i), v[j][i], g);
              f[q] = kq[j][q] * g;
            }
#pragma unroll
            for (int i = 0; i < N1; ++i) {
              Number a = wms[half(j)][half(i)] * (RES ? w[j][i] : v[j][i]);
#pragma unroll
              for (int q = 0; q < N1; ++q) a = fma(P.D(q, i), f[q], a);
              e[j][i] = a;
            }
          }
          // y derivative and flux column by column
#pragma unroll
          for (int i = 0; i < N1; ++i) {
            Number f[N1];
#pragma unroll
            for (int q = 0; q < N1; ++q) {
              Number g = 0;
#pragma unroll
              for (int j = 0; j < N1; ++j) g = fma(P.D(q, j), v[j][i], g);
              f[q] = kq[q][i] * g;
            }
#pragma unroll
            for (int j = 0; j < N1; ++j) {
              Number a = e[j][i];
#pragma unroll
              for (int q = 0; q < N1; ++q) a = fma(P.Dy(q, j), f[q], a);
              e[j][i] = a;
            }
          }
        }
        // ---- back to the DoFs ----
        z_backward<N1>(P, zt, e, gz, v);
        sweep_y<N1, true, false>(P.S, v, e);
        sweep_x<N1, true, false>(P.S, e, v);
      }
      // ---- sums over the brick's cells ----
      const int f = opaque(flags);
      double r[N1][N1];
#pragma unroll
      for (int j = 0; j < N1; ++j)
#pragma unroll
        for (int i = 0; i < N1; ++i) r[j][i] = (double)v[j][i];
      double(&yr)[N1][64] = yrow[wave][pen];
      if (cy > cy0) {
#pragma unroll
        for (int i = 0; i < N1; ++i) r[0][i] += yr[i][lane];
      }
      if (!last) {
#pragma unroll
        for (int i = 0; i < N1; ++i) yr[i][lane] = r[K][i];
      }
#pragma unroll
      for (int j = 0; j < N1; ++j) {
        if (j == K && !last) continue;
        r[j][0] += from_previous_cell(r[j][K], pen > 0 ? xcol[wave][j][row] : 0.0);
      }
      if (cxb + kNX < cx_end && (f & F_LAST)) {
#pragma unroll
        for (int j = 0; j < N1; ++j)
          if (j < K || last) xcol[wave][j][row] = r[j][K];
      }
      double(&tp)[B::ZC][K][N1][kNX] = top[parity];
      if (f & F_TOP) {
#pragma unroll
        for (int j = 0; j < K; ++j)
#pragma unroll
          for (int i = 0; i < N1; ++i) tp[zc][j][i][c] = r[j][i];
      }
      __syncthreads();
      if (f & F_LOW) {
#pragma unroll
        for (int j = 0; j < K; ++j)
#pragma unroll
          for (int i = 0; i < N1; ++i) r[j][i] += tp[zc - 1][j][i][c];
      }
      if (last) {  // the top row takes another round
        __syncthreads();
        if (f & F_TOP) {
#pragma unroll
          for (int i = 0; i < N1; ++i) tp[zc][0][i][c] = r[K][i];
        }
        __syncthreads();
        if (f & F_LOW) {
#pragma unroll
          for (int i = 0; i < N1; ++i) r[K][i] += tp[zc - 1][0][i][c];
        }
      }
      const auto &Z = fresh_args<BrickArgs<Number, N1>>();
      const bool hy = cy != Z.nc[1] - 1;  // the top row is not the mesh's
      if constexpr (RES) {
#pragma unroll
        for (int j = 0; j < N1; ++j)
#pragma unroll
          for (int i = 0; i < N1; ++i) r[j][i] = -r[j][i];
      }
      // dst = x, or dst += x (RES); the classes are always stored
      auto put = [&](Number *p, Number x, bool owner) { *p = RES && owner ? *p + x : x; };
      constrain(cxb, cy, r);

      // ---- store rows 0..K-1, and the top row after the last step: to dst, or to the class of the
      //      brick's upper y / z plane ----
      if constexpr (K == 1) {
        // the lanes already hold consecutive columns
        const int cx = cxb + c;
        if ((f & F_STORE) && cx < Z.nc[0]) {
          const bool hz = f & F_HZ;
          Number *o = (hz ? Z.scratch + Z.g.off[4] + (long)bz * sz : dst + sz * iz) + cx;
          put(o + sy * cy, (Number)r[0][0], !hz);
          if (last) {
            Number *t = !hy ? o + sy * (cy + 1)
                            : Z.scratch + (hz ? Z.g.off[6] + ((long)by + (long)(Z.g.nb[1] - 1) * bz) * sy
                                              : Z.g.off[2] + ((long)by + (long)(Z.g.nb[1] - 1) * iz) * sy) + cx;
            put(t, (Number)r[1][0], !hz && !hy);
          }
        }
      } else {
        constexpr int RPI = 64 / W;    // rows stored at a time
        Number *const tl = buf[wave];  // [lane row][j of RPI][x]
        const int x = lane % W, jr = lane / W, czw = bz * B::ZC + wave;
        if (czw < Z.nc[2]) {
          const long at = sy * ((long)K * cy) + K * cxb;  // uniform
          const int mine = x + (int)sy * jr;
          const bool st = jr < RPI && x < K * (cx_end - cxb);
          Number *o = dst + (sz * (K * czw) + at) + mine;
          const bool end = czw == Z.nc[2] - 1;
          Number *oz = end ? o + sz * K : Z.scratch + (Z.g.off[4] + (long)bz * sz + at) + mine;
          const Number *t = tl + lane;
#pragma unroll
          for (int j = 0; j < K; j += RPI) {
#pragma unroll
            for (int k = j; k < j + RPI; ++k)
#pragma unroll
              for (int i = 0; i < K; ++i) tl[(row * RPI + k - j) * W + K * c + i] = (Number)r[k][i];
            lds_fence();
            if (st) {
#pragma unroll
              for (int rw = 0; rw < K; ++rw) put(o + sz * rw + sy * j, t[rw * RPI * W], true);
              if (end || wave == kNW - 1) put(oz + sy * j, t[K * RPI * W], end);
            }
            lds_fence();
          }
          if (last) {
#pragma unroll
            for (int i = 0; i < K; ++i) tl[row * W + K * c + i] = (Number)r[K][i];
            lds_fence();
#pragma unroll
            for (int rw = 0; rw < N1; ++rw) {
              const int z = K * czw + rw;
              const bool up = rw == K && czw != Z.nc[2] - 1;
              if (up && wave != kNW - 1) continue;
              Number *p;
              if (hy)
                p = Z.scratch + (up ? Z.g.off[6] + ((long)by + (long)(Z.g.nb[1] - 1) * bz) * sy
                                    : Z.g.off[2] + ((long)by + (long)(Z.g.nb[1] - 1) * z) * sy);
              else
                p = (up ? Z.scratch + Z.g.off[4] + (long)bz * sz : dst + sz * z) + sy * ((long)K * cy + K);
              if (jr == 0 && x < K * (cx_end - cxb)) put(p + K * cxb + x, tl[rw * W + x], !hy && !up);
            }
            lds_fence();
          }
        }
      }
      // ---- column K of the brick's last cells: to dst at the mesh's end, else to the x classes ----
      if (cxb + kNX >= cx_end) {
        const int cx = cxb + c;
        if ((f & F_STORE) && cx == cx_end - 1) {
          const bool hx = cx_end != Z.nc[0], hz = f & F_HZ;
          const long ny1 = Z.g.nb[1] - 1, nz1 = Z.g.nb[2] - 1;
#pragma unroll
          for (int j = 0; j < N1; ++j) {
            if (j == K && !last) continue;
            const bool y = j == K && hy;
            const int iy = K * cy + j;
            Number *o;
            if (hx) {
              if (y) o = Z.scratch + (hz ? Z.g.off[7] + (bx * ny1 + by) * nz1 + bz : Z.g.off[3] + (bx * ny1 + by) * Z.nd[2] + iz);
              else o = Z.scratch + (hz ? Z.g.off[5] + (bx * nz1 + bz) * Z.nd[1] + iy : Z.g.off[1] + ((long)bx * Z.nd[2] + iz) * Z.nd[1] + iy);
            } else {
              if (y) o = Z.scratch + (hz ? Z.g.off[6] + (by + ny1 * bz) * sy : Z.g.off[2] + (by + ny1 * iz) * sy);
              else o = (hz ? Z.scratch + Z.g.off[4] + (long)bz * sz : dst + sz * iz) + sy * iy;
              o += K * cx + K;
            }
            put(o, (Number)r[j][K], !hx && !y && !hz);
          }
        }
      }
    }
  }
}

// ---- the apply of Q1 and Q2 on Cartesian cells: one lane per cell ----

// sweep of a cell's values [z][y][x] along direction DIR (0 x, 1 y, 2 z)
template <int N1, int DIR, bool TR, bool ADD, typename Number, typename Mat>
__device__ __forceinline__ void sweep_cell(const Mat &M, const Number (&in)[N1][N1][N1], Number (&out)[N1][N1][N1]) {
#pragma unroll
  for (int a = 0; a < N1; ++a)
#pragma unroll
    for (int b = 0; b < N1; ++b) {
      auto at = [&](auto &v, int t) -> auto & { return DIR == 0 ? v[a][b][t] : (DIR == 1 ? v[a][t][b] : v[t][a][b]); };
#pragma unroll
      for (int q = 0; q < N1; ++q) {
        Number s = ADD ? at(out, q) : Number(0);
#pragma unroll
        for (int t = 0; t < N1; ++t) s = fma(TR ? M(t, q) : M(q, t), at(in, t), s);
        at(out, q) = s;
      }
    }
}
// f(z, y, x) for every value or point of a cell
template <int N1, typename F> __device__ __forceinline__ void for_cell(F f) {
#pragma unroll
  for (int l = 0; l < N1; ++l)
#pragma unroll
    for (int j = 0; j < N1; ++j)
#pragma unroll
      for (int i = 0; i < N1; ++i) f(l, j, i);
}
// values at the points of the field in u (u is overwritten)
template <int N1, typename Number, typename Mat>
__device__ __forceinline__ void cell_to_points(const Mat &S, Number (&u)[N1][N1][N1], Number (&v)[N1][N1][N1]) {
  sweep_cell<N1, 0, false, false>(S, u, v);
  sweep_cell<N1, 1, false, false>(S, v, u);
  sweep_cell<N1, 2, false, false>(S, u, v);
}
// e += D^T (k * (D v)) along DIR
template <int N1, int DIR, typename Number, typename Mat, typename MatT>
__device__ __forceinline__ void flux_cell(const Mat &D, const MatT &Dt, const Number (&v)[N1][N1][N1], const Number (&k)[N1][N1][N1],
                                          Number (&e)[N1][N1][N1]) {
#pragma unroll
  for (int a = 0; a < N1; ++a)
#pragma unroll
    for (int b = 0; b < N1; ++b) {
      auto at = [&](auto &x, int t) -> auto & { return DIR == 0 ? x[a][b][t] : (DIR == 1 ? x[a][t][b] : x[t][a][b]); };
      Number f[N1];
#pragma unroll
      for (int q = 0; q < N1; ++q) {
        Number g = 0;
#pragma unroll
        for (int t = 0; t < N1; ++t) g = fma(D(q, t), at(v, t), g);
        f[q] = at(k, q) * g;
      }
#pragma unroll
      for (int t = 0; t < N1; ++t)
#pragma unroll
        for (int q = 0; q < N1; ++q) at(e, t) = fma(Dt(q, t), f[q], at(e, t));
    }
}
// value of a lower lane (the cell below in z)
__device__ __forceinline__ double from_lane(double x, int lane) {
  const int lo = __builtin_amdgcn_ds_bpermute(4 * lane, __double2loint(x));
  const int hi = __builtin_amdgcn_ds_bpermute(4 * lane, __double2hiint(x));
  return __hiloint2double(hi, lo);
}

// A whole cell per lane: a wavefront (= workgroup) holds LX x 64 / LX cells (x, z) and marches along y, pencils of
// LX cells side by side along x done one after the other. All sweeps are register-local: per 64 cells Q2
// takes half the VALU instructions of the kernel above, whose lane rows hold four planes, and there is no
// barrier. What bounds it: the VALU, at few wavefronts per SIMD (Q2 FP64: two with one k per cell, 235 registers;
// one with k per point or a law, 320 and 346; Q2 FP32 two or three; Q1 FP64 two to four, FP32 four). Against the
// kernel above with these degrees: Q2 100^3 k per point FP64 178 -> 140 us, FP32 126 -> 79 us (101 us for a
// kernel with LDS transposes between the sweeps), with a law FP32 196 -> 118 us (136), Q2 64^3 one k per cell
// FP32 29 -> 24 us, Q1 112 x 116 x 132 k per point FP32 47 -> 33 us (40). Mapped cells, the residual and the
// tangent have more values per point than fit (Q2 FP64: tangent of 70 x 50 x 33 47 -> 123 us, mapped
// 100 x 80 x 70 289 -> 316 us, residual with a law 80 us both) and stay above, as does Q3.
template <int N1, typename Number, int KMODE, int LX>
__global__ __launch_bounds__(64) void heat_cells_kernel(const BrickArgs<Number, N1> P, const Number *__restrict__ src,
                                                        Number *__restrict__ dst) {
  constexpr int K = N1 - 1, NQ = N1 * N1 * N1, LZ = 64 / LX;
  constexpr bool TENSOR = KMODE == KAPPA_CONST || KMODE == KAPPA_CELL;
  __shared__ double yrow[kMaxPencils][N1 * N1][64];  // top rows of the previous y step's cells
  __shared__ double xcol[N1 * N1][LZ];          // last x column of the previous pencil
  const int lane = threadIdx.x, c = lane % LX, zc = lane / LX;
  const int nbr = gridDim.x, xcd = blockIdx.x & 7;
  int b = xcd * (nbr >> 3) + min(xcd, nbr & 7) + (blockIdx.x >> 3);
  const int bx = b % P.g.nb[0];
  b /= P.g.nb[0];
  const int by = b % P.g.nb[1], bz = b / P.g.nb[1];
  const int cz = bz * LZ + zc, cy0 = by * P.g.cells[1], cx0 = bx * P.g.cells[0];
  const int cy_end = min(cy0 + P.g.cells[1], P.nc[1]), cx_end = min(cx0 + P.g.cells[0], P.nc[0]);
  const long sy = P.nd[0], sz = (long)P.nd[0] * P.nd[1];
  // lanes without a cell work on the mesh's last one: sums pass upwards in x and z only
  const int czc = min(cz, P.nc[2] - 1);
  // constrained planes that touch the brick
  int bmask = P.dmask;
  if (cx0 > 0) bmask &= ~1;
  if (cx_end < P.nc[0]) bmask &= ~2;
  if (cy0 > 0) bmask &= ~4;
  if (cy_end < P.nc[1]) bmask &= ~8;
  if (bz > 0) bmask &= ~16;
  if (bz + 1 < P.g.nb[2]) bmask &= ~32;
  // ... that touch the cell: zero plane l's DoFs on them
  auto constrain_plane = [&](int cx, int cy, int l, auto &u) {
    int m = bmask;
    if (cx > 0) m &= ~1;
    if (cx + 1 < P.nc[0]) m &= ~2;
    if (cy > 0) m &= ~4;
    if (cy + 1 < P.nc[1]) m &= ~8;
    if (cz > 0) m &= ~16;
    if (cz + 1 < P.nc[2]) m &= ~32;
#pragma unroll
    for (int j = 0; j < N1; ++j)
#pragma unroll
      for (int i = 0; i < N1; ++i) {
        const int faces = (i == 0 ? 1 : 0) | (i == K ? 2 : 0) | (j == 0 ? 4 : 0) | (j == K ? 8 : 0) | (l == 0 ? 16 : 0) |
                          (l == K ? 32 : 0);
        if (m & faces) u[j][i] = 0;
      }
  };
  auto constrain = [&](int cx, int cy, Number (&u)[N1][N1][N1]) {
    if (bmask) {
#pragma unroll
      for (int l = 0; l < N1; ++l) constrain_plane(cx, cy, l, u[l]);
    }
  };
  auto cell_dofs = [&](const Number *field, int cx, int cy) {
    return field + sz * ((long)K * czc) + sy * ((long)K * cy) + K * min(cx, P.nc[0] - 1);
  };
  auto load = [&](const Number *field, int cx, int cy, Number (&u)[N1][N1][N1]) {
    const Number *p = cell_dofs(field, cx, cy);
    for_cell<N1>([&](int l, int j, int i) { u[l][j][i] = p[sz * l + sy * j + i]; });
  };
  auto half = [](int a) { return a < N1 - 1 - a ? a : N1 - 1 - a; };
  for (int cy = cy0; cy < cy_end; ++cy) {
    const bool last = cy + 1 == cy_end;
    int pen = 0;
    for (int cxb = cx0; cxb < cx_end; cxb += LX, ++pen) {
      const int cx = cxb + c;
      const long cell = min(cx, P.nc[0] - 1) + (long)P.nc[0] * (cy + (long)P.nc[1] * czc);
      Number u[N1][N1][N1], v[N1][N1][N1];
      load(src, cx, cy, u);
      constrain(cx, cy, u);
      if constexpr (TENSOR) {
        // a conductivity that is constant on a Cartesian cell:
        // J u = M_x [M_y (c_m M_z + k k_z K_z) + k k_y K_y M_z] u + k k_x K_x M_y M_z u
        const Number kc = KMODE == KAPPA_CELL ? P.kappa_arr[cell] : P.kappa;
        const Number kx = kc * P.kx, ky = kc * P.ky, kz = kc * P.kz;
        Number m[N1][N1][N1], p[N1][N1][N1];
        sweep_cell<N1, 2, false, false>(P.K1, u, p);
        sweep_cell<N1, 2, false, false>(P.M1, u, m);
        for_cell<N1>([&](int l, int j, int i) { p[l][j][i] = fma(P.cm, m[l][j][i], kz * p[l][j][i]); });
        sweep_cell<N1, 1, false, false>(P.M1, m, u);
        sweep_cell<N1, 1, false, false>(P.M1, p, v);
        for_cell<N1>([&](int l, int j, int i) {
          m[l][j][i] *= ky;
          u[l][j][i] *= kx;
        });
        sweep_cell<N1, 1, false, true>(P.K1, m, v);
        sweep_cell<N1, 0, false, false>(P.M1, v, m);
        sweep_cell<N1, 0, false, true>(P.K1, u, m);
        for_cell<N1>([&](int l, int j, int i) { v[l][j][i] = m[l][j][i]; });
      } else {
        Number e[N1][N1][N1], k[N1][N1][N1];
        if constexpr (KMODE == KAPPA_LAW) {
          load(P.T, cx, cy, k);
          cell_to_points<N1>(P.S, k, v);
          for_cell<N1>([&](int l, int j, int i) { k[l][j][i] = law_kappa<Number>(P.law, P.law_p, v[l][j][i]); });
        } else {
          const Number *p = P.kappa_arr + cell * NQ;
          for_cell<N1>([&](int l, int j, int i) { k[l][j][i] = p[(N1 * l + j) * N1 + i]; });
        }
        cell_to_points<N1>(P.S, u, v);
        // at the points (heat_diffuse_operator.cpp:1029-1077): e = c_m W v + D^T f
        for_cell<N1>([&](int l, int j, int i) {
          const Number w = (P.w[half(l)] * P.w[half(j)]) * P.w[half(i)];
          k[l][j][i] *= w * P.kx;
          e[l][j][i] = (w * P.cm) * v[l][j][i];
        });
        flux_cell<N1, 0>(P.D, P.D, v, k, e);
        flux_cell<N1, 1>(P.D, P.Dy, v, k, e);
        flux_cell<N1, 2>(P.D, P.Gz, v, k, e);  // (Gz: here the collocation derivative times k_z / k_x)
        sweep_cell<N1, 2, true, false>(P.S, e, u);
        sweep_cell<N1, 1, true, false>(P.S, u, e);
        sweep_cell<N1, 0, true, false>(P.S, e, v);
      }
      // ---- per plane, from the top: sums over the brick's cells (along y through LDS, along x to the next
      //      lane, along z to the next row of lanes), then the stores: to dst, or to the classes of the brick's
      //      upper planes ----
      const bool more = cxb + LX < cx_end, hy = last && cy_end != P.nc[1], hx = cx_end != P.nc[0];
      const bool on = cx < P.nc[0] && cz < P.nc[2], end_z = cz == P.nc[2] - 1, end_x = cx == cx_end - 1;
      const long ny1 = P.g.nb[1] - 1, nz1 = P.g.nb[2] - 1;
      double up[N1][N1];
#pragma unroll
      for (int l = K; l >= 0; --l) {
        double r[N1][N1];
#pragma unroll
        for (int j = 0; j < N1; ++j)
#pragma unroll
          for (int i = 0; i < N1; ++i) r[j][i] = (double)v[l][j][i];
        if (cy > cy0) {
#pragma unroll
          for (int i = 0; i < N1; ++i) r[0][i] += yrow[pen][N1 * l + i][lane];
        }
        if (!last) {
#pragma unroll
          for (int i = 0; i < N1; ++i) yrow[pen][N1 * l + i][lane] = r[K][i];
        }
#pragma unroll
        for (int j = 0; j < N1; ++j) {
          if (j == K && !last) continue;
          const double carried = pen > 0 ? xcol[N1 * l + j][zc] : 0.0, left = from_previous_cell(r[j][K], carried);
          r[j][0] += c == 0 ? carried : left;
          if (more && c == LX - 1) xcol[N1 * l + j][zc] = r[j][K];
#pragma unroll
          for (int i = 0; i < N1; ++i) {
            if (l == K) up[j][i] = from_lane(r[j][i], lane - LX);
            if (l == 0) r[j][i] += zc > 0 ? up[j][i] : 0.0;
          }
        }
        if (bmask) constrain_plane(cx, cy, l, r);
        if (!on || (l == K && !end_z && zc != LZ - 1)) continue;
        const bool hz = l == K && !end_z;
        const int iz = K * cz + l;
#pragma unroll
        for (int j = 0; j < N1; ++j) {
          if (j == K && !last) continue;
          const bool y = j == K && hy;
          const int iy = K * cy + j;
          Number *o = (hz ? P.scratch + P.g.off[4] + bz * sz : dst + sz * iz) + sy * iy;
          if (y) o = P.scratch + (hz ? P.g.off[6] + (by + ny1 * bz) * sy : P.g.off[2] + (by + ny1 * iz) * sy);
          o += K * cx;
#pragma unroll
          for (int i = 0; i < K; ++i) o[i] = (Number)r[j][i];
          if (end_x) {
            o += K;
            if (hx) {
              if (y) o = P.scratch + (hz ? P.g.off[7] + (bx * ny1 + by) * nz1 + bz : P.g.off[3] + (bx * ny1 + by) * P.nd[2] + iz);
              else o = P.scratch + (hz ? P.g.off[5] + (bx * nz1 + bz) * P.nd[1] + iy : P.g.off[1] + ((long)bx * P.nd[2] + iz) * P.nd[1] + iy);
            }
            *o = (Number)r[j][K];
          }
        }
      }
      if (more) lds_fence();  // (xcol: other lanes read it)
    }
  }
}

// dst += the classes of the planes bricks share, in class order (sums in FP64). A wavefront takes up
// to 64 kFixup DoFs of a line: of an x row of the shared z planes, then of the shared y planes (rows
// off the z planes), then of a y line of the shared x planes (off both). All its loads are issued
// before the sums and stores.
constexpr int kFixup = 4;
template <typename Number>
__global__ __launch_bounds__(256) void brick_fixup_kernel(Number *__restrict__ dst, const Number *__restrict__ scratch,
                                                          BrickGrid g, int K, int nd0, int nd1, int nd2, int parts) {
  const int lane = threadIdx.x & 63;
  long line = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  const int i0 = (int)(line % parts) * (64 * kFixup) + lane;
  line /= parts;
  const long nz = (long)(g.nb[2] - 1) * nd1, ny = (long)(g.nb[1] - 1) * nd2, nx = (long)(g.nb[0] - 1) * nd2;
  const int px = K * g.cells[0], py = K * g.cells[1], pz = K * g.cells[2];
  const long sy = nd0, sz = (long)nd0 * nd1;
  // the shared plane a coordinate lies on (-1: none): the multiples of p inside the mesh
  auto plane = [](int i, int p, int nb) { return i > 0 && i % p == 0 && i / p < nb ? i / p - 1 : -1; };
  int iy = -1, iz = -1, hy = -1, hz = -1;
  if (line < nz) {
    hz = (int)(line / nd1);
    iy = (int)(line - (long)hz * nd1);
    iz = pz * (hz + 1);
    hy = plane(iy, py, g.nb[1]);
  } else if ((line -= nz) < ny) {
    iz = (int)(line / (g.nb[1] - 1));
    hy = (int)(line - (long)iz * (g.nb[1] - 1));
    iy = py * (hy + 1);
    if (plane(iz, pz, g.nb[2]) >= 0) return;
  } else if ((line -= ny) < nx) {
    const int hx = (int)(line / nd2);
    iz = (int)(line - (long)hx * nd2);
    if (plane(iz, pz, g.nb[2]) >= 0) return;
    const Number *s = scratch + g.off[1] + line * nd1;
    Number *d = dst + (long)px * (hx + 1) + sz * iz;
    Number a[kFixup], b[kFixup];
#pragma unroll
    for (int t = 0; t < kFixup; ++t) {
      const int i = min(i0 + 64 * t, nd1 - 1);
      a[t] = d[sy * i];
      b[t] = s[i];
    }
#pragma unroll
    for (int t = 0; t < kFixup; ++t) {
      const int i = i0 + 64 * t;
      if (i < nd1 && plane(i, py, g.nb[1]) < 0) d[sy * i] = (Number)((double)a[t] + (double)b[t]);
    }
    return;
  } else {
    return;
  }
  Number *d = dst + sy * iy + sz * iz;
  const Number *cy = scratch + g.off[2] + (hy + (long)(g.nb[1] - 1) * iz) * nd0;
  const Number *cz = scratch + g.off[4] + ((long)hz * nd1 + iy) * nd0;
  const Number *cyz = scratch + g.off[6] + (hy + (long)(g.nb[1] - 1) * hz) * nd0;
  Number a[kFixup], b[kFixup], e[kFixup], f[kFixup];
#pragma unroll
  for (int t = 0; t < kFixup; ++t) {
    const int ix = min(i0 + 64 * t, nd0 - 1);
    a[t] = d[ix];
    b[t] = hy >= 0 ? cy[ix] : Number(0);
    e[t] = hz >= 0 ? cz[ix] : Number(0);
    f[t] = hy >= 0 && hz >= 0 ? cyz[ix] : Number(0);
  }
#pragma unroll
  for (int t = 0; t < kFixup; ++t) {
    const int ix = i0 + 64 * t;
    if (ix >= nd0) continue;
    const int hx = plane(ix, px, g.nb[0]);
    double s = (double)a[t];
    if (hx >= 0) s += (double)scratch[g.off[1] + ((long)hx * nd2 + iz) * nd1 + iy];
    s += (double)b[t];
    if (hx >= 0 && hy >= 0) s += (double)scratch[g.off[3] + ((long)hx * (g.nb[1] - 1) + hy) * nd2 + iz];
    s += (double)e[t];
    if (hx >= 0 && hz >= 0) s += (double)scratch[g.off[5] + ((long)hx * (g.nb[2] - 1) + hz) * nd1 + iy];
    s += (double)f[t];
    if (hx >= 0 && hy >= 0 && hz >= 0)
      s += (double)scratch[g.off[7] + ((long)hx * (g.nb[1] - 1) + hy) * (g.nb[2] - 1) + hz];
    d[ix] = (Number)s;
  }
}

template <int N1> struct TangentPoints {
  BrickArgs<double, N1> A;
  mpdg_heat_material mat;
  double rdt, vol, rh[3], vel[3];  // 1 / dt, 1 / h: a division per point and term would take most of the time
  const double *vf;
  long n_dofs;
};

// The tangent's coefficients (tangent.hip) at the points of Q1..Q3 cells. One wavefront per pencil of 16
// cells along x in the apply's lane layout, so that a coefficient of 16 cells is stored at once. What bounds
// it: the stores, 6 of the 8 values per point with a constant velocity (Q2 70 x 50 x 33 with solidification,
// 150 MB: 54 us with 8 values and the lanes of a cell side by side, 35 us here; 49 us with three wavefronts per
// SIMD, which spill. Stored past the caches it is no faster and the apply that follows takes 77 us, not 56).
template <int N1>
__global__ __launch_bounds__(64 * kNW) __attribute__((amdgpu_waves_per_eu(N1 == 4 ? 1 : 2)))
void tangent_points_kernel(const TangentPoints<N1> X, const double *__restrict__ T,
                                                                  const double *__restrict__ T_old, double *__restrict__ td) {
  using B = BrickShape<N1>;
  constexpr int K = B::K, NQ = N1 * N1 * N1;
  const auto &P = X.A;
  const int lane = threadIdx.x & 63, row = lane >> 4, c = lane & 15, l = N1 == 2 ? row & 1 : row;
  const int px = (P.nc[0] + kNX - 1) / kNX, pz = (P.nc[2] + B::ZPW - 1) / B::ZPW;
  long p = (long)blockIdx.x * kNW + (threadIdx.x >> 6);
  if (p >= (long)px * P.nc[1] * pz) return;
  const int cxb = kNX * (int)(p % px);
  p /= px;
  const int cy = (int)(p % P.nc[1]), cz = B::ZPW * (int)(p / P.nc[1]) + (N1 == 2 ? row >> 1 : 0);
  // lanes without a cell work on the mesh's last one and store nothing; Q2's idle row holds zeros
  const int cx = min(cxb + c, P.nc[0] - 1);
  const long sy = P.nd[0], at = K * cx + sy * ((long)K * cy + P.nd[1] * ((long)K * min(cz, P.nc[2] - 1) + min(l, K)));
  auto load = [&](const double *f, double (&u)[N1][N1]) {
#pragma unroll
    for (int j = 0; j < N1; ++j)
#pragma unroll
      for (int i = 0; i < N1; ++i) u[j][i] = N1 != 3 || row < 3 ? f[at + i + sy * j] : 0.0;
  };
  const ZTables<N1, double> zt(P, P.S, P.G, lane);
  auto to_points = [&](const double *f, double (&v)[N1][N1]) {
    double u[N1][N1], t[N1][N1];
    load(f, u);
    sweep_x<N1, false, false>(P.S, u, t);
    sweep_y<N1, false, false>(P.S, t, u);
    z_forward<N1, false>(P.S, P.G, zt, u, v, v);
  };
  double v[N1][N1], g[3][N1][N1], r[N1][N1];
  {
    double u[N1][N1], t[N1][N1];
    load(T, u);
    sweep_x<N1, false, false>(P.S, u, t);
    sweep_y<N1, false, false>(P.S, t, u);
    z_forward<N1, true>(P.S, P.G, zt, u, v, g[2]);
    sweep_x<N1, false, false>(P.D, v, g[0]);
    sweep_y<N1, false, false>(P.D, v, g[1]);
  }
  // r = (T - T_old) / dt + grad T . velocity, the factor of d rho c_p / dT
  const bool solid = P.solid;
  if (solid) {
    to_points(T_old, r);
#pragma unroll
    for (int j = 0; j < N1; ++j)
#pragma unroll
      for (int i = 0; i < N1; ++i) {
        r[j][i] = (v[j][i] - r[j][i]) * X.rdt;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          g[d][j][i] *= X.rh[d];
          if (!X.vf) r[j][i] += g[d][j][i] * X.vel[d];
        }
      }
  }
  const bool mine = cxb + c < P.nc[0] && cz < P.nc[2] && l <= K;
  long block = (unsigned)cxb / kNX + (long)((unsigned)P.nc[0] / kNX) * (cy + (long)P.nc[1] * cz);
  int place = c;
  if (cxb + kNX > P.nc[0]) block = point_block(P.nc[0], cy + (long)P.nc[1] * min(cz, P.nc[2] - 1), (long)P.nc[1] * P.nc[2], cx, place);
  double *const out = td + (block * kTangentCoeffs * NQ + l) * kNX + place;
  auto put = [&](int comp, int j, int i, double x) {
    if (mine) out[(comp * NQ + (N1 * j + i) * N1) * kNX] = x;
  };
  double wz = 0.0;
#pragma unroll
  for (int a = 0; a < N1; ++a) wz = l == a ? P.w[a < N1 - 1 - a ? a : N1 - 1 - a] : wz;
  auto weight = [&](int j, int i) {
    return X.vol * wz * P.w[j < N1 - 1 - j ? j : N1 - 1 - j] * P.w[i < N1 - 1 - i ? i : N1 - 1 - i];
  };
  if (X.vf) {
    double rc[N1][N1];
#pragma unroll
    for (int j = 0; j < N1; ++j)
#pragma unroll
      for (int i = 0; i < N1; ++i) {
        double k, drc, dk;
        material(X.mat, v[j][i], rc[j][i], k, drc, dk);
      }
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      double w[N1][N1];
      to_points(X.vf + d * X.n_dofs, w);
#pragma unroll
      for (int j = 0; j < N1; ++j)
#pragma unroll
        for (int i = 0; i < N1; ++i) {
          if (solid) r[j][i] += g[d][j][i] * w[j][i];
          put(2 + d, j, i, weight(j, i) * rc[j][i] * w[j][i] * X.rh[d]);
        }
    }
  }
#pragma unroll
  for (int j = 0; j < N1; ++j)
#pragma unroll
    for (int i = 0; i < N1; ++i) {
      const double JxW = weight(j, i);
      double rc, k, drc, dk;
      material(X.mat, v[j][i], rc, k, drc, dk);
      double m = rc * X.rdt;
      if (solid) m += drc * r[j][i];
      put(0, j, i, JxW * m);
      put(1, j, i, JxW * k);
      if (P.conv == 1) put(2, j, i, JxW * rc);
      if (solid) {
#pragma unroll
        for (int d = 0; d < 3; ++d) put(5 + d, j, i, JxW * dk * g[d][j][i] * X.rh[d]);
      }
    }
}

// unit: the data per point carries the volume and 1/h (mapped cells, the tangent); cells: for the kernel with
// one cell per lane
template <int N1, typename Number>
int fill_brick_args(const OperatorData<Number> &op, bool unit, BrickArgs<Number, N1> &A, bool cells = false) {
  const FE1D &fe = fe1d(N1 - 1);
  const double vol = unit ? 1.0 : op.h[0] * op.h[1] * op.h[2];
  double Dy[kMaxN1][kMaxN1], Gz[kMaxN1][kMaxN1], M1[kMaxN1][kMaxN1] = {}, K1[kMaxN1][kMaxN1] = {};
  const double ry = unit ? 1.0 : (op.h[0] * op.h[0]) / (op.h[1] * op.h[1]);
  const double rz = unit ? 1.0 : (op.h[0] * op.h[0]) / (op.h[2] * op.h[2]);
  for (int q = 0; q < N1; ++q)
    for (int i = 0; i < N1; ++i) {
      Dy[q][i] = fe.D[q][i] * ry;
      Gz[q][i] = (cells ? fe.D : fe.G)[q][i] * rz;
      for (int j = 0; j < N1; ++j) {
        M1[i][j] += fe.S[q][i] * fe.qw[q] * fe.S[q][j];
        K1[i][j] += fe.G[q][i] * fe.qw[q] * fe.G[q][j];
      }
    }
  A.S.set(fe.S);
  A.D.set(fe.D);
  A.G.set(fe.G);
  A.Dy.set(Dy);
  A.Gz.set(Gz);
  A.M1.set(M1);
  A.K1.set(K1);
  for (int a = 0; 2 * a < N1; ++a) A.w[a] = (Number)fe.qw[a];
  for (int d = 0; d < 3; ++d) {
    A.nc[d] = op.nc[d];
    A.nd[d] = op.nd[d];
  }
  A.n_cells = op.n_cells;
  A.g = brick_grid(N1 - 1, op.nc, cells ? op.brick_cells : op.brick, cells);
  A.dmask = op.dmask;
  A.law = op.law;
  A.cm = (Number)(op.c_mass * vol);
  A.kx = (Number)(unit ? 1.0 : vol / (op.h[0] * op.h[0]));
  A.ky = (Number)(unit ? 1.0 : vol / (op.h[1] * op.h[1]));
  A.kz = (Number)(unit ? 1.0 : vol / (op.h[2] * op.h[2]));
  A.kappa = (Number)op.kappa;
  for (int i = 0; i < 4; ++i) A.law_p[i] = (Number)op.law_p[i];
  A.kappa_arr = op.kappa_arr;
  A.T = op.T;
  A.metric = op.metric;
  A.scratch = op.edge;
  A.T_old = A.q = nullptr;
  A.fa = A.fb = A.fc = Number(0);
  A.conv = A.solid = 0;
  A.vh[0] = A.vh[1] = A.vh[2] = Number(0);
  return A.g.total > 0 && (op.edge == nullptr || (size_t)A.g.total > op.edge_elems) ? MPDG_ERR_INVALID : MPDG_OK;
}

template <int N1, typename Number>
int finish_brick(const BrickArgs<Number, N1> &A, Number *dst, hipStream_t stream) {
  const long lines = (long)(A.g.nb[2] - 1) * A.nd[1] + (long)(A.g.nb[1] - 1) * A.nd[2] + (long)(A.g.nb[0] - 1) * A.nd[2];
  const int longest = A.g.nb[0] > 1 ? std::max(A.nd[0], A.nd[1]) : A.nd[0];
  const int parts = (longest + 64 * kFixup - 1) / (64 * kFixup);
  if (lines > 0)
    hipLaunchKernelGGL(brick_fixup_kernel<Number>, dim3((unsigned)((lines * parts + 3) / 4)), dim3(256), 0, stream, dst,
                       A.scratch, A.g, N1 - 1, A.nd[0], A.nd[1], A.nd[2], parts);
  return hipGetLastError() == hipSuccess ? MPDG_OK : MPDG_ERR_DEVICE;
}
template <int N1, typename Number> dim3 brick_blocks(const BrickArgs<Number, N1> &A) {
  return dim3((unsigned)((long)A.g.nb[0] * A.g.nb[1] * A.g.nb[2]));
}
#define MPDG_BRICK(KM, MP, RES_) \
  hipLaunchKernelGGL((heat_brick_kernel<N1, Number, KM, MP, RES_>), brick_blocks(A), dim3(64 * kNW), 0, stream, A, src, dst)

#define MPDG_APPLY(KM)                                                                                                 \
  do {                                                                                                                 \
    if constexpr (N1 < 4)                                                                                              \
      if (op.brick_cells[2] == 8)                                                                                      \
        hipLaunchKernelGGL((heat_cells_kernel<N1, Number, KM, 8>), brick_blocks(A), dim3(64), 0, stream, A, src, dst); \
      else                                                                                                             \
        hipLaunchKernelGGL((heat_cells_kernel<N1, Number, KM, 16>), brick_blocks(A), dim3(64), 0, stream, A, src, dst); \
    else                                                                                                               \
      MPDG_BRICK(KM, false, false);                                                                                    \
  } while (0)

template <int N1, typename Number>
int launch_brick_n1(const OperatorData<Number> &op, const Number *src, Number *dst, hipStream_t stream,
                    hipEvent_t kernel_start, hipEvent_t kernel_end, BrickSums<Number> *sums) {
  BrickArgs<Number, N1> A;
  const bool cells = N1 < 4 && !op.metric;
  if (const int rc = fill_brick_args(op, op.metric != nullptr, A, cells)) return rc;
  if (kernel_start) (void)hipEventRecord(kernel_start, stream);
  if (op.metric) {
    switch (op.kappa_mode) {
      case KAPPA_CONST: MPDG_BRICK(KAPPA_CONST, true, false); break;
      case KAPPA_CELL: MPDG_BRICK(KAPPA_CELL, true, false); break;
      default: return MPDG_ERR_INVALID;  // per-qp conductivity on mapped meshes runs through metric_k
    }
  } else {
    switch (op.kappa_mode) {
      case KAPPA_CONST: MPDG_APPLY(KAPPA_CONST); break;
      case KAPPA_QP: MPDG_APPLY(KAPPA_QP); break;
      case KAPPA_CELL: MPDG_APPLY(KAPPA_CELL); break;
      case KAPPA_LAW: MPDG_APPLY(KAPPA_LAW); break;
      default: return MPDG_ERR_INVALID;
    }
  }
  if (kernel_end) (void)hipEventRecord(kernel_end, stream);
  if (sums && A.g.total > 0 && op.n_dofs < (1l << 31)) {
    *sums = BrickSums<Number>(A.scratch, A.g, N1 - 1, op.nd);
    return hipGetLastError() == hipSuccess ? MPDG_OK : MPDG_ERR_DEVICE;
  }
  return finish_brick(A, dst, stream);
}

template <int N1>
int launch_brick_residual_n1(const OperatorData<double> &op, const double *src, const double *T_old, const double *q, double a,
                             double b, double c, double *dst, hipStream_t stream) {
  using Number = double;
  BrickArgs<Number, N1> A;
  if (const int rc = fill_brick_args(op, false, A)) return rc;
  A.fa = a;
  A.fb = b;
  A.fc = c;
  A.T_old = T_old;
  A.q = q;
  switch (op.kappa_mode) {
    case KAPPA_CONST: MPDG_BRICK(KAPPA_CONST, false, true); break;
    case KAPPA_QP: MPDG_BRICK(KAPPA_QP, false, true); break;
    case KAPPA_CELL: MPDG_BRICK(KAPPA_CELL, false, true); break;
    case KAPPA_LAW: MPDG_BRICK(KAPPA_LAW, false, true); break;
    default: return MPDG_ERR_INVALID;
  }
  return finish_brick(A, dst, stream);
}

template <int N1>
void fill_tangent_args(const OperatorData<double> &op, const double *vel, const double *vfield, int solid, BrickArgs<double, N1> &A) {
  A.conv = tangent_convects(vel, vfield);
  A.solid = solid;
  for (int d = 0; d < 3; ++d) A.vh[d] = vel[d] / op.h[d];
}

// src null: the diagonal
template <int N1>
int launch_brick_tangent_n1(const OperatorData<double> &op, const double *td, const double *vel, const double *vfield, int solid,
                            const double *src, double *dst, hipStream_t stream) {
  using Number = double;
  BrickArgs<Number, N1> A;
  if (const int rc = fill_brick_args(op, true, A)) return rc;
  fill_tangent_args(op, vel, vfield, solid, A);
  A.metric = td;
  A.kx = 1.0 / (op.h[0] * op.h[0]);
  A.ky = 1.0 / (op.h[1] * op.h[1]);
  A.kz = 1.0 / (op.h[2] * op.h[2]);
  if (src) {
    MPDG_BRICK(KAPPA_TANGENT, false, false);
  } else {
    const FE1D &fe = fe1d(N1 - 1);
    double SS[kMaxN1][kMaxN1], SG[kMaxN1][kMaxN1], GG[kMaxN1][kMaxN1];
    for (int q = 0; q < N1; ++q)
      for (int i = 0; i < N1; ++i) {
        SS[i][q] = fe.S[q][i] * fe.S[q][i];
        SG[i][q] = fe.S[q][i] * fe.G[q][i];
        GG[i][q] = fe.G[q][i] * fe.G[q][i];
      }
    A.S.set(SS);
    A.G.set(SG);
    A.M1.set(GG);
    MPDG_BRICK(TANGENT_DIAGONAL, false, false);
  }
  return finish_brick(A, dst, stream);
}
#undef MPDG_APPLY
#undef MPDG_BRICK

template <int N1>
int launch_brick_tangent_data_n1(const OperatorData<double> &op, double dt, const mpdg_heat_material &mat, int solid,
                                 const double *vel, const double *vfield, const double *T, const double *T_old, double *td,
                                 hipStream_t stream) {
  TangentPoints<N1> X;
  X.A.dmask = 0;
  OperatorData<double> plain = op;
  plain.edge = nullptr;
  plain.edge_elems = 0;
  (void)fill_brick_args(plain, false, X.A);  // (no scratch is used)
  fill_tangent_args(op, vel, vfield, solid, X.A);
  X.mat = mat;
  X.rdt = 1.0 / dt;
  X.vol = op.h[0] * op.h[1] * op.h[2];
  for (int d = 0; d < 3; ++d) {
    X.rh[d] = 1.0 / op.h[d];
    X.vel[d] = vel[d];
  }
  X.vf = vfield;
  X.n_dofs = op.n_dofs;
  const long waves = (long)((op.nc[0] + kNX - 1) / kNX) * op.nc[1] * ((op.nc[2] + BrickShape<N1>::ZPW - 1) / BrickShape<N1>::ZPW);
  hipLaunchKernelGGL(tangent_points_kernel<N1>, dim3((unsigned)((waves + kNW - 1) / kNW)), dim3(64 * kNW), 0, stream, X, T,
                     T_old, td);
  return hipGetLastError() == hipSuccess ? MPDG_OK : MPDG_ERR_DEVICE;
}

}  // namespace

// Long bricks share fewer planes and set their tables up less often; short ones give every CU work, and end
// the launch evenly. Taken is the shape with the least modelled time, in steps of one CU: full rounds of
// `resident` workgroups per CU, the rest (no faster than the latency of one workgroup, which shows below
// `latency` per CU), start-up, and the sums of the shared planes (of the x planes, which are strided,
// separately). The constants are fitted to measured times, one set per degree for all its kernels: `resident` is
// not what the compiler lets a CU hold (Q3 FP64 with k per point two workgroups, Q2 FP64 cells with k per point
// four wavefronts). Measured over 28 meshes and kernels: 1.6% above the best shape on average (at most 15%); about
// 2048 workgroups for every mesh: 5.7% (24%) (Q3 75 x 62 x 49 FP32 49.6 -> 45.4 us, mapped Q3 96^3 FP64
// 809 -> 781 us, Q2 and Q3 64^3 and 128^3 the same shapes); one cell per lane: 24 meshes, 2.5% (9%). It depends
// on the mesh only, so every apply of a mesh sums in the same order.
struct BrickModel {
  double resident, latency, startup, planes, x_planes;
};
static void least_time(const BrickModel &m, int k, const int *nc, int lx, int zc, int *brick) {
  const long px = (nc[0] + lx - 1) / lx, nz = (nc[2] + zc - 1) / zc, cus = 256;
  const double nd[3] = {k * (double)nc[0] + 1, k * (double)nc[1] + 1, k * (double)nc[2] + 1};
  const double steps = (double)px * nc[1] * nz / cus;
  double best = 0.0;
  for (long xb = std::min<long>(kMaxPencils, px); xb >= 1; --xb)
    for (long seg = std::min(kMaxSteps, nc[1]); seg >= 1; --seg) {
      const long nx = (px + xb - 1) / xb, ny = (nc[1] + seg - 1) / seg, n = nx * ny * nz;
      const long round = cus * (long)m.resident, rest = n % round;
      double t = (double)(n / round) * m.resident;
      if (rest) t += std::max(m.latency, (double)((rest + cus - 1) / cus));
      t *= (double)(xb * seg) + m.startup;
      t += steps * (m.planes * ((ny - 1) / nd[1] + (nz - 1) / nd[2]) + m.x_planes * (nx - 1) / nd[0]);
      if (best == 0.0 || t < best) {
        best = t;
        brick[0] = (int)xb;
        brick[1] = (int)seg;
      }
    }
}
void choose_brick(int k, const int *nc, int *brick, int *brick_cells) {
  static const BrickModel bricks[4] = {{}, {6, 4, 0.2, 1.0, 8}, {4, 2.5, 0.7, 0.0, 8}, {4, 2.5, 0.2, 0.5, 8}};
  static const BrickModel cells = {12, 12, 0.2, 0.5, 1};
  if (k > 3) return;
  least_time(bricks[k], k, nc, kNX, zc_of(k), brick);
  if (k > 2) return;
  // Pencils of 8 cells where those of 16 leave many lanes without a cell; they load and store shorter runs and
  // share more x planes. Q2 17 x 90 x 90 k per point FP32 31.6 -> 26.8 us, with a law 44.5 -> 35.3; 24 x 50 x 50
  // 16.0 -> 16.1 us (FP64 21.9 -> 20.7); on the other side 56^3 FP64 22.4 -> 25.3 us, 72^3 56.5 -> 52.9 us.
  auto lanes = [&](int lx) { return (nc[0] + lx - 1) / lx * lx * (double)((nc[2] + 64 / lx - 1) / (64 / lx) * (64 / lx)); };
  brick_cells[2] = lanes(16) >= 1.2 * lanes(8) ? 8 : 16;
  least_time(cells, k, nc, brick_cells[2], 64 / brick_cells[2], brick_cells);
}

size_t brick_scratch_elems(int degree, const int *nc, const int *brick, const int *brick_cells) {
  const size_t n = brick_grid(degree, nc, brick, false).total;
  return degree < 3 ? std::max(n, (size_t)brick_grid(degree, nc, brick_cells, true).total) : n;
}

template <typename Number>
int launch_brick(const OperatorData<Number> &op, const Number *src, Number *dst, hipStream_t stream,
                 hipEvent_t kernel_start, hipEvent_t kernel_end, BrickSums<Number> *sums) {
  switch (op.degree) {
    case 1: return launch_brick_n1<2, Number>(op, src, dst, stream, kernel_start, kernel_end, sums);
    case 2: return launch_brick_n1<3, Number>(op, src, dst, stream, kernel_start, kernel_end, sums);
    case 3: return launch_brick_n1<4, Number>(op, src, dst, stream, kernel_start, kernel_end, sums);
    default: return MPDG_ERR_INVALID;
  }
}
template int launch_brick<double>(const OperatorData<double> &, const double *, double *, hipStream_t, hipEvent_t, hipEvent_t,
                                  BrickSums<double> *);
template int launch_brick<float>(const OperatorData<float> &, const float *, float *, hipStream_t, hipEvent_t, hipEvent_t,
                                 BrickSums<float> *);

int launch_brick_residual(const OperatorData<double> &op, const double *T, const double *T_old, const double *q, double a,
                          double b, double c, double *dst, hipStream_t stream) {
  if (op.metric) return MPDG_ERR_INVALID;
  switch (op.degree) {
    case 1: return launch_brick_residual_n1<2>(op, T, T_old, q, a, b, c, dst, stream);
    case 2: return launch_brick_residual_n1<3>(op, T, T_old, q, a, b, c, dst, stream);
    case 3: return launch_brick_residual_n1<4>(op, T, T_old, q, a, b, c, dst, stream);
    default: return MPDG_ERR_INVALID;
  }
}
int launch_brick_tangent_data(const OperatorData<double> &op, double dt, const mpdg_heat_material &mat, int solid,
                              const double *vel, const double *vfield, const double *T, const double *T_old, double *td,
                              hipStream_t stream) {
  switch (op.degree) {
    case 1: return launch_brick_tangent_data_n1<2>(op, dt, mat, solid, vel, vfield, T, T_old, td, stream);
    case 2: return launch_brick_tangent_data_n1<3>(op, dt, mat, solid, vel, vfield, T, T_old, td, stream);
    case 3: return launch_brick_tangent_data_n1<4>(op, dt, mat, solid, vel, vfield, T, T_old, td, stream);
    default: return MPDG_ERR_INVALID;
  }
}
int launch_brick_tangent(const OperatorData<double> &op, const double *td, const double *vel, const double *vfield, int solid,
                         const double *src, double *dst, hipStream_t stream) {
  switch (op.degree) {
    case 1: return launch_brick_tangent_n1<2>(op, td, vel, vfield, solid, src, dst, stream);
    case 2: return launch_brick_tangent_n1<3>(op, td, vel, vfield, solid, src, dst, stream);
    case 3: return launch_brick_tangent_n1<4>(op, td, vel, vfield, solid, src, dst, stream);
    default: return MPDG_ERR_INVALID;
  }
}

}  // namespace mpdg
