// Launchers of the full Newton tangent kernels (tangent.hip), Cartesian cells.
#pragma once

#include "kernels.hpp"

namespace mpdg {

// coefficients per quadrature point in the tangent data
constexpr int kTangentCoeffs = 8;

// td: point_data_elems(k + 1, nc, kTangentCoeffs) values (point_data_at). vfield: null (the constant
// vel) or a velocity DoF field, 3 n_dofs values (x, y, z blocks) on the temperature's nodes.
int launch_tangent_data(const OperatorData<double> &op, double dt, const mpdg_heat_material &mat, int solid,
                        const double *vel, const double *vfield, const double *T, const double *T_old, double *td,
                        hipStream_t s);
// dst = J src (dst zeroed first; constrained rows stay 0, constrained src entries read as 0)
// (vel, vfield and solid as given to launch_tangent_data; Q1..Q3 use op.edge)
int launch_tangent_apply(const OperatorData<double> &op, const double *td, const double *vel, const double *vfield, int solid,
                         const double *src, double *dst, hipStream_t s);
// dst += -R(T) (cell part; q may be null)
int launch_tangent_residual(const OperatorData<double> &op, double dt, const mpdg_heat_material &mat,
                            const double *vel, const double *vfield, const double *T, const double *T_old,
                            const double *q, double *dst, hipStream_t s);
// diag = diagonal of the cell part of J (constrained rows: 1)
int launch_tangent_diagonal(const OperatorData<double> &op, const double *td, const double *vel, const double *vfield,
                            int solid, double *diag, hipStream_t s);
// Q1..Q3 (heat_brick.hip); src null: the diagonal (constrained rows 0)
int launch_brick_tangent_data(const OperatorData<double> &op, double dt, const mpdg_heat_material &mat, int solid,
                              const double *vel, const double *vfield, const double *T, const double *T_old, double *td,
                              hipStream_t s);
int launch_brick_tangent(const OperatorData<double> &op, const double *td, const double *vel, const double *vfield, int solid,
                         const double *src, double *dst, hipStream_t s);
// the tangent's convection term: 0 none, 1 a non-zero constant velocity, 2 a velocity field
inline int tangent_convects(const double *vel, const double *vfield) {
  return vfield ? 2 : (vel[0] != 0.0 || vel[1] != 0.0 || vel[2] != 0.0) ? 1 : 0;
}

#ifdef __HIPCC__
// material of the tangent (the oracle's `material`, material.templates.hpp:296-380, :546-598, :765-778)
__device__ __forceinline__ void material(const mpdg_heat_material &m, double T, double &rc, double &k, double &drc,
                                         double &dk) {
  if (m.transition == MPDG_TRANSITION_NONE) {
    rc = m.density[0] * m.specific_heat[0];
    k = m.conductivity[0];
    drc = dk = 0.0;
    return;
  }
  const double inv = 1.0 / (m.liquidus - m.solidus);
  const double fs = fmin(1.0, fmax(0.0, (m.liquidus - T) * inv));
  const bool pure = fs == 0.0 || fs == 1.0;
  const double c = 3.0 * fs * fs - 2.0 * fs * fs * fs, dc = pure ? 0.0 : -inv * (6.0 * fs - 6.0 * fs * fs);
  auto blend = [&](const double *x) { return fs == 0.0 ? x[0] : (fs == 1.0 ? x[1] : x[0] + (x[1] - x[0]) * c); };
  const double rho = blend(m.density), cp = blend(m.specific_heat);
  k = blend(m.conductivity);
  dk = (m.conductivity[1] - m.conductivity[0]) * dc;
  rc = rho * cp;
  drc = (m.specific_heat[1] - m.specific_heat[0]) * dc * rho + (m.density[1] - m.density[0]) * dc * cp;
}
#endif

}  // namespace mpdg
