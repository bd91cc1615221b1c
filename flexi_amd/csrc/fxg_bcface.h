// Boundary sides of the fused Gauss-Lobatto split-form stage, per boundary side point (FP64 states, gradients and
// fluxes in the working precision).
#pragma once
#include "fxg_bc.h"
#include "fxg_elem.h"

namespace fxg {

// The outer slot's viscous flux fo, so that with the inner element's half fi it makes the boundary's viscous flux
// (getboundaryflux.f90:561-776): Riemann type 0.5 (f_in + f_b).n with the boundary state's velocity, walls
// f_wall.n with the wall's velocity (none, or the tangential part at a slip wall) and the inner gradients q (slip
// walls: as slip_wall_gradients leaves them; no heat flux at an adiabatic wall). n SurfElem is the side's. Uin: the
// inner face state.
template <class RF>
__device__ __forceinline__ void bc_visc_point(const DevMesh& m, const double* Uin, RF* q, const RF* fi, RF* fo,
                                            const double* bcP, const Gas& gas, size_t fp, int side) {
  const int type = m.bcInfo[2 * side];
  const GasT<RF> gt(gas);
  const RF se = (RF)m.SurfElem[fp];
  const RF nh[3] = {(RF)m.NormVec[3 * fp], (RF)m.NormVec[3 * fp + 1], (RF)m.NormVec[3 * fp + 2]};
  RF ub[3] = {RF(0), RF(0), RF(0)};
  const bool riemann = bc_riemann_type(type);
  if (type == BC_DIRICHLET) {
    const double* ref = m.refPrim + 6 * m.bcInfo[2 * side + 1];
    ub[0] = (RF)ref[1]; ub[1] = (RF)ref[2]; ub[2] = (RF)ref[3];
  } else if (riemann) {  // the boundary state's velocity, as bc_ghost_point formed it
    ub[0] = (RF)bcP[4 * fp + 1]; ub[1] = (RF)bcP[4 * fp + 2]; ub[2] = (RF)bcP[4 * fp + 3];
  } else if (bc_slip_wall(type)) {
    const Prim p = cons_to_prim(Uin, gas);
    const RF vn = (RF)p.u * nh[0] + (RF)p.v * nh[1] + (RF)p.w * nh[2];
    ub[0] = (RF)p.u - vn * nh[0]; ub[1] = (RF)p.v - vn * nh[1]; ub[2] = (RF)p.w - vn * nh[2];
    const RF t1[3] = {(RF)m.TangVec1[3 * fp], (RF)m.TangVec1[3 * fp + 1],
                      (RF)m.TangVec1[3 * fp + 2]};
    const RF t2[3] = {(RF)m.TangVec2[3 * fp], (RF)m.TangVec2[3 * fp + 1],
                      (RF)m.TangVec2[3 * fp + 2]};
    slip_wall_gradients<RF>(type, nh, t1, t2, q);
  }
  RF bx[4], by[4], bz[4];
  diff_flux<RF>(gt, ub[0], ub[1], ub[2], q, q + 4, q + 8, bx, by, bz);
  if (type == BC_WALL_ADIABATIC) bx[3] = by[3] = bz[3] = RF(0);
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const RF fb = (bx[c] * nh[0] + by[c] * nh[1] + bz[c] * nh[2]) * se;
    fo[c] = riemann ? -fb : fi[c] - RF(2) * fb;
  }
}

// The outer slot of a boundary side, from the inner face state Uin and GetBoundaryState
// (getboundaryflux.f90:224-472). Riemann type: the boundary state itself (the Riemann solver and the lifting then
// see it as FLEXI's boundary flux does); its velocity also goes to bcP for bc_visc_point. Walls: a state whose
// lifting variables are 2 f - q_in, f the boundary lifting value (Lifting_GetBoundaryFlux, :855-939), so that the
// BR1 difference (q_out - q_in)/2 is FLEXI's f - q_in; their inviscid flux (0, p_wall n, 0) is formed by the stage
// kernel from bcP.
__device__ __forceinline__ void bc_ghost_point(const DevMesh& m, const double* Uin, double* o, double* bcP, const Gas& gas,
                                             size_t fp, int side) {
  const Prim q = cons_to_prim(Uin, gas);
  const double Pm[6] = {q.rho, q.u, q.v, q.w, q.p, q.T};
  double nv[3], t1[3], t2[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    nv[c] = m.NormVec[3 * fp + c];
    t1[c] = m.TangVec1[3 * fp + c];
    t2[c] = m.TangVec2[3 * fp + c];
  }
  const int type = m.bcInfo[2 * side], st = m.bcInfo[2 * side + 1];
  double Pb[6];
  boundary_state(gas, type, st >= 0 ? m.refPrim + 6 * st : nullptr, m.bcData ? m.bcData + 6 * fp : nullptr,
                 Pm, nv, t1, t2, Pb);
  double G[6];
  double* bp = bcP + 4 * fp;
  if (bc_riemann_type(type)) {
#pragma unroll
    for (int v = 0; v < 6; ++v) G[v] = Pb[v];
    bp[0] = Pb[4]; bp[1] = Pb[1]; bp[2] = Pb[2]; bp[3] = Pb[3];
  } else {
    double F[4];
    boundary_lifting_flux(type, Pm, Pb, F);
    G[0] = Pm[0];
    G[1] = Pm[1] + 2.0 * F[0]; G[2] = Pm[2] + 2.0 * F[1]; G[3] = Pm[3] + 2.0 * F[2];
    G[5] = Pm[5] + 2.0 * F[3];
    G[4] = G[0] * gas.R * G[5];
    bp[0] = Pb[4];
  }
  o[0] = G[0];
  o[1] = G[1] * G[0]; o[2] = G[2] * G[0]; o[3] = G[3] * G[0];
  o[4] = gas.sKappaM1 * G[4] + 0.5 * (o[1] * G[1] + o[2] * G[2] + o[3] * G[3]);
}

}  // namespace fxg
