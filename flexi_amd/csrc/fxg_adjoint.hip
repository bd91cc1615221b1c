// Discrete adjoint of the Gauss-Lobatto split-form right-hand side (the fused stage's arithmetic):
// out = (dUt/dU)^T lam at a state U, written as three element kernels.
//
// Forward, per element and node i (mu_i = -sJ_i lam_i is the adjoint of the accumulated terms):
//   Ut_i = -sJ_i [ sum_d sum_l DVolSurf(l,i) F#(P_i,P_l; Ja^d_i,Ja^d_l)            split Euler part
//                + sum_d sum_l D_Hat_T(l,i) Ja^d_l . f_v(l)                           viscous volume
//                + sum_{faces} L_hat [ ms F*(U_m,U_s) SurfElem + (g_own - g_nb)/2 ] ] surface
//   with P = (rho,u,v,w,p,H), f_v(q, G(q)) the viscous flux of the BR1 gradients G of the
//   lifting variables q = (u,v,w,T), g = f_v . n SurfElem at a face node.
// Reverse:
//   k_adj_euler  split-flux adjoint (each pair's flux depends on sums of the two nodes' primitive
//                variables, so one pair Jacobian serves both nodes), Riemann-flux adjoint per own
//                face point (the hand-written reverse of riemann_rot; with -DFXG_ADJ_DUAL=1
//                directional derivatives in dual numbers instead), the primitive-to-conservative
//                chain; writes out and, per own face point, the parts that belong to the
//                neighbour: XU (its face state) and Xg (its viscous face flux). In the reverse
//                stepper it first applies the previous reverse stage's register update.
//   k_adj_visc   BR1 gradients recomputed; viscous-flux adjoint (volume, own face half, the
//                neighbour's half from Xg); lifting adjoint (transposed line derivatives and face
//                corrections); adds to out, and adds the neighbour's lifting part, taken to its
//                conservative variables, to XU.
//   k_adj_gather adds the neighbours' XU at the face nodes (k_adj_stage_update: and the register
//                update of the last reverse stage).
// References for the forward terms: src/dg/volint.f90:211-371, src/equations/navierstokes/
// splitflux.f90:603-700, riemann.f90:267-855, fillflux.f90:40-215, surfint.t90:471-616,
// lifting_br1.t90:48-292, flux.f90:149-241.
#include "fxg_dual.h"
#include "fxg_line.h"

// FXG_ADJ_DUAL=1 takes the Riemann-flux derivatives from dual-number evaluations instead of the
// hand-written reverse (a cross-check of the reverse; slower).
#ifndef FXG_ADJ_DUAL
#define FXG_ADJ_DUAL 0
#endif

namespace fxg {
namespace {

// Adjoint of the primitive variables (rho,u,v,w,p,T,H) of one node mapped to the conservative
// state: ConsToPrim (idealgas/eos.f90:203-230) and H = (E+p)/rho, differentiated.
__device__ __forceinline__ void prim_adjoint(const Prim& q, double E, const Gas& g, double lrho, double lu, double lv,
                                             double lw, double lp, double lT, double lH, double* lU) {
  const double sr = 1.0 / q.rho;
  const double H = (E + q.p) * sr;
  double lE = lH * sr;
  lp += lH * sr;
  lrho -= H * lH * sr;
  lp += lT * sr * g.sR;
  lrho -= q.T * lT * sr;
  lE += g.kappaM1 * lp;
  lrho += g.kappaM1 * 0.5 * (q.u * q.u + q.v * q.v + q.w * q.w) * lp;
  lU[1] = lu * sr - g.kappaM1 * q.u * lp;
  lU[2] = lv * sr - g.kappaM1 * q.v * lp;
  lU[3] = lw * sr - g.kappaM1 * q.w * lp;
  lrho -= (q.u * lu + q.v * lv + q.w * lw) * sr;
  lU[0] = lrho;
  lU[4] = lE;
}

// Rotated state of conservative variables in dual arithmetic (cons_to_prim + rotate).
__device__ __forceinline__ RotState<Dual> rot_state(const Dual* c, double kappaM1, const Dual* nv, const Dual* t1,
                                                     const Dual* t2) {
  const Dual sr = Dual(1.0) / c[0];
  const Dual u = c[1] * sr, v = c[2] * sr, w = c[3] * sr;
  const Dual p = Dual(kappaM1) * (c[4] - Dual(0.5) * (c[1] * u + c[2] * v + c[3] * w));
  return rotate<Dual>(c[0], c[4], p, u, v, w, nv, t1, t2);
}

// Reverse of riemann_rot (split form) at one side point: lF is the adjoint of F in the side
// frame; the adjoints of the two rotated states' (rho, E, p, vn, vt1, vt2) are returned in aL, aR.
// Line by line the transpose of the forward arithmetic in fxg_physics.h (riemann.f90:558-855,
// splitflux.f90:672-700); srho = 1/rho is folded into rho. Divisions are taken as products with
// reciprocals formed once (1/rho, 1/c, 1/sqrt(rho)): the adjoint's rounding needs no match.
struct RotAdj {
  double rho, E, p, vn, vt1, vt2;
};

template <int SOLVER>
__device__ __forceinline__ void riemann_rot_vjp(const Gas& g, const RotState<double>& L, const RotState<double>& R,
                                                const double* lF, RotAdj& aL, RotAdj& aR) {
  aL = RotAdj{0, 0, 0, 0, 0, 0};
  aR = RotAdj{0, 0, 0, 0, 0, 0};
  // central part, Pirozzoli surface flux: F += Fc
  {
    const double HL = (L.E + L.p) * L.srho, HR = (R.E + R.p) * R.srho;
    const double rs = L.rho + R.rho, us = L.vn + R.vn, sv1 = L.vt1 + R.vt1, sv2 = L.vt2 + R.vt2, Hs = HL + HR;
    const double lrs = 0.25 * us * lF[0] + 0.125 * us * us * lF[1] + 0.125 * us * sv1 * lF[2] +
                       0.125 * us * sv2 * lF[3] + 0.125 * Hs * us * lF[4];
    const double lus = 0.25 * rs * lF[0] + 0.25 * rs * us * lF[1] + 0.125 * rs * sv1 * lF[2] +
                       0.125 * rs * sv2 * lF[3] + 0.125 * rs * Hs * lF[4];
    const double lsv1 = 0.125 * rs * us * lF[2], lsv2 = 0.125 * rs * us * lF[3], lHs = 0.125 * rs * us * lF[4];
    aL.p += 0.5 * lF[1]; aR.p += 0.5 * lF[1];
    aL.rho += lrs - HL * lHs * L.srho; aR.rho += lrs - HR * lHs * R.srho;
    aL.vn += lus; aR.vn += lus;
    aL.vt1 += lsv1; aR.vt1 += lsv1;
    aL.vt2 += lsv2; aR.vt2 += lsv2;
    aL.E += lHs * L.srho; aR.E += lHs * R.srho;
    aL.p += lHs * L.srho; aR.p += lHs * R.srho;
  }
  const double UL[5] = {L.rho, L.rho * L.vn, L.rho * L.vt1, L.rho * L.vt2, L.E};
  const double UR[5] = {R.rho, R.rho * R.vn, R.rho * R.vt1, R.rho * R.vt2, R.E};
  double ld[5] = {0, 0, 0, 0, 0};  // adjoint of UR - UL
  // d(sqrt(kappa p / rho)): c = sqrt(kappa p srho)
  auto sound_adj = [&](const RotState<double>& S, double c, double lc, RotAdj& a) {
    const double f = 0.5 * g.kappa / c;
    a.p += f * S.srho * lc;
    a.rho -= f * S.p * S.srho * S.srho * lc;
  };
  if (SOLVER == 1) {  // Lax-Friedrichs: F -= 0.5*lmax*(UR - UL)
    const double cL = sqrt(g.kappa * L.p * L.srho), cR = sqrt(g.kappa * R.p * R.srho);
    const double vmax = fmax(fabs(R.vn), fabs(L.vn)), cmax = fmax(cL, cR);
    const double lmax = vmax + cmax;
    double llmax = 0.0;
    for (int k = 0; k < 5; ++k) {
      ld[k] = -0.5 * lmax * lF[k];
      llmax -= 0.5 * (UR[k] - UL[k]) * lF[k];
    }
    if (fabs(R.vn) >= fabs(L.vn)) aR.vn += (R.vn < 0.0 ? -llmax : llmax);
    else aL.vn += (L.vn < 0.0 ? -llmax : llmax);
    if (cL >= cR) sound_adj(L, cL, llmax, aL);
    else sound_adj(R, cR, llmax, aR);
  } else {
    // Roe averages
    const double HLr = (L.E + L.p) * L.srho, HRr = (R.E + R.p) * R.srho;
    const double sqL = sqrt(L.rho), sqR = sqrt(R.rho);
    const double ss = 1.0 / (sqL + sqR), isqL = 1.0 / sqL, isqR = 1.0 / sqR;
    const double ru = (sqR * R.vn + sqL * L.vn) * ss;
    const double rv = (sqR * R.vt1 + sqL * L.vt1) * ss;
    const double rw = (sqR * R.vt2 + sqL * L.vt2) * ss;
    const double absVel = ru * ru + rv * rv + rw * rw;
    const double H = (sqR * HRr + sqL * HLr) * ss;
    const double c = sqrt(g.kappaM1 * (H - 0.5 * absVel));
    const double ic = 1.0 / c;
    double al[5], a[5];
    double d[5];
    for (int k = 0; k < 5; ++k) d[k] = UR[k] - UL[k];
    // entropy-fix quantities
    double cL = 0, cR = 0, rd = 0, tmp = 0, du = 0, dp = 0;
    if (SOLVER == 3) {
      const double d5 = d[4] - (d[2] - rv * d[0]) * rv - (d[3] - rw * d[0]) * rw;
      al[2] = d[2] - rv * d[0];
      al[3] = d[3] - rw * d[0];
      al[1] = g.kappaM1 * ic * ic * (d[0] * (H - ru * ru) - d5 + ru * d[1]);
      al[0] = 0.5 * ic * (d[0] * (ru + c) - d[1] - c * al[1]);
      al[4] = d[0] - al[0] - al[1];
      a[0] = fabs(ru - c); a[1] = a[2] = a[3] = fabs(ru); a[4] = fabs(ru + c);
    } else {
      cL = sqrt(g.kappa * L.p * L.srho); cR = sqrt(g.kappa * R.p * R.srho);
      rd = sqrt(L.rho * R.rho);
      const double d1 = R.rho - L.rho, dv = R.vt1 - L.vt1, dw = R.vt2 - L.vt2;
      du = R.vn - L.vn; dp = R.p - L.p;
      tmp = 0.5 * ic * ic;
      al[0] = tmp * (dp - rd * c * du);
      al[1] = d1 - dp * 2.0 * tmp;
      al[2] = rd * dv;
      al[3] = rd * dw;
      al[4] = tmp * (dp + rd * c * du);
      const double ar[5] = {ru - c, ru, ru, ru, ru + c};
      const double aLk[5] = {L.vn - cL, L.vn, L.vn, L.vn, L.vn + cL};
      const double aRk[5] = {R.vn - cR, R.vn, R.vn, R.vn, R.vn + cR};
      for (int k = 0; k < 5; ++k) {
        const double da = fmax(fmax(0.0, ar[k] - aLk[k]), aRk[k] - ar[k]);
        a[k] = (fabs(ar[k]) < da) ? 0.5 * (ar[k] * ar[k] / da + da) : fabs(ar[k]);
      }
    }
    const double w[5] = {al[0] * a[0], al[1] * a[1], al[2] * a[2], al[3] * a[3], al[4] * a[4]};
    // F -= 0.5*D with D the dissipation sum_k w_k r_k
    double lD[5];
    for (int k = 0; k < 5; ++k) lD[k] = -0.5 * lF[k];
    double lw[5];
    lw[0] = lD[0] + (ru - c) * lD[1] + rv * lD[2] + rw * lD[3] + (H - ru * c) * lD[4];
    lw[1] = lD[0] + ru * lD[1] + rv * lD[2] + rw * lD[3] + 0.5 * absVel * lD[4];
    lw[2] = lD[2] + rv * lD[4];
    lw[3] = lD[3] + rw * lD[4];
    lw[4] = lD[0] + (ru + c) * lD[1] + rv * lD[2] + rw * lD[3] + (H + ru * c) * lD[4];
    const double wsum = w[0] + w[1] + w[4];
    double lru = lD[1] * wsum + lD[4] * (w[4] - w[0]) * c;
    double lc = lD[1] * (w[4] - w[0]) + lD[4] * (w[4] - w[0]) * ru;
    double lrv = lD[2] * wsum + lD[4] * w[2];
    double lrw = lD[3] * wsum + lD[4] * w[3];
    double lH = lD[4] * (w[0] + w[4]);
    double labs = 0.5 * w[1] * lD[4];
    double lal[5], la[5];
    for (int k = 0; k < 5; ++k) {
      lal[k] = a[k] * lw[k];
      la[k] = al[k] * lw[k];
    }
    if (SOLVER == 3) {
      // al4 = d0 - al0 - al1
      ld[0] += lal[4]; lal[0] -= lal[4]; lal[1] -= lal[4];
      // al0 = 0.5/c*Y, Y = d0(ru+c) - d1 - c al1
      const double lY = 0.5 * lal[0] * ic;
      lc -= al[0] * ic * lal[0];
      ld[0] += (ru + c) * lY; lru += d[0] * lY; lc += (d[0] - al[1]) * lY; ld[1] -= lY; lal[1] -= c * lY;
      // al1 = kappaM1/c^2*X, X = d0(H - ru^2) - d5 + ru d1
      const double lX = g.kappaM1 * lal[1] * ic * ic;
      lc -= 2.0 * al[1] * ic * lal[1];
      double ld5 = -lX;
      ld[0] += (H - ru * ru) * lX; lH += d[0] * lX; lru += (d[1] - 2.0 * ru * d[0]) * lX; ld[1] += ru * lX;
      // al2 = d2 - rv d0, al3 = d3 - rw d0
      ld[2] += lal[2]; lrv -= d[0] * lal[2]; ld[0] -= rv * lal[2];
      ld[3] += lal[3]; lrw -= d[0] * lal[3]; ld[0] -= rw * lal[3];
      // d5 = d4 - e2 rv - e3 rw, e2 = d2 - rv d0, e3 = d3 - rw d0
      const double e2 = d[2] - rv * d[0], e3 = d[3] - rw * d[0];
      ld[4] += ld5;
      const double le2 = -rv * ld5, le3 = -rw * ld5;
      lrv -= e2 * ld5; lrw -= e3 * ld5;
      ld[2] += le2; lrv -= d[0] * le2; ld[0] -= rv * le2;
      ld[3] += le3; lrw -= d[0] * le3; ld[0] -= rw * le3;
      // a = |ru -/+ c|, |ru|
      const double s0 = (ru - c) < 0.0 ? -1.0 : 1.0, s1 = ru < 0.0 ? -1.0 : 1.0, s4 = (ru + c) < 0.0 ? -1.0 : 1.0;
      lru += s0 * la[0] + s1 * (la[1] + la[2] + la[3]) + s4 * la[4];
      lc += -s0 * la[0] + s4 * la[4];
    } else {
      // entropy-fixed |a_k|
      const double ar[5] = {ru - c, ru, ru, ru, ru + c};
      const double aLk[5] = {L.vn - cL, L.vn, L.vn, L.vn, L.vn + cL};
      const double aRk[5] = {R.vn - cR, R.vn, R.vn, R.vn, R.vn + cR};
      double lar[5] = {0, 0, 0, 0, 0}, laL[5] = {0, 0, 0, 0, 0}, laR[5] = {0, 0, 0, 0, 0};
      for (int k = 0; k < 5; ++k) {
        const double x = ar[k] - aLk[k], y = aRk[k] - ar[k];
        const double m1 = fmax(0.0, x);
        const double da = fmax(m1, y);
        double lda = 0.0;
        if (fabs(ar[k]) < da) {
          lar[k] += ar[k] / da * la[k];
          lda = 0.5 * (1.0 - ar[k] * ar[k] / (da * da)) * la[k];
        } else {
          lar[k] += (ar[k] < 0.0 ? -la[k] : la[k]);
        }
        if (m1 >= y) {
          if (x > 0.0) { lar[k] += lda; laL[k] -= lda; }
        } else {
          laR[k] += lda; lar[k] -= lda;
        }
      }
      lru += lar[0] + lar[1] + lar[2] + lar[3] + lar[4];
      lc += -lar[0] + lar[4];
      aL.vn += laL[0] + laL[1] + laL[2] + laL[3] + laL[4];
      aR.vn += laR[0] + laR[1] + laR[2] + laR[3] + laR[4];
      double lcL = -laL[0] + laL[4], lcR = -laR[0] + laR[4];
      // wave strengths from primitive jumps
      const double dv = R.vt1 - L.vt1, dw = R.vt2 - L.vt2;
      double ltmp = (dp - rd * c * du) * lal[0] + (dp + rd * c * du) * lal[4] - 2.0 * dp * lal[1];
      const double ldp = tmp * (lal[0] + lal[4]) - 2.0 * tmp * lal[1];
      const double lrd = -tmp * c * du * lal[0] + tmp * c * du * lal[4] + dv * lal[2] + dw * lal[3];
      lc += -tmp * rd * du * lal[0] + tmp * rd * du * lal[4];
      const double ldu = -tmp * rd * c * lal[0] + tmp * rd * c * lal[4];
      const double ld1 = lal[1];
      const double ldv = rd * lal[2], ldw = rd * lal[3];
      lc -= ltmp * ic * ic * ic;  // tmp = 0.5/c^2
      const double hrd = 0.5 / rd;
      aL.rho += R.rho * hrd * lrd; aR.rho += L.rho * hrd * lrd;
      aR.rho += ld1; aL.rho -= ld1;
      aR.vn += ldu; aL.vn -= ldu;
      aR.vt1 += ldv; aL.vt1 -= ldv;
      aR.vt2 += ldw; aL.vt2 -= ldw;
      aR.p += ldp; aL.p -= ldp;
      sound_adj(L, cL, lcL, aL);
      sound_adj(R, cR, lcR, aR);
    }
    // c = sqrt(kappaM1 (H - absVel/2))
    lH += 0.5 * g.kappaM1 * ic * lc;
    labs -= 0.25 * g.kappaM1 * ic * lc;
    lru += 2.0 * ru * labs; lrv += 2.0 * rv * labs; lrw += 2.0 * rw * labs;
    // H, ru, rv, rw: Roe averages with weights sqL*ss, sqR*ss
    double lsqL = HLr * ss * lH + L.vn * ss * lru + L.vt1 * ss * lrv + L.vt2 * ss * lrw;
    double lsqR = HRr * ss * lH + R.vn * ss * lru + R.vt1 * ss * lrv + R.vt2 * ss * lrw;
    const double lss = (sqR * HRr + sqL * HLr) * lH + (sqR * R.vn + sqL * L.vn) * lru +
                       (sqR * R.vt1 + sqL * L.vt1) * lrv + (sqR * R.vt2 + sqL * L.vt2) * lrw;
    lsqL -= ss * ss * lss; lsqR -= ss * ss * lss;
    aL.vn += sqL * ss * lru; aR.vn += sqR * ss * lru;
    aL.vt1 += sqL * ss * lrv; aR.vt1 += sqR * ss * lrv;
    aL.vt2 += sqL * ss * lrw; aR.vt2 += sqR * ss * lrw;
    const double lHL = sqL * ss * lH, lHR = sqR * ss * lH;
    aL.E += L.srho * lHL; aL.p += L.srho * lHL; aL.rho -= (L.E + L.p) * L.srho * L.srho * lHL;
    aR.E += R.srho * lHR; aR.p += R.srho * lHR; aR.rho -= (R.E + R.p) * R.srho * R.srho * lHR;
    aL.rho += 0.5 * lsqL * isqL; aR.rho += 0.5 * lsqR * isqR;
  }
  // U = (rho, rho vn, rho vt1, rho vt2, E) of both sides through d = UR - UL
  aR.rho += ld[0] + R.vn * ld[1] + R.vt1 * ld[2] + R.vt2 * ld[3];
  aR.vn += R.rho * ld[1]; aR.vt1 += R.rho * ld[2]; aR.vt2 += R.rho * ld[3]; aR.E += ld[4];
  aL.rho -= ld[0] + L.vn * ld[1] + L.vt1 * ld[2] + L.vt2 * ld[3];
  aL.vn -= L.rho * ld[1]; aL.vt1 -= L.rho * ld[2]; aL.vt2 -= L.rho * ld[3]; aL.E -= ld[4];
}

// Adjoint of a rotated state (rho, E, p, vn, vt1, vt2) to the conservative state it was built
// from (cons_to_prim + rotation by n, t1, t2).
__device__ __forceinline__ void rot_state_adjoint(const double* c, const Gas& g, const double* nv, const double* t1,
                                                  const double* t2, const RotAdj& a, double* lU) {
  const double sr = 1.0 / c[0];
  const double u = c[1] * sr, v = c[2] * sr, w = c[3] * sr;
  const double lu = a.vn * nv[0] + a.vt1 * t1[0] + a.vt2 * t2[0];
  const double lv = a.vn * nv[1] + a.vt1 * t1[1] + a.vt2 * t2[1];
  const double lw = a.vn * nv[2] + a.vt1 * t1[2] + a.vt2 * t2[2];
  // p = kappaM1 (E - (m.u)/2)
  lU[4] = a.E + g.kappaM1 * a.p;
  lU[1] = lu * sr - g.kappaM1 * u * a.p;
  lU[2] = lv * sr - g.kappaM1 * v * a.p;
  lU[3] = lw * sr - g.kappaM1 * w * a.p;
  lU[0] = a.rho + g.kappaM1 * 0.5 * (u * u + v * v + w * w) * a.p - (u * lu + v * lv + w * lw) * sr;
}

// ---------------------------------------------------------------------------------------------
// Both element kernels give each lane a line of nodes, as the forward stage kernel does (fxg_stage.hip): a
// pair's Jacobian serves both of its nodes, so evaluating it once per pair halves it, and the LDS reads
// per node fall from about 330 to 90 (k_adj_euler) and from 290 to 110 (k_adj_visc), which bound the forms with
// one lane per node. TGV 16^3, N=5, Roe, parallelepipeds: 134 -> 110 us and 90 -> 58 us per reverse stage (491 and 321
// bytes per node at 4.0 and 4.9 TB/s). Two waves per SIMD: at three the Riemann reverse spills (143 and 88 us); with
// Roe-entropy-fix 3 to 11 VGPRs spill at two as well. At N = 7 with general metric terms k_adj_euler's 93 KB of
// LDS leave one workgroup per CU, one wave per SIMD: vjp at 12^3, Roe 0.241 -> 0.206 ms all the same
// (parallelepipeds 0.248 -> 0.161).

// The lane's line: direction, end nodes (offset in the element), local sides and side slots of its ends.
template <int N>
struct AdjLine {
  int d, ln, a, b, first, last, ls[2], fp[2];  // fp: own face points
  unsigned own[2];
  __device__ __forceinline__ AdjLine(const DevMesh& m, int e, int t) {
    constexpr int n = N + 1, nf = n * n;
    d = t / nf; ln = t - d * nf; a = ln % n; b = ln / n;
    first = d == 0 ? n * ln : (d == 1 ? a + nf * b : ln);
    last = first + N * (d == 0 ? 1 : (d == 1 ? n : nf));
    ls[0] = d == 0 ? 5 : (d == 1 ? 2 : 1);
    ls[1] = d == 0 ? 3 : (d == 1 ? 4 : 6);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      fp[s] = (ls[s] - 1) * nf + ln;
      own[s] = m.slotTab[(size_t)6 * nf * e + fp[s]];
    }
  }
};

// Sum over a node's face points (up to three) of the NV values kept per own face point, rows of NF,
// place (2 d + s) nf + ln.
template <int N, int NV>
__device__ __forceinline__ void add_faces(const double* sF, int nd, double* x) {
  constexpr int n = N + 1, nf = n * n, NF = 6 * nf;
  const int at[3] = {nd % n, (nd / n) % n, nd / nf};
  const int ln[3] = {nd / n, at[0] + n * at[2], nd % nf};
#pragma unroll
  for (int d = 0; d < 3; ++d)
    if (at[d] == 0 || at[d] == N) {
      const double* f = sF + (2 * d + (at[d] == N ? 1 : 0)) * nf + ln[d];
#pragma unroll
      for (int v = 0; v < NV; ++v) x[v] += f[v * NF];
    }
}

// LDS rows of k_adj_euler: 0 rho/4, 1 H, 2 u, 3 v, 4 w, 5..9 -sJ*lam; general metrics: 10..18 Ja^1..3 / 2. Then
// five values per own face point.
template <int N, bool AFF>
struct LdsAE {
  static constexpr int ROWS = AFF ? 10 : 19, FACE = ROWS * S<N>::RS, NF = 6 * S<N>::nf, SIZE = FACE + 5 * NF;
};

template <int N, int SOLVER, bool AFF>
__global__ __launch_bounds__(S<N>::NT) __attribute__((amdgpu_waves_per_eu(2))) void k_adj_euler(
    const double* __restrict__ U, DevMesh m, const double* __restrict__ basis, const double* __restrict__ FUa,
    double* __restrict__ lam, double* __restrict__ ub, double cub, Gas gas, double* __restrict__ out,
    double* __restrict__ XU, double* __restrict__ Xg, Pending pd) {
  constexpr int n = S<N>::n, nf = S<N>::nf, np = S<N>::np, NL = S<N>::NL, NT = S<N>::NT, RN = S<N>::RN, RS = S<N>::RS;
  using L = LdsAE<N, AFF>;
  __shared__ double sL[L::SIZE];
  double* sF = sL + L::FACE;
  const BasisLayout B{n};
  const int e = blockIdx.x, t = N == 7 ? (threadIdx.x + 64 * (e & 3)) % NT : threadIdx.x;
  const bool line = t < NL;
  const AdjLine<N> q(m, e, line ? t : 0);
  const size_t e0 = (size_t)np * e;
  const double* je = AFF ? m.aff + 10 * (size_t)e : nullptr;
  // Staging: the loads of a lane's nodes are issued together, before the first wait; all stores come after.
  double c5[RN][5], l0[RN][5], u0[RN][5], o5[RN][5], sj[RN];
#pragma unroll
  for (int r = 0; r < RN; ++r) {
    const bool in = t + r * NT < np;
    const size_t gid = e0 + (in ? t + r * NT : 0);
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      c5[r][v] = U[5 * gid + v];
      l0[r][v] = lam[5 * gid + v];
      u0[r][v] = ub ? ub[5 * gid + v] : 0.0;
      o5[r][v] = pd.XU ? out[5 * gid + v] : 0.0;
    }
    sj[r] = AFF ? je[9] : m.sJ[gid];
  }
  if (pd.XU) {  // the neighbours' face parts of the previous reverse stage, to the nodes through the face rows
    if (line) {
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int v = 0; v < 5; ++v)
          sF[v * L::NF + (2 * q.d + s) * nf + q.ln] = pd.XU[5 * (size_t)slot_nbr<N>(q.own[s]) + v];
    }
    __syncthreads();
  }
#pragma unroll
  for (int r = 0; r < RN; ++r) {
    const int nd = t + r * NT;
    if (nd >= np) continue;
    const size_t gid = e0 + nd;
    const Prim p = cons_to_prim(c5[r], gas);
    double* s = sL + pos<N>(nd % n, (nd / n) % n, nd / nf);
    s[0] = 0.25 * p.rho; s[RS] = (c5[r][4] + p.p) * p.srho; s[2 * RS] = p.u; s[3 * RS] = p.v; s[4 * RS] = p.w;
    double l5[5];
    if (pd.XU) {
      // the register update of the previous reverse stage: ub += its out + the neighbours' face
      // parts, rbar = a*lam of that stage
      add_faces<N, 5>(sF, nd, o5[r]);
#pragma unroll
      for (int v = 0; v < 5; ++v) {
        const double u1 = u0[r][v] + o5[r][v];
        ub[5 * gid + v] = u1;
        l5[v] = pd.a * l0[r][v] + cub * u1;
      }
    } else {
#pragma unroll
      for (int v = 0; v < 5; ++v) l5[v] = l0[r][v] + cub * u0[r][v];
    }
    if (ub) {  // lam of this stage, for k_adj_visc and for the update that is still to come
#pragma unroll
      for (int v = 0; v < 5; ++v) lam[5 * gid + v] = l5[v];
    }
#pragma unroll
    for (int v = 0; v < 5; ++v) s[(5 + v) * RS] = -sj[r] * l5[v];
    if constexpr (!AFF) {
#pragma unroll
      for (int x = 0; x < 3; ++x) {
        s[(10 + x) * RS] = 0.5 * m.Mf[3 * gid + x];
        s[(13 + x) * RS] = 0.5 * m.Mg[3 * gid + x];
        s[(16 + x) * RS] = 0.5 * m.Mh[3 * gid + x];
      }
    }
  }
  Line<N> lp(q.d, q.a, q.b);
  __syncthreads();

  // own face points, the two ends of the line: the neighbour's share of the viscous face term, and the Riemann adjoint
  if (line) {
#pragma unroll 1
    for (int s = 0; s < 2; ++s) {
      const unsigned own = s ? q.own[1] : q.own[0];  // (selected: an index into registers goes through scratch)
      const bool master = slot_is_master<N>(own);
      const unsigned nb = slot_nbr<N>(own);
      const int id = s ? q.last : q.first;
      const double lh = s ? basis[B.L_HatPlus() + N] : basis[B.L_HatMinus()];
      const double* me = lp.at(sL, s ? N : 0);
#pragma unroll
      for (int c = 0; c < 4; ++c) Xg[4 * (size_t)own + c] = -0.5 * lh * me[(6 + c) * RS];
      double nv[3], t1[3], t2[3];
      const double* Jd = AFF ? je + 3 * q.d : (q.d == 0 ? m.Mf : (q.d == 1 ? m.Mg : m.Mh)) + 3 * (e0 + id);
      const double se = face_frame<N, double>(m, Jd, s ? q.ls[1] : q.ls[0], own, master, nv, t1, t2);
      const double ms = master ? 1.0 : -1.0;
      double lF[5];
#pragma unroll
      for (int v = 0; v < 5; ++v) lF[v] = ms * se * lh * me[(5 + v) * RS];
      const double* Uo = U + 5 * (e0 + id);
      const double* Un = FUa ? FUa + 5 * (size_t)nb : U + 5 * (size_t)m.nbNode[(size_t)L::NF * e + (s ? q.fp[1] : q.fp[0])];
      double* dst = sF + (2 * q.d + s) * nf + q.ln;
#if FXG_ADJ_DUAL
      // directional derivatives in dual arithmetic (10 evaluations): the reference for the reverse
      const Dual nd[3] = {nv[0], nv[1], nv[2]}, t1d[3] = {t1[0], t1[1], t1[2]}, t2d[3] = {t2[0], t2[1], t2[2]};
      const GasT<Dual> gd(gas);
#pragma unroll 1
      for (int k = 0; k < 10; ++k) {
        Dual a[5], b[5];
#pragma unroll
        for (int v = 0; v < 5; ++v) {
          a[v] = Dual(Uo[v], k == v ? 1.0 : 0.0);
          b[v] = Dual(Un[v], k == 5 + v ? 1.0 : 0.0);
        }
        const RotState<Dual> So = rot_state(a, gas.kappaM1, nd, t1d, t2d);
        const RotState<Dual> Sn = rot_state(b, gas.kappaM1, nd, t1d, t2d);
        Dual F[5];
        if (master) riemann_rot<Dual>(gd, SOLVER, true, So, Sn, F);
        else riemann_rot<Dual>(gd, SOLVER, true, Sn, So, F);
        double x = lF[0] * F[0].d + lF[4] * F[4].d;
#pragma unroll
        for (int c = 0; c < 3; ++c) x += lF[1 + c] * (nv[c] * F[1].d + t1[c] * F[2].d + t2[c] * F[3].d);
        if (k < 5) dst[k * L::NF] = x;
        else XU[5 * (size_t)own + (k - 5)] = x;
      }
#else
      // flux adjoint in the side frame, then the reverse of the Riemann solver and of the rotation
      double lFr[5];
      lFr[0] = lF[0];
      lFr[1] = nv[0] * lF[1] + nv[1] * lF[2] + nv[2] * lF[3];
      lFr[2] = t1[0] * lF[1] + t1[1] * lF[2] + t1[2] * lF[3];
      lFr[3] = t2[0] * lF[1] + t2[1] * lF[2] + t2[2] * lF[3];
      lFr[4] = lF[4];
      const Prim po = cons_to_prim(Uo, gas), pn = cons_to_prim(Un, gas);
      const RotState<double> So = rotate<double>(po.rho, Uo[4], po.p, po.u, po.v, po.w, nv, t1, t2);
      const RotState<double> Sn = rotate<double>(pn.rho, Un[4], pn.p, pn.u, pn.v, pn.w, nv, t1, t2);
      // the master's state on the left, operands selected rather than branched on (one copy of the
      // reverse; a wave may hold master and slave points)
      const RotState<double> SL = master ? So : Sn, SR = master ? Sn : So;
      RotAdj aL, aR;
      riemann_rot_vjp<SOLVER>(gas, SL, SR, lFr, aL, aR);
      const RotAdj ao = master ? aL : aR, an = master ? aR : aL;
      double gOwn[5], gNb[5];
      rot_state_adjoint(Uo, gas, nv, t1, t2, ao, gOwn);
      rot_state_adjoint(Un, gas, nv, t1, t2, an, gNb);
#pragma unroll
      for (int v = 0; v < 5; ++v) {
        dst[v * L::NF] = gOwn[v];
        XU[5 * (size_t)own + v] = gNb[v];
      }
#endif
    }
  }

  // split-flux adjoint: each pair (i,l) contributes J_s^T (D(i,l) mu_i + D(l,i) mu_l) to both
  // nodes' primitive adjoints, J_s the flux Jacobian w.r.t. the pair sums (rho,u,v,w,p,H)
  double acc[6][n];  // rho, u, v, w, p, H
  if (line) {
#pragma unroll
    for (int v = 0; v < 6; ++v)
#pragma unroll
      for (int i = 0; i < n; ++i) acc[v][i] = 0.0;
    const double* W = basis + B.PairD() + fresh();
    lp.again();
    double* sJ9 = sL + (10 + 3 * q.d) * RS;
    struct Nd {
      double r, H, u, v, w, mu[5], j[3];
    };
    double mj[3] = {0, 0, 0};
    if constexpr (AFF) {
#pragma unroll
      for (int x = 0; x < 3; ++x) mj[x] = q.d == 0 ? je[x] : (q.d == 1 ? je[3 + x] : je[6 + x]);
    }
    auto load = [&](int l) {
      const double* s = lp.at(sL, l);
      Nd x;
      x.r = s[0]; x.H = s[RS]; x.u = s[2 * RS]; x.v = s[3 * RS]; x.w = s[4 * RS];
#pragma unroll
      for (int c = 0; c < 5; ++c) x.mu[c] = s[(5 + c) * RS];
      if constexpr (!AFF) {
        const double* J = lp.at(sJ9, l);
        x.j[0] = J[0]; x.j[1] = J[RS]; x.j[2] = J[2 * RS];
      }
      return x;
    };
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const Nd A = load(i);
#pragma unroll
      for (int l = i + 1; l < n; ++l) {
        const Nd C = load(l);
        const int pr = i * (2 * n - i - 1) / 2 + l - i - 1;
        const double wi = W[2 * pr], wl = W[2 * pr + 1];
        double a0, a1, a2;
        if constexpr (AFF) {
          a0 = mj[0]; a1 = mj[1]; a2 = mj[2];
        } else {
          a0 = A.j[0] + C.j[0]; a1 = A.j[1] + C.j[1]; a2 = A.j[2] + C.j[2];
        }
        const double us = A.u + C.u, vs = A.v + C.v, ws = A.w + C.w, Hs = A.H + C.H, rq = A.r + C.r;  // rq: rho sum / 4
        const double mv = a0 * us + a1 * vs + a2 * ws, qq = rq * mv;
        double vec[5];
#pragma unroll
        for (int c = 0; c < 5; ++c) vec[c] = wi * A.mu[c] + wl * C.mu[c];
        const double beta = 2.0 * vec[0] + (vec[1] * us + vec[2] * vs + vec[3] * ws) + Hs * vec[4];  // times 4
        const double rb = rq * beta;
        const double x[6] = {0.25 * mv * beta,        a0 * rb + qq * vec[1], a1 * rb + qq * vec[2],
                             a2 * rb + qq * vec[3],   a0 * vec[1] + a1 * vec[2] + a2 * vec[3], qq * vec[4]};
#pragma unroll
        for (int v = 0; v < 6; ++v) {
          acc[v][i] += x[v];
          acc[v][l] += x[v];
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  __syncthreads();  // the pair loop's rows are free
  // the three directions' sums at the nodes, VR variables at a time
  constexpr int VR = L::ROWS >= 18 ? 6 : 3;
  double sum[RN][6];
#pragma unroll
  for (int v0 = 0; v0 < 6; v0 += VR) {
    if (line) {
      lp.again();
      double* sS = sL + VR * q.d * RS;
#pragma unroll
      for (int v = 0; v < VR; ++v)
#pragma unroll
        for (int i = 0; i < n; ++i) lp.at(sS, i)[v * RS] = acc[v0 + v][i];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RN; ++r) {
      const int nd = t + r * NT < np ? t + r * NT : 0;
      const double* s = sL + pos<N>(nd % n, (nd / n) % n, nd / nf);
#pragma unroll
      for (int v = 0; v < VR; ++v) sum[r][v0 + v] = s[v * RS] + s[(VR + v) * RS] + s[(2 * VR + v) * RS];
    }
    if (v0 + VR < 6) __syncthreads();
  }
#pragma unroll
  for (int r = 0; r < RN; ++r) {
    const int nd = t + r * NT;
    if (nd >= np) continue;
    const size_t gid = e0 + nd;
    double cc[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) cc[v] = U[5 * gid + v];
    const Prim p = cons_to_prim(cc, gas);
    double lU[5];
    prim_adjoint(p, cc[4], gas, sum[r][0], sum[r][1], sum[r][2], sum[r][3], sum[r][4], 0.0, sum[r][5], lU);
    add_faces<N, 5>(sF, nd, lU);
#pragma unroll
    for (int v = 0; v < 5; ++v) out[5 * gid + v] = lU[v];
  }
}

// ---------------------------------------------------------------------------------------------
// XU: the Riemann part of the neighbour's face adjoint (k_adj_euler); the lifting part w.r.t. the
// neighbour's (u,v,w,T), taken to its conservative variables with its face state, is added here.
// LDS rows: 0 u, 1 v, 2 w, 3 T, 4..7 -sJ*lam of momentum and energy, 8..13 exchange between line and node phases
// (two variables in three directions).
template <int N, bool AFF>
__global__ __launch_bounds__(S<N>::NT) __attribute__((amdgpu_waves_per_eu(N <= 4 ? 3 : 2))) void k_adj_visc(
    const double* __restrict__ U, DevMesh m, const double* __restrict__ basis, const double* __restrict__ FUa,
    const double* __restrict__ lam, const double* __restrict__ Xg, Gas gas, double* __restrict__ out,
    double* __restrict__ XU) {
  constexpr int n = S<N>::n, nf = S<N>::nf, np = S<N>::np, NL = S<N>::NL, NT = S<N>::NT, RN = S<N>::RN, RS = S<N>::RS;
  constexpr int X = 8;
  __shared__ double sL[14 * RS];
  const BasisLayout B{n};
  const int e = blockIdx.x, t = N == 7 ? (threadIdx.x + 64 * (e & 3)) % NT : threadIdx.x;
  const bool line = t < NL;
  const AdjLine<N> q(m, e, line ? t : 0);
  const size_t e0 = (size_t)np * e;
  const double* je = AFF ? m.aff + 10 * (size_t)e : nullptr;
  double c5[RN][5], l4[RN][4], sj[RN];
#pragma unroll
  for (int r = 0; r < RN; ++r) {
    const size_t gid = e0 + (t + r * NT < np ? t + r * NT : 0);
#pragma unroll
    for (int v = 0; v < 5; ++v) c5[r][v] = U[5 * gid + v];
#pragma unroll
    for (int c = 0; c < 4; ++c) l4[r][c] = lam[5 * gid + 1 + c];
    sj[r] = AFF ? je[9] : m.sJ[gid];
  }
  double fn[2][5], xg[2][4];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const size_t nb = slot_nbr<N>(q.own[s]);
#pragma unroll
    for (int v = 0; v < 5; ++v) fn[s][v] = FUa ? FUa[5 * nb + v] : U[5 * (size_t)m.nbNode[(size_t)6 * nf * e + q.fp[s]] + v];
#pragma unroll
    for (int c = 0; c < 4; ++c) xg[s][c] = Xg[4 * nb + c];
  }
  int place[RN];
#pragma unroll
  for (int r = 0; r < RN; ++r) {
    const int nd = t + r * NT < np ? t + r * NT : 0;
    place[r] = pos<N>(nd % n, (nd / n) % n, nd / nf);
    if (t + r * NT < np) {
      const Prim p = cons_to_prim(c5[r], gas);
      double* s = sL + place[r];
      s[0] = p.u; s[RS] = p.v; s[2 * RS] = p.w; s[3 * RS] = p.T;
#pragma unroll
      for (int c = 0; c < 4; ++c) s[(4 + c) * RS] = -sj[r] * l4[r][c];
    }
  }
  Prim qn[2];  // the neighbours' face states
#pragma unroll
  for (int s = 0; s < 2; ++s) qn[s] = cons_to_prim(fn[s], gas);
  Line<N> lp(q.d, q.a, q.b);
  const double lhm = basis[B.L_HatMinus()], lhp = basis[B.L_HatPlus() + N];
  __syncthreads();
  double jq[2][4];  // BR1 jumps with their sign and weight
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const double* o = lp.at(sL, s ? N : 0);
    const double h = s ? 0.5 * lhp : -0.5 * lhm;
    jq[s][0] = h * (qn[s].u - o[0]); jq[s][1] = h * (qn[s].v - o[RS]); jq[s][2] = h * (qn[s].w - o[2 * RS]);
    jq[s][3] = h * (qn[s].T - o[3 * RS]);
  }
  // to the nodes: the reference derivatives of u,v,w,T (g) and, from the adjoint of the viscous flux, the
  // transposed weak derivative of mu along each direction with the face terms at the ends (lc)
  double g[RN][12], lc[RN][12];  // [d][variable]
#pragma unroll
  for (int h = 0; h < 4; ++h) {
    const int w0 = 2 * (h & 1);
    if (line) {
      const double* M = basis + (h < 2 ? B.D_T() : B.D_Hat_T()) + fresh();
      lp.again();
      double* sX = sL + (X + 2 * q.d) * RS;
      double x[2][n];
#pragma unroll
      for (int w = 0; w < 2; ++w)
#pragma unroll
        for (int l = 0; l < n; ++l) x[w][l] = lp.at(sL, l)[((h < 2 ? 0 : 4) + w0 + w) * RS];
      double y[2][n];
#pragma unroll
      for (int l = 0; l < n; ++l)
#pragma unroll
        for (int i = 0; i < n; ++i)
#pragma unroll
          for (int w = 0; w < 2; ++w) {
            // D_T(l,i) for the derivative at i; D_Hat_T(i,l) for its transpose
            const double z = (h < 2 ? M[l + n * i] : M[i + n * l]) * x[w][l];
            y[w][i] = l == 0 ? z : y[w][i] + z;
          }
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        if (h < 2) {
          y[w][0] += jq[0][w0 + w];
          y[w][N] += jq[1][w0 + w];
        } else {
          y[w][0] -= 0.5 * lhm * x[w][0] + xg[0][w0 + w];
          y[w][N] += 0.5 * lhp * x[w][N] + xg[1][w0 + w];
        }
#pragma unroll
        for (int i = 0; i < n; ++i) lp.at(sX, i)[w * RS] = y[w][i];
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RN; ++r)
#pragma unroll
      for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int w = 0; w < 2; ++w) (h < 2 ? g : lc)[r][4 * d + w0 + w] = sL[(X + 2 * d + w) * RS + place[r]];
    __syncthreads();
  }
  // node lanes: in place of g the adjoint per reference derivative kappa^d = Ja^d . nu, in lq that of u,v,w
  double lq[RN][4];
#pragma unroll
  for (int r = 0; r < RN; ++r) {
    double Ja[9], sjr = sj[r];
    if constexpr (AFF) {
#pragma unroll
      for (int x = 0; x < 9; ++x) Ja[x] = je[x];
    } else {
      double z;
      load_metrics<double>(m, e0 + (t + r * NT < np ? t + r * NT : 0), Ja, z);
    }
    double p[12], lf[3][4];
#pragma unroll
    for (int x = 0; x < 3; ++x)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        p[4 * x + v] = (Ja[x] * g[r][v] + Ja[3 + x] * g[r][4 + v] + Ja[6 + x] * g[r][8 + v]) * sjr;
        lf[x][v] = Ja[x] * lc[r][v] + Ja[3 + x] * lc[r][4 + v] + Ja[6 + x] * lc[r][8 + v];
      }
    // diff_flux adjoint (flux.f90:149-241): stresses, velocities, temperature gradient
    const double mu0 = gas.mu0;
    const double txx = mu0 * (gas.s43 * p[0] - gas.s23 * p[5] - gas.s23 * p[10]);
    const double tyy = mu0 * (-gas.s23 * p[0] + gas.s43 * p[5] - gas.s23 * p[10]);
    const double tzz = mu0 * (-gas.s23 * p[0] - gas.s23 * p[5] + gas.s43 * p[10]);
    const double txy = mu0 * (p[4] + p[1]), txz = mu0 * (p[8] + p[2]), tyz = mu0 * (p[9] + p[6]);
    const double* sn = sL + place[r];
    const double u = sn[0], v = sn[RS], w = sn[2 * RS];
    const double ltxx = -lf[0][0] - u * lf[0][3];
    const double ltxy = -lf[0][1] - v * lf[0][3] - lf[1][0] - u * lf[1][3];
    const double ltxz = -lf[0][2] - w * lf[0][3] - lf[2][0] - u * lf[2][3];
    const double ltyy = -lf[1][1] - v * lf[1][3];
    const double ltyz = -lf[1][2] - w * lf[1][3] - lf[2][1] - v * lf[2][3];
    const double ltzz = -lf[2][2] - w * lf[2][3];
    lq[r][0] = -(txx * lf[0][3] + txy * lf[1][3] + txz * lf[2][3]);
    lq[r][1] = -(txy * lf[0][3] + tyy * lf[1][3] + tyz * lf[2][3]);
    lq[r][2] = -(txz * lf[0][3] + tyz * lf[1][3] + tzz * lf[2][3]);
    lq[r][3] = 0.0;
    // nu = sJ times the adjoint of the gradients, [x][u v w T]
    const double ms = mu0 * sjr, ls = gas.lambda * sjr;
    const double nu[12] = {ms * (gas.s43 * ltxx - gas.s23 * ltyy - gas.s23 * ltzz), ms * ltxy, ms * ltxz, -ls * lf[0][3],
                           ms * ltxy, ms * (-gas.s23 * ltxx + gas.s43 * ltyy - gas.s23 * ltzz), ms * ltyz, -ls * lf[1][3],
                           ms * ltxz, ms * ltyz, ms * (-gas.s23 * ltxx - gas.s23 * ltyy + gas.s43 * ltzz), -ls * lf[2][3]};
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
      for (int x = 0; x < 4; ++x)
        g[r][4 * d + x] = Ja[3 * d] * nu[x] + Ja[3 * d + 1] * nu[4 + x] + Ja[3 * d + 2] * nu[8 + x];
#pragma unroll
    for (int x = 0; x < 12; ++x) now(g[r][x]);
#pragma unroll
    for (int x = 0; x < 3; ++x) now(lq[r][x]);
  }
  // along the lines: transposed derivatives, and the face corrections 0.5*L_hat*(q_nb - q_own).(n SurfElem)
  // at the ends (own part here, the neighbour's part zn to its exchange slot); back to the nodes in place
  double zn[2][4];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int r = 0; r < RN; ++r)
      if (t + r * NT < np) {
#pragma unroll
        for (int d = 0; d < 3; ++d)
#pragma unroll
          for (int w = 0; w < 2; ++w) sL[(X + 2 * d + w) * RS + place[r]] = g[r][4 * d + 2 * h + w];
      }
    __syncthreads();
    if (line) {
      const double* DT = basis + B.D_T() + fresh();
      lp.again();
      double* sX = sL + (X + 2 * q.d) * RS;
      double x[2][n], y[2][n];
#pragma unroll
      for (int w = 0; w < 2; ++w)
#pragma unroll
        for (int l = 0; l < n; ++l) x[w][l] = lp.at(sX, l)[w * RS];
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        zn[0][2 * h + w] = -0.5 * lhm * x[w][0];
        zn[1][2 * h + w] = 0.5 * lhp * x[w][N];
      }
#pragma unroll
      for (int l = 0; l < n; ++l)
#pragma unroll
        for (int i = 0; i < n; ++i)
#pragma unroll
          for (int w = 0; w < 2; ++w) {
            const double z = DT[i + n * l] * x[w][l];
            y[w][i] = l == 0 ? z : y[w][i] + z;
          }
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        y[w][0] -= zn[0][2 * h + w];
        y[w][N] -= zn[1][2 * h + w];
#pragma unroll
        for (int i = 0; i < n; ++i) lp.at(sX, i)[w * RS] = y[w][i];
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RN; ++r)
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        const double* s = sL + (X + w) * RS + place[r];
        lq[r][2 * h + w] += s[0] + s[2 * RS] + s[4 * RS];
      }
  }
  if (line) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      double lP[5];
      prim_adjoint(qn[s], 0.0, gas, 0.0, zn[s][0], zn[s][1], zn[s][2], 0.0, zn[s][3], 0.0, lP);
#pragma unroll
      for (int v = 0; v < 5; ++v) XU[5 * (size_t)q.own[s] + v] += lP[v];
    }
  }
#pragma unroll
  for (int r = 0; r < RN; ++r) {
    if (t + r * NT >= np) continue;
    const size_t gid = e0 + t + r * NT;
    const Prim p = cons_to_prim(c5[r], gas);
    double lU[5];
    prim_adjoint(p, c5[r][4], gas, 0.0, lq[r][0], lq[r][1], lq[r][2], 0.0, lq[r][3], 0.0, lU);
#pragma unroll
    for (int v = 0; v < 5; ++v) out[5 * gid + v] += lU[v];
  }
}

// ---------------------------------------------------------------------------------------------
// out += the neighbours' face parts (XU of the neighbour slot of every own face point)
template <int N>
__global__ __launch_bounds__(D<N>::NT) void k_adj_gather(DevMesh m, const double* __restrict__ XU,
                                                       double* __restrict__ out) {
  constexpr int n = D<N>::n, np = D<N>::np, NT = D<N>::NT, NF = D<N>::NF;
  __shared__ unsigned sIdx[NF];
  const int e = blockIdx.x, t = threadIdx.x;
  for (int x = t; x < NF; x += NT) sIdx[x] = face_slot_tab<N>(m, e, x);
  __syncthreads();
  if (t >= np) return;
  const int i = t % n, j = (t / n) % n, k = t / (n * n);
  const int sides = node_sides<N>(i, j, k);
  if (!sides) return;
  const size_t gid = (size_t)np * e + t;
  double lU[5] = {0, 0, 0, 0, 0};
#pragma unroll 1
  for (int ls = 1; ls <= 6; ++ls) {
    if (!(sides & (1 << (ls - 1)))) continue;
    const unsigned nb = slot_nbr<N>(sIdx[face_point<N>(ls, i, j, k)]);
#pragma unroll
    for (int v = 0; v < 5; ++v) lU[v] += XU[5 * (size_t)nb + v];
  }
#pragma unroll
  for (int v = 0; v < 5; ++v) out[5 * gid + v] += lU[v];
}

// The register update of a reverse LSERK stage (the last one of a chain; the others are applied
// by the next stage's k_adj_euler): ub += out + the neighbours' face parts, rbar = a*lam, in place of lam.
template <int N>
__global__ __launch_bounds__(D<N>::NT) void k_adj_stage_update(DevMesh m, const double* __restrict__ XU,
                                                             const double* __restrict__ out, double* __restrict__ ub,
                                                             double* __restrict__ rbar, double a) {
  constexpr int n = D<N>::n, np = D<N>::np, NT = D<N>::NT, NF = D<N>::NF;
  __shared__ unsigned sIdx[NF];
  const int e = blockIdx.x, t = threadIdx.x;
  for (int x = t; x < NF; x += NT) sIdx[x] = face_slot_tab<N>(m, e, x);
  __syncthreads();
  if (t >= np) return;
  const int i = t % n, j = (t / n) % n, k = t / (n * n);
  const int sides = node_sides<N>(i, j, k);
  const size_t gid = (size_t)np * e + t;
  double g5[5];
#pragma unroll
  for (int v = 0; v < 5; ++v) g5[v] = out[5 * gid + v];
#pragma unroll 1
  for (int ls = 1; ls <= 6; ++ls) {
    if (!(sides & (1 << (ls - 1)))) continue;
    const unsigned nb = slot_nbr<N>(sIdx[face_point<N>(ls, i, j, k)]);
#pragma unroll
    for (int v = 0; v < 5; ++v) g5[v] += XU[5 * (size_t)nb + v];
  }
#pragma unroll
  for (int v = 0; v < 5; ++v) {
    const double u0 = ub[5 * gid + v];
    rbar[5 * gid + v] = a * rbar[5 * gid + v];
    ub[5 * gid + v] = u0 + g5[v];
  }
}

// y += a*x over n doubles
__global__ __launch_bounds__(256) void k_axpy(size_t n, double a, const double* __restrict__ x, double* __restrict__ y) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] += a * x[i];
}

// The transposed-Jacobian parts of one right-hand side at U (FU: its face states, or null: the neighbours'
// states are read from U through m.nbNode): out = the element's
// own parts, XU = the parts of the neighbours' face nodes. lam (+ cub*ub when ub is given) is the
// adjoint of Ut; with pd.XU a previous stage's register update is applied first (k_adj_euler).
template <int N, bool AFF>
hipError_t adj_parts_n(const DevMesh& m, const AdjointWork& w, const Gas& gas, int riemann, const double* U,
                       const double* FU, double* lam, double* ub, double cub, double* out, double* XU, Pending pd,
                       hipStream_t s) {
  const dim3 g(m.nElems), b(S<N>::NT);
#define FXG_LAUNCH(SOLV)                                                                                        \
  hipLaunchKernelGGL((k_adj_euler<N, SOLV, AFF>), g, b, 0, s, U, m, m.basis, FU, lam, ub, cub, gas, out, XU, w.Xg, pd)
  if (riemann == 1) FXG_LAUNCH(1);
  else if (riemann == 3) FXG_LAUNCH(3);
  else FXG_LAUNCH(33);
#undef FXG_LAUNCH
  hipLaunchKernelGGL((k_adj_visc<N, AFF>), g, b, 0, s, U, m, m.basis, FU, (const double*)lam, (const double*)w.Xg, gas,
                     out, XU);
  return hipGetLastError();
}
template <int N>
hipError_t adj_parts(const DevMesh& m, const AdjointWork& w, const Gas& gas, int riemann, const double* U,
                     const double* FU, double* lam, double* ub, double cub, double* out, double* XU, Pending pd,
                     hipStream_t s) {
  return m.aff ? adj_parts_n<N, true>(m, w, gas, riemann, U, FU, lam, ub, cub, out, XU, pd, s)
               : adj_parts_n<N, false>(m, w, gas, riemann, U, FU, lam, ub, cub, out, XU, pd, s);
}

template <int N>
hipError_t adj_gather(const DevMesh& m, const double* XU, double* out, hipStream_t s) {
  hipLaunchKernelGGL((k_adj_gather<N>), dim3(m.nElems), dim3(D<N>::NT), 0, s, m, XU, out);
  return hipGetLastError();
}

template <int N>
hipError_t adj_update(const DevMesh& m, const double* XU, const double* out, double* ub, double* rbar, double a,
                      hipStream_t s) {
  hipLaunchKernelGGL((k_adj_stage_update<N>), dim3(m.nElems), dim3(D<N>::NT), 0, s, m, XU, out, ub, rbar, a);
  return hipGetLastError();
}

}  // namespace

#define FXG_ADJ_SWITCH(CALL)                                                                     \
  switch (m.N) {                                                                                 \
    case 2: return CALL(2);                                                                      \
    case 3: return CALL(3);                                                                      \
    case 4: return CALL(4);                                                                      \
    case 5: return CALL(5);                                                                      \
    case 6: return CALL(6);                                                                      \
    case 7: return CALL(7);                                                                      \
    default: return hipErrorInvalidValue;                                                        \
  }

hipError_t launch_rhs_vjp(const DevMesh& m, const AdjointWork& w, const Gas& gas, int riemann, const double* U,
                          const double* lam, double* out, hipStream_t s) {
  if (!m.nbNode) return hipErrorInvalidValue;
  double* lw = const_cast<double*>(lam);  // read only without a pending update
#define FXG_PARTS(NN) adj_parts<NN>(m, w, gas, riemann, U, nullptr, lw, nullptr, 0.0, out, w.XU[0], Pending{}, s)
  const hipError_t err = [&]() -> hipError_t { FXG_ADJ_SWITCH(FXG_PARTS) }();
#undef FXG_PARTS
  if (err != hipSuccess) return err;
#define FXG_GATHER(NN) adj_gather<NN>(m, w.XU[0], out, s)
  FXG_ADJ_SWITCH(FXG_GATHER)
#undef FXG_GATHER
}

hipError_t launch_adjoint_stage(const DevMesh& m, const AdjointWork& w, const Gas& gas, int riemann, const double* U,
                                const double* FU, double* rbar, double* ubar, double cub, double a, double* out,
                                AdjointChain& ch, hipStream_t s) {
  if (!FU && !m.nbNode) return hipErrorInvalidValue;
  const Pending pd{ch.pending ? w.XU[ch.cur] : nullptr, ch.a};
  const int nxt = ch.pending ? 1 - ch.cur : ch.cur;
#define FXG_PARTS(NN) adj_parts<NN>(m, w, gas, riemann, U, FU, rbar, ubar, cub, out, w.XU[nxt], pd, s)
  const hipError_t err = [&]() -> hipError_t { FXG_ADJ_SWITCH(FXG_PARTS) }();
#undef FXG_PARTS
  ch.cur = nxt;
  ch.pending = true;
  ch.a = a;
  return err;
}

hipError_t launch_adjoint_flush(const DevMesh& m, const AdjointWork& w, double* rbar, double* ubar,
                                const double* out, AdjointChain& ch, hipStream_t s) {
  if (!ch.pending) return hipSuccess;
  ch.pending = false;
#define FXG_UPDATE(NN) adj_update<NN>(m, w.XU[ch.cur], out, ubar, rbar, ch.a, s)
  FXG_ADJ_SWITCH(FXG_UPDATE)
#undef FXG_UPDATE
}
#undef FXG_ADJ_SWITCH

hipError_t launch_axpy(size_t n, double a, const double* x, double* y, hipStream_t s) {
  hipLaunchKernelGGL(k_axpy, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, a, x, y);
  return hipGetLastError();
}

}  // namespace fxg
