// Helpers of the kernels that give each lane a line of nodes of an element (fxg_stage.hip, fxg_weak.hip):
// workgroup sizes, the place of a node in an LDS row, register control, the numerical flux in
// vector form.
#pragma once
#include "fxg_elem.h"

namespace fxg {

// Sizes of a workgroup: one element, one lane per line. At N = 7 one wave more than the 192 lines
// fill, so that a lane has two nodes in the node phases and not three (246 VGPRs, 1.47 ms).
template <int N>
struct S {
  static constexpr int n = N + 1, nf = n * n, np = n * n * n;
  static constexpr int NL = 3 * nf;
  static constexpr int NT = N == 7 ? 256 : ((NL + 63) / 64) * 64;
  static constexpr int RN = (np + NT - 1) / NT;  // nodes per lane in the node phases
  static constexpr int RS = np;                  // doubles per LDS row
};

// Place of node (i,j,k) in an LDS row. For n = 8 and n = 4 an XOR swizzle, so that the lanes of a
// wave, one line each, read n consecutive nodes of their lines without bank conflicts in all three
// directions (the natural order gives the x lines a stride of n doubles, an 8-way conflict at n = 8).
template <int N>
__device__ __forceinline__ int pos(int i, int j, int k) {
  constexpr int n = N + 1;
  if constexpr (n == 8 || n == 4) return (i ^ j) + n * (j ^ k) + n * n * k;
  else return i + n * (j + n * k);
}

// A line of nodes in an LDS row, in bytes: node l stands at first ^ (l * step) with the swizzle
// (step 1, n+1, n(n+1) doubles in the three directions), at first + l * step without. The places are
// formed again in each phase (again()): eight registers less than keeping them.
template <int N>
struct Line {
  int first, step;
  __device__ __forceinline__ Line(int d, int a, int b) {
    constexpr int n = N + 1;
    constexpr bool X = n == 8 || n == 4;
    first = 8 * pos<N>(d == 0 ? 0 : a, d == 0 ? a : (d == 1 ? 0 : b), d == 2 ? 0 : b);
    step = 8 * (d == 0 ? 1 : (d == 1 ? (X ? n + 1 : n) : (X ? n * (n + 1) : n * n)));
  }
  __device__ __forceinline__ void again() { asm volatile("" : "+v"(first), "+v"(step)); }
  __device__ __forceinline__ double* at(double* rows, int l) const {
    constexpr int n = N + 1;
    const int o = (n == 8 || n == 4) ? first ^ (l * step) : first + l * step;
    return reinterpret_cast<double*>(reinterpret_cast<char*>(rows) + o);
  }
};

// A uniform zero the compiler cannot see through: operator tables addressed with it are read again
// (scalar loads) in every phase instead of being kept, and spilled, across all of them.
__device__ __forceinline__ int fresh() {
  int z = 0;
  asm volatile("" : "+s"(z));
  return z;
}

// Computes x here and not later, where its operands would have to be kept.
__device__ __forceinline__ void now(double& x) { asm volatile("" : "+v"(x)); }

struct FaceState {
  double rho, E, H, p, v[3];
};

// Numerical flux (mass, momentum vector, energy) through a face with unit normal n, L on the side n
// points away from: the central part (Pirozzoli's split surface flux, or the mean of the two Euler fluxes)
// and the dissipation of LF, Roe or Roe-entropy-fix. The same flux as riemann_rot's in vector form: the shear waves share one eigenvalue, so
// their part of the dissipation is the tangential vector itself and no tangents are needed; total
// enthalpies come with the states, so no division by the densities.
template <int SOLVER, bool SPLIT>
__device__ __forceinline__ void riemann_vec(const Gas& g, const FaceState& L, const FaceState& R, const double* n, double* F) {
  const double vl = L.v[0] * n[0] + L.v[1] * n[1] + L.v[2] * n[2];
  const double vr = R.v[0] * n[0] + R.v[1] * n[1] + R.v[2] * n[2];
  const double ph = 0.5 * (L.p + R.p);
  const double d0 = R.rho - L.rho, dp = R.p - L.p;
  if constexpr (SPLIT) {
    const double q = 0.125 * (L.rho + R.rho) * (vl + vr);
    F[0] = 2.0 * q;
#pragma unroll
    for (int a = 0; a < 3; ++a) F[1 + a] = ph * n[a] + q * (L.v[a] + R.v[a]);
    F[4] = q * (L.H + R.H);
  } else {
    const double ml = 0.5 * L.rho * vl, mr = 0.5 * R.rho * vr;
    F[0] = ml + mr;
#pragma unroll
    for (int a = 0; a < 3; ++a) F[1 + a] = ph * n[a] + (ml * L.v[a] + mr * R.v[a]);
    F[4] = 0.5 * ((L.E + L.p) * vl + (R.E + R.p) * vr);
  }
  if constexpr (SOLVER == 1) {
    const double cl = sqrt(g.kappa * L.p / L.rho), cr = sqrt(g.kappa * R.p / R.rho);
    const double hm = 0.5 * (fmax(fabs(vr), fabs(vl)) + fmax(cl, cr));
    F[0] -= hm * d0;
#pragma unroll
    for (int a = 0; a < 3; ++a) F[1 + a] -= hm * (R.rho * R.v[a] - L.rho * L.v[a]);
    F[4] -= hm * (R.E - L.E);
  } else {
    const double sl = sqrt(L.rho), sr = sqrt(R.rho);
    const double ss = 1.0 / (sl + sr);
    const double wl = sl * ss, wr = sr * ss;
    double v[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) v[a] = wr * R.v[a] + wl * L.v[a];
    const double u = wr * vr + wl * vl, H = wr * R.H + wl * L.H;
    const double k = v[0] * v[0] + v[1] * v[1] + v[2] * v[2];
    const double c = sqrt(g.kappaM1 * (H - 0.5 * k));
    const double sc = 1.0 / c;
    double vt[3], t[3];  // tangential Roe velocity, tangential jump of the shear waves
#pragma unroll
    for (int a = 0; a < 3; ++a) vt[a] = v[a] - u * n[a];
    double a1, a2, a3, l1, l2, l3;
    if constexpr (SOLVER == 3) {
      double dm[3];
#pragma unroll
      for (int a = 0; a < 3; ++a) dm[a] = R.rho * R.v[a] - L.rho * L.v[a];
      const double dn = R.rho * vr - L.rho * vl;
#pragma unroll
      for (int a = 0; a < 3; ++a) t[a] = dm[a] - dn * n[a] - vt[a] * d0;
      const double d5 = (R.E - L.E) - (t[0] * vt[0] + t[1] * vt[1] + t[2] * vt[2]);
      a2 = g.kappaM1 * (sc * sc) * (d0 * (H - u * u) - d5 + u * dn);
      a1 = 0.5 * sc * (d0 * (u + c) - dn - c * a2);
      a3 = d0 - a1 - a2;
      l1 = fabs(u - c); l2 = fabs(u); l3 = fabs(u + c);
    } else {
      const double cl = sqrt(g.kappa * L.p / L.rho), cr = sqrt(g.kappa * R.p / R.rho);
      const double rd = sqrt(L.rho * R.rho), dv = vr - vl;
      const double h = 0.5 * (sc * sc);
      a1 = h * (dp - rd * c * dv);
      a2 = d0 - dp * 2.0 * h;
      a3 = h * (dp + rd * c * dv);
#pragma unroll
      for (int a = 0; a < 3; ++a) t[a] = rd * (R.v[a] - L.v[a] - dv * n[a]);
      const double x[3] = {u - c, u, u + c}, xl[3] = {vl - cl, vl, vl + cl}, xr[3] = {vr - cr, vr, vr + cr};
      double ab[3];
#pragma unroll
      for (int w = 0; w < 3; ++w) {
        const double da = fmax(fmax(0.0, x[w] - xl[w]), xr[w] - x[w]);
        ab[w] = (fabs(x[w]) < da) ? 0.5 * (x[w] * x[w] / da + da) : fabs(x[w]);
      }
      l1 = ab[0]; l2 = ab[1]; l3 = ab[2];
    }
    const double w1 = 0.5 * a1 * l1, w2 = 0.5 * a2 * l2, w3 = 0.5 * a3 * l3, hl = 0.5 * l2;
    const double s = w1 + w2 + w3, mc = (w3 - w1) * c;
    F[0] -= s;
#pragma unroll
    for (int a = 0; a < 3; ++a) F[1 + a] -= s * v[a] + mc * n[a] + hl * t[a];
    F[4] -= (w1 + w3) * H + mc * u + w2 * (0.5 * k) + hl * (t[0] * vt[0] + t[1] * vt[1] + t[2] * vt[2]);
  }
}

}  // namespace fxg
