// Kernel B of the fused Gauss-Lobatto split-form stage in FP64: everything of a stage after the
// viscous face fluxes (kernel A, fxg_visc.hip), that is the Riemann fluxes of the element's own face
// points, the BR1 gradients (recomputed, never stored), the split-form volume integral, Ut=-Ut*sJ, the
// LSERK register update, the new state's face values and, in the last stage of a step, CALCTIMESTEP's
// spectral radii. The face arrays and the conventions at a face are those described in fxg_fused.hip,
// which holds the FP32-bulk form of this kernel.
#include "fxg_bcface.h"
#include "fxg_line.h"

namespace fxg {
namespace {

// Why lines. One lane per node reads, for each of the 3 (N+1) nodes on its lines, the six primitive
// variables, three metric terms, four viscous fluxes and two operator entries from LDS: about 480 reads
// per node at N = 7, 1 ms of LDS time per launch at 32^3 elements beside 0.8 ms of arithmetic, and every
// pair flux is evaluated twice. Here one lane owns a line of N+1 nodes in one direction (3 (N+1)^2 lanes
// per element): it reads the line once per phase, keeps the sums of all its nodes in registers, evaluates
// each pair once, and takes the operators from scalar registers, since all lanes run the same (i,l). Its
// two end points are face points, so the Riemann fluxes and the surface terms stay in the lane too.
// What couples the directions (the gradients, the sum of the three directions) goes through LDS to
// the node phases, in which the lanes own nodes; about 130 LDS accesses per node in all. At 32^3
// elements, N = 7, Roe: 1.71 -> 1.30 ms per launch, bound by memory (324 bytes per node at 4.2 TB/s;
// a plain copy reaches 4.9). Others: N = 3, 32^3 0.289 -> 0.194 ms, N = 4, 32^3 0.510 -> 0.381,
// N = 5, 24^3 0.346 -> 0.266, N = 6, 24^3 0.889 -> 0.475.
//
// AFF: where every element's metric terms are the same at all of its nodes (parallelepipeds: m.aff, checked
// bitwise at set-up) they are ten uniform values: no metric rows in LDS (13 rows instead of 15, three
// workgroups per CU instead of two at N = 7), 80 bytes per node less to read, and the pair flux needs only the
// sum of the contravariant velocities. N = 7, 32^3: 1.31 -> 1.05 ms (282 bytes per node, 4.5 TB/s); N = 4, 32^3
// 0.381 -> 0.333, N = 5, 24^3 0.268 -> 0.224, N = 6, 24^3 0.475 -> 0.337.

// LDS rows: 0 u, 1 v, 2 w, 3 rho/4, 4 p, 5 H, 6 T; 7..12 exchange between line and node phases
// (two variables in three directions); general metrics: 6..14 Ja^1..3 / 2 in the pair loop. At the
// end the rows carry the three directions' sums to the node lanes.
template <int N, bool AFF>
struct Lds {
  static constexpr int ROWS = AFF ? 13 : 15;
  static constexpr int T = 6, X = 7, JA = 6;
  // the rows, and at least the new state's five and the reduction of the last stage
  static constexpr int RED = 6 * S<N>::NT + 6 + (S<N>::NT / 64 + 1) / 2;
  static constexpr int SIZE = ROWS * S<N>::RS > 5 * S<N>::RS + RED ? ROWS * S<N>::RS : 5 * S<N>::RS + RED;
};

template <int N, int SOLVER, bool BC, bool LAM, bool AFF>
__global__ __launch_bounds__(S<N>::NT)
__attribute__((amdgpu_waves_per_eu(AFF || N <= 5 ? 3 : 2))) void k_stage(const double* U, DevMesh m, const double* __restrict__ basis, const double* __restrict__ FU,
                                                double* __restrict__ FUnext, const double* __restrict__ FG, Gas gas,
                                                double* Ut, RKStage st, double* __restrict__ Gout,
                                                double* __restrict__ bcP) {
  constexpr int n = S<N>::n, nf = S<N>::nf, np = S<N>::np, NL = S<N>::NL, NT = S<N>::NT, RN = S<N>::RN, RS = S<N>::RS;
  using L = Lds<N, AFF>;
  __shared__ double sL[L::SIZE];
  const BasisLayout B{n};
  // U kept in registers for the update where it costs no wave per SIMD (else read again)
  constexpr bool KEEP = AFF ? N <= 4 : (N <= 4 || N >= 6);
  const int e = blockIdx.x;
  // N = 7: the wave without lines is another one in each workgroup, so that no SIMD has it every time
  const int t = N == 7 ? (threadIdx.x + 64 * (e & 3)) % NT : threadIdx.x;
  const bool line = t < NL;
  // line (d; a, b): nodes l = 0..N; its end points are face points of the minus and plus side of d
  const int tl = line ? t : 0;
  const int d = tl / nf, ln = tl - d * nf, la = ln % n, lb = ln / n;
  const int lsm = d == 0 ? 5 : (d == 1 ? 2 : 1), lsp = d == 0 ? 3 : (d == 1 ? 4 : 6);
  const unsigned own0 = m.slotTab[(size_t)6 * nf * e + (lsm - 1) * nf + ln];
  const unsigned own1 = m.slotTab[(size_t)6 * nf * e + (lsp - 1) * nf + ln];
  const size_t e0 = (size_t)np * e;
  const int end0 = d == 0 ? n * ln : (d == 1 ? la + nf * lb : ln);  // the line's first node

  const double* je = AFF ? m.aff + 10 * (size_t)e : nullptr;  // the element's constant metric terms
  double c[RN][5];
#pragma unroll
  for (int r = 0; r < RN; ++r) {
    const int nd = t + r * NT;
#pragma unroll
    for (int v = 0; v < 5; ++v) c[r][v] = nd < np ? U[5 * (e0 + nd) + v] : 1.0;
  }
  double nb[2][5], gn[2][4], Eo[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const size_t o = slot_nbr<N>(s ? own1 : own0);
#pragma unroll
    for (int v = 0; v < 5; ++v) nb[s][v] = FU[5 * o + v];
#pragma unroll
    for (int v = 0; v < 4; ++v) gn[s][v] = FG[4 * o + v];
    // the own energy as stored: from the enthalpy its rounding would enter the energy jump times c
    Eo[s] = U[5 * (e0 + end0 + s * N * (d == 0 ? 1 : (d == 1 ? n : nf))) + 4];
  }
  int np_[RN];  // LDS places of the lane's nodes
#pragma unroll
  for (int r = 0; r < RN; ++r) {
    const int nd = t + r * NT;
    np_[r] = nd < np ? pos<N>(nd % n, (nd / n) % n, nd / nf) : 0;
  }
#pragma unroll
  for (int r = 0; r < RN; ++r) {
    if (t + r * NT < np) {
      const Prim q = cons_to_prim(c[r], gas);
      double* s = sL + np_[r];
      s[0] = q.u; s[RS] = q.v; s[2 * RS] = q.w; s[3 * RS] = 0.25 * q.rho; s[4 * RS] = q.p;
      s[5 * RS] = (c[r][4] + q.p) * q.srho; s[6 * RS] = q.T;
    }
  }
  Line<N> lp(d, la, lb);
  const double lhm = basis[B.L_HatMinus()], lhp = basis[B.L_HatPlus() + N];
  __syncthreads();

  // Surface terms at the two ends of the line: the Riemann flux with the neighbour's state and the
  // neighbour's half of the viscous normal flux (fs), and the BR1 jump of u, v, w, T (jq).
  double fs[2][5], jq[2][4];
  double mj[3] = {0, 0, 0};  // AFF: Ja^d of the line
  if constexpr (AFF) {
#pragma unroll
    for (int x = 0; x < 3; ++x) mj[x] = d == 0 ? je[x] : (d == 1 ? je[3 + x] : je[6 + x]);
  }
  if (line) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const unsigned own = s ? own1 : own0;
      const bool master = slot_is_master<N>(own);
      const double ms = master ? 1.0 : -1.0, sg = s ? 1.0 : -1.0, lh = s ? lhp : lhm;
      double se, nv[3];  // master normal
      if (m.ownFaceMetric) {
        double ns[3];
        if constexpr (AFF) {
#pragma unroll
          for (int x = 0; x < 3; ++x) ns[x] = mj[x];
        } else {
          const int id = end0 + (s ? N * (d == 0 ? 1 : (d == 1 ? n : nf)) : 0);
          const double* Jd = (d == 0 ? m.Mf : (d == 1 ? m.Mg : m.Mh)) + 3 * (e0 + id);
#pragma unroll
          for (int x = 0; x < 3; ++x) ns[x] = Jd[x];
        }
        se = sqrt(ns[0] * ns[0] + ns[1] * ns[1] + ns[2] * ns[2]);
        const double f = ms * sg / se;
#pragma unroll
        for (int x = 0; x < 3; ++x) nv[x] = ns[x] * f;
      } else {
        const size_t sp = slot_side_point<N>(own);
        se = m.SurfElem[sp];
#pragma unroll
        for (int x = 0; x < 3; ++x) nv[x] = m.NormVec[3 * sp + x];
      }
      const double* so = lp.at(sL, s ? N : 0);
      const FaceState o{4.0 * so[3 * RS], Eo[s], so[5 * RS], so[4 * RS], {so[0], so[RS], so[2 * RS]}};
      const Prim q = cons_to_prim(nb[s], gas);
      const FaceState b{q.rho, nb[s][4], (nb[s][4] + q.p) * q.srho, q.p, {q.u, q.v, q.w}};
      const double hs = sg * 0.5 * lh;
      jq[s][0] = hs * (q.u - o.v[0]); jq[s][1] = hs * (q.v - o.v[1]); jq[s][2] = hs * (q.w - o.v[2]);
      jq[s][3] = hs * (q.T - so[6 * RS]);
      double F[5];
      bool wall = false;
      if constexpr (BC) {
        // a wall side: the inviscid flux is (0, p_wall n, 0) (getboundaryflux.f90:580-592)
        const int side = (int)(own / (2u * (unsigned)nf));
        if (side < m.nBC && !bc_riemann_type(m.bcInfo[2 * side])) {
          wall = true;
          const double pw = bcP[4 * slot_side_point<N>(own)];
          F[0] = F[4] = 0.0;
#pragma unroll
          for (int x = 0; x < 3; ++x) F[1 + x] = pw * nv[x];
        }
      }
      if (!wall) {
        // the master's state on the left, so that both elements of a side evaluate the same flux
        FaceState l = o, r = b;
        if (!master) { l = b; r = o; }
        riemann_vec<SOLVER, true>(gas, l, r, nv, F);
      }
      const double f = ms * se;
      fs[s][0] = 0.5 * (f * F[0]) * lh;
#pragma unroll
      for (int v = 0; v < 4; ++v) fs[s][1 + v] = (f * F[1 + v] - 0.5 * gn[s][v]) * lh;
#pragma unroll
      for (int v = 0; v < 5; ++v) now(fs[s][v]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  // BR1 gradients: reference derivatives along the lines with the face corrections at their ends, two
  // variables at a time through the exchange rows to the node lanes
  double g[RN][12];  // reference derivatives, then contravariant viscous fluxes: [d][u v w T]
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    if (line) {
      const double* DT = basis + B.D_T() + fresh();
      lp.again();
      double* sX = sL + (L::X + 2 * d) * RS;
      double q[2][n];
#pragma unroll
      for (int w = 0; w < 2; ++w)
#pragma unroll
        for (int l = 0; l < n; ++l) q[w][l] = lp.at(sL, l)[(2 * h + w < 3 ? 2 * h + w : L::T) * RS];
#pragma unroll
      for (int i = 0; i < n; ++i)
#pragma unroll
        for (int w = 0; w < 2; ++w) {
          double a = DT[n * i] * q[w][0];
#pragma unroll
          for (int l = 1; l < n; ++l) a += DT[l + n * i] * q[w][l];
          if (i == 0) a += jq[0][2 * h + w];
          if (i == N) a += jq[1][2 * h + w];
          lp.at(sX, i)[w * RS] = a;
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RN; ++r)
#pragma unroll
      for (int x = 0; x < 3; ++x)
#pragma unroll
        for (int w = 0; w < 2; ++w) g[r][4 * x + 2 * h + w] = sL[(L::X + 2 * x + w) * RS + np_[r]];
    __syncthreads();
  }
  // node lanes: physical gradients, viscous flux, contravariant viscous flux in place of g
  constexpr int RJ = AFF ? 1 : RN;
  double Ja[RJ][9];
  const GasT<double> gt(gas);
  const double* jn = AFF ? je + fresh() : nullptr;
#pragma unroll
  for (int r = 0; r < RN; ++r) {
    const int nd = t + r * NT;
    double sj;
    const int rj = AFF ? 0 : r;
    if constexpr (AFF) {
      sj = jn[9];
      if (r == 0)
#pragma unroll
        for (int x = 0; x < 9; ++x) Ja[0][x] = jn[x];
    } else {
      load_metrics<double>(m, e0 + (nd < np ? nd : 0), Ja[r], sj);
    }
    double p[12];
#pragma unroll
    for (int x = 0; x < 3; ++x)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        p[4 * x + v] = (Ja[rj][x] * g[r][v] + Ja[rj][3 + x] * g[r][4 + v] + Ja[rj][6 + x] * g[r][8 + v]) * sj;
    if (Gout && nd < np) {  // (np, 12, nElems)
#pragma unroll
      for (int x = 0; x < 12; ++x) Gout[nd + (size_t)np * (x + 12 * (size_t)e)] = p[x];
    }
    double fx[4], fy[4], fz[4];
    const double* s = sL + np_[r];
    diff_flux<double>(gt, s[0], s[RS], s[2 * RS], p, p + 4, p + 8, fx, fy, fz);
#pragma unroll
    for (int x = 0; x < 3; ++x)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        g[r][4 * x + v] = Ja[rj][3 * x] * fx[v] + Ja[rj][3 * x + 1] * fy[v] + Ja[rj][3 * x + 2] * fz[v];
#pragma unroll
    for (int x = 0; x < 12; ++x) now(g[r][x]);
  }

  // viscous part of the volume integral: back through the exchange rows, contracted along the lines
  // (acc[0] holds half the mass sum)
  double acc[5][n];
  if (line) {
#pragma unroll
    for (int v = 0; v < 5; ++v) {
#pragma unroll
      for (int i = 0; i < n; ++i) acc[v][i] = 0.0;
      acc[v][0] = fs[0][v];
      acc[v][N] = fs[1][v];
    }
  }
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int r = 0; r < RN; ++r)
      if (t + r * NT < np) {
#pragma unroll
        for (int x = 0; x < 3; ++x)
#pragma unroll
          for (int w = 0; w < 2; ++w) sL[(L::X + 2 * x + w) * RS + np_[r]] = g[r][4 * x + 2 * h + w];
      }
    __syncthreads();
    if (line) {
      const double* DH = basis + B.D_Hat_T() + fresh();
      lp.again();
      double* sX = sL + (L::X + 2 * d) * RS;
      double f[2][n];
#pragma unroll
      for (int w = 0; w < 2; ++w)
#pragma unroll
        for (int l = 0; l < n; ++l) f[w][l] = lp.at(sX, l)[w * RS];
#pragma unroll
      for (int w = 0; w < 2; ++w) {  // the own half of the viscous normal flux at the line's ends
        acc[1 + 2 * h + w][0] -= 0.5 * lhm * f[w][0];
        acc[1 + 2 * h + w][N] += 0.5 * lhp * f[w][N];
      }
#pragma unroll
      for (int i = 0; i < n; ++i)
#pragma unroll
        for (int l = 0; l < n; ++l)
#pragma unroll
          for (int w = 0; w < 2; ++w) acc[1 + 2 * h + w][i] += DH[l + n * i] * f[w][l];
    }
    __syncthreads();
  }
  if constexpr (!AFF) {
#pragma unroll
    for (int r = 0; r < RN; ++r)
      if (t + r * NT < np)
#pragma unroll
        for (int x = 0; x < 9; ++x) sL[(L::JA + x) * RS + np_[r]] = 0.5 * Ja[r][x];
    __syncthreads();
  }

  // Split-form volume integral (volint.f90:211-371 with splitflux.f90:603-666): each pair of a line
  // once, with z = (rho_s/4) (a . v_s), a the metric average: F = (2 z, z v_s + a p_s, z H_s).
  if (line) {
    const double* W = basis + B.PairD() + fresh();
    lp.again();
    double* sJ9 = sL + (L::JA + 3 * d) * RS;
    constexpr int TB = 2;  // nodes held at a time; the later ones of the line are read once per block
    struct Nd {
      double r, u, v, w, p, H, c, j[3];
    };
    auto load = [&](int l) {
      const double* s = lp.at(sL, l);
      Nd q;
      q.u = s[0]; q.v = s[RS]; q.w = s[2 * RS]; q.r = s[3 * RS]; q.p = s[4 * RS]; q.H = s[5 * RS];
      if constexpr (AFF) {
        q.c = mj[0] * q.u + mj[1] * q.v + mj[2] * q.w;
      } else {
        const double* J = lp.at(sJ9, l);
        q.j[0] = J[0]; q.j[1] = J[RS]; q.j[2] = J[2 * RS];
      }
      return q;
    };
    auto pair = [&](const Nd& A, const Nd& C, int i, int l) {
      const double us = A.u + C.u, vs = A.v + C.v, ws = A.w + C.w, ps = A.p + C.p;
      double b0, b1, b2, z;
      if constexpr (AFF) {
        b0 = mj[0]; b1 = mj[1]; b2 = mj[2];
        z = (A.r + C.r) * (A.c + C.c);
      } else {
        b0 = A.j[0] + C.j[0]; b1 = A.j[1] + C.j[1]; b2 = A.j[2] + C.j[2];
        z = (A.r + C.r) * (b0 * us + b1 * vs + b2 * ws);
      }
      // (the pressure, the large term at low Mach number, in the fused multiply-add: one rounding)
      const double F1 = b0 * ps + z * us, F2 = b1 * ps + z * vs, F3 = b2 * ps + z * ws, F4 = z * (A.H + C.H);
      const int pr = i * (2 * n - i - 1) / 2 + l - i - 1;
      const double x = W[2 * pr], y = W[2 * pr + 1];  // D(i,l), D(l,i)
      acc[0][i] += x * z; acc[1][i] += x * F1; acc[2][i] += x * F2; acc[3][i] += x * F3; acc[4][i] += x * F4;
      acc[0][l] += y * z; acc[1][l] += y * F1; acc[2][l] += y * F2; acc[3][l] += y * F3; acc[4][l] += y * F4;
    };
#pragma unroll
    for (int i0 = 0; i0 < n; i0 += TB) {
      Nd A[TB];
#pragma unroll
      for (int a = 0; a < TB; ++a)
        if (i0 + a < n) A[a] = load(i0 + a);
#pragma unroll
      for (int a = 0; a < TB; ++a)
#pragma unroll
        for (int b = a + 1; b < TB; ++b)
          if (i0 + b < n) pair(A[a], A[b], i0 + a, i0 + b);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int l = i0 + TB; l < n; ++l) {
        const Nd C = load(l);
#pragma unroll
        for (int a = 0; a < TB; ++a)
          if (i0 + a < n) pair(A[a], C, i0 + a, l);
        __builtin_amdgcn_sched_barrier(0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  __syncthreads();  // the pair loop's rows are free

  // sum of the three directions at each node, through all rows at once or (13 rows) with the third
  // direction's last two components in a second round
  double sum[RN][5];
  constexpr int C1 = L::ROWS >= 15 ? 5 : 3;
  if (line) {
    lp.again();
    double* sS = sL + 5 * d * RS;
#pragma unroll
    for (int v = 0; v < 5; ++v)
      if (v < C1 || d < 2) {
#pragma unroll
        for (int i = 0; i < n; ++i) lp.at(sS, i)[v * RS] = acc[v][i];
      }
  }
  // register and state of the update
  double up[RN][5], rp[RN][5], sj[RN];
#pragma unroll
  for (int r = 0; r < RN; ++r) {
    const size_t gid = e0 + (t + r * NT < np ? t + r * NT : 0);
    if constexpr (AFF) sj[r] = je[9 + fresh()]; else sj[r] = m.sJ[gid];
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      up[r][v] = KEEP ? c[r][v] : (st.mode != 0 ? U[5 * gid + v] : 0.0);
      rp[r][v] = st.mode == 2 ? st.R[5 * gid + v] : 0.0;
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < RN; ++r)
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      sum[r][v] = sL[v * RS + np_[r]] + sL[(5 + v) * RS + np_[r]];
      if (v < C1) sum[r][v] += sL[(10 + v) * RS + np_[r]];
    }
  __syncthreads();
  if constexpr (C1 < 5) {
    if (line && d == 2) {
#pragma unroll
      for (int v = C1; v < 5; ++v)
#pragma unroll
        for (int i = 0; i < n; ++i) lp.at(sL, i)[v * RS] = acc[v][i];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RN; ++r)
#pragma unroll
      for (int v = C1; v < 5; ++v) sum[r][v] += sL[v * RS + np_[r]];
    __syncthreads();
  }
  // Ut = -Ut*sJ and the register update
  if (st.mode == 0) {
#pragma unroll
    for (int r = 0; r < RN; ++r) {
      const int nd = t + r * NT;
      if (nd < np)
#pragma unroll
        for (int v = 0; v < 5; ++v) Ut[5 * (e0 + nd) + v] = (-(v == 0 ? 2.0 : 1.0) * sum[r][v]) * sj[r];
    }
    return;
  }
#pragma unroll
  for (int r = 0; r < RN; ++r)
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      const double ut = (-(v == 0 ? 2.0 : 1.0) * sum[r][v]) * sj[r];
      rp[r][v] = (st.mode == 1) ? ut : rp[r][v] * st.minusA + ut;
      up[r][v] = up[r][v] + rp[r][v] * st.b_dt;
      if (t + r * NT < np) sL[v * RS + np_[r]] = up[r][v];
    }
  if constexpr (LAM) {
    // CALCTIMESTEP's spectral radii of the new state, before the stores (a wait for the wave's
    // outstanding memory operations precedes the reduction's cross-lane moves)
    double lam[6] = {0, 0, 0, 0, 0, 0};
    int isnan_rho = 0;
#pragma unroll
    for (int r = 0; r < RN; ++r) {
      const int nd = t + r * NT;
      if (nd < np) {
        double ln6[6];
        int nr;
        if constexpr (AFF) dt_node_lambda(up[r], gas, je[9], je, je + 3, je + 6, ln6, nr);
        else dt_node_lambda(up[r], gas, sj[r], m.Mf + 3 * (e0 + nd), m.Mg + 3 * (e0 + nd), m.Mh + 3 * (e0 + nd), ln6, nr);
        isnan_rho |= nr;
#pragma unroll
        for (int x = 0; x < 6; ++x) lam[x] = (ln6[x] > lam[x] || ln6[x] != ln6[x]) ? ln6[x] : lam[x];
      }
    }
    double mx[6];
    int nanr = 0;
    double* red = sL + 5 * RS;  // rows beyond the new state's
    block_lambda_max_rows<NT, NT>(lam, isnan_rho, red, red + 6 * NT, reinterpret_cast<int*>(red + 6 * NT + 6), t, mx, nanr);
    if (t == 0) {
      st.lamSum[2 * e] = mx[0] + mx[1] + mx[2];
      st.lamSum[2 * e + 1] = mx[3] + mx[4] + mx[5];
      st.lamNan[e] = nanr;
    }
  }
#pragma unroll
  for (int r = 0; r < RN; ++r) {
    const size_t o = 5 * (e0 + t + r * NT);
    if (t + r * NT < np) {
#pragma unroll
      for (int v = 0; v < 5; ++v) st.R[o + v] = rp[r][v];
#pragma unroll
      for (int v = 0; v < 5; ++v) st.U[o + v] = up[r][v];
    }
  }
  __syncthreads();
  // the new state's face values for the next stage, by the lines' ends
  if (line) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const unsigned own = m.slotTab[(size_t)6 * nf * e + ((s ? lsp : lsm) - 1) * nf + ln];
      double* dst = FUnext + 5 * (size_t)own;
      const double* src = lp.at(sL, s ? N : 0);
      double u[5];
#pragma unroll
      for (int v = 0; v < 5; ++v) dst[v] = u[v] = src[v * RS];
      if constexpr (BC) {
        // a boundary side: its outer slot of the next stage too (a kernel of its own otherwise). bcP of this
        // point was last read above, by this lane
        const int side = (int)(own / (2u * (unsigned)nf));
        if (side < m.nBC) bc_ghost_point(m, u, dst + 5 * nf, bcP, gas, slot_side_point<N>(own), side);
      }
    }
  }
}

template <int N, bool AFF>
hipError_t stage_n(const DevMesh& m, const FusedWork& w, const Gas& gas, int riemann, const double* U, double* Ut,
                   const RKStage& st, int cur, double* G, hipStream_t s) {
  const dim3 g(m.nElems), b(S<N>::NT);
  const bool bc = m.nBC > 0;
  const double* FUc = w.FU[cur];
  double* FUn = w.FU[1 - cur];
#define FXG_LAUNCH(SOLV, BCV)                                                                                          \
  if (st.lamSum)                                                                                                       \
    hipLaunchKernelGGL((k_stage<N, SOLV, BCV, true, AFF>), g, b, 0, s, U, m, m.basis, FUc, FUn, (const double*)w.FG,  \
                       gas, Ut, st, G, w.bcP);                                                                         \
  else                                                                                                                 \
    hipLaunchKernelGGL((k_stage<N, SOLV, BCV, false, AFF>), g, b, 0, s, U, m, m.basis, FUc, FUn, (const double*)w.FG, \
                       gas, Ut, st, G, w.bcP)
  if (riemann == 1) {
    if (bc) FXG_LAUNCH(1, true); else FXG_LAUNCH(1, false);
  } else if (riemann == 3) {
    if (bc) FXG_LAUNCH(3, true); else FXG_LAUNCH(3, false);
  } else {
    if (bc) FXG_LAUNCH(33, true); else FXG_LAUNCH(33, false);
  }
#undef FXG_LAUNCH
  return hipGetLastError();
}

}  // namespace

hipError_t launch_stage(const DevMesh& m, const FusedWork& w, const Gas& gas, int riemann, const double* U, double* Ut,
                        const RKStage& st, int cur, double* G, hipStream_t s) {
  switch (m.N) {
#define FXG_CASE(NN) \
  case NN:           \
    return m.aff ? stage_n<NN, true>(m, w, gas, riemann, U, Ut, st, cur, G, s) \
                 : stage_n<NN, false>(m, w, gas, riemann, U, Ut, st, cur, G, s);
    FXG_CASE(2) FXG_CASE(3) FXG_CASE(4) FXG_CASE(5) FXG_CASE(6) FXG_CASE(7)
#undef FXG_CASE
    default: return hipErrorInvalidValue;
  }
}

}  // namespace fxg
