// Two-kernel stage of the weak form in FP64 (Gauss and Gauss-Lobatto nodes) on meshes without boundary
// sides, with one lane per line of nodes as in fxg_stage.hip.
//
//   A  k_weak_visc:  per element, the BR1 gradients (lifting_br1.t90:48-181), the viscous stresses and
//      heat fluxes, prolonged to its six faces, and there the viscous normal flux f_v . (n SurfElem) seen
//      from that element (riemann.f90:448-498) into FG, 4 values per face point.
//   B  k_weak_stage: per element, the Riemann fluxes of its own face points, the gradients once more, the
//      weak volume integral of the Euler and viscous fluxes (volint.f90:117-187), the surface integral,
//      Ut=-Ut*sJ, the register update and the new state's face values for the next stage.
// The face states FU are kept per side slot, ((side*2 + slot)*(N+1)^2 + pq), slot 0 master, and
// double-buffered across stages as on the split form's path; k_weak_faces fills them where no stage has.
//
// The four-kernel path (fxg_kernels.hip) stores the gradients (96 bytes per node written and read again) and
// reads the metric terms and U in two more passes: about 950 bytes per node at N = 5 against 742 here (on
// parallelepipeds 558 at N = 3, 402 at N = 7), and its element kernels, one lane per node, are bound by LDS reads. A stage
// (all kernels) on Gauss nodes, Roe: N = 3, 32^3 0.67 -> 0.29 ms; N = 5, 24^3 0.85 -> 0.36 (curved 0.86 -> 0.51);
// N = 7, 32^3 4.75 -> 1.70. At 8^3, N = 3 two kernels of 13 us together instead of four of 31.
// N = 7 is held to two waves per SIMD: at three both kernels spill, at the same time. Below, Roe-entropy-fix
// spills 2 to 24 VGPRs at three (Roe at most 4); a step at 17^3, N = 5: 1.57 -> 1.03 ms curved, 1.58 -> 0.77 straight
// (Roe 1.57 -> 0.97 and 1.58 -> 0.68).
#include "fxg_line.h"

namespace fxg {
namespace {

// LDS rows: 0 u, 1 v, 2 w, 3 T; 4..9 exchange between line and node phases. Then, on Gauss nodes with general
// metric terms, per own face point the lifting flux (4) and n SurfElem (3): these differ from the
// metric terms along the line, so the node lanes add the surface part of the gradients themselves.
template <int N, bool FOLD>
struct LdsW {
  static constexpr int X = 4, ROWS = 10, FACE = ROWS * S<N>::RS, NF = 6 * S<N>::nf;
  static constexpr int SIZE = FACE + (FOLD ? 0 : 7 * NF);
};

// The line of a lane: direction, place, end points' side slots.
struct LineId {
  int d, ln, a, b, lsm, lsp;
};
template <int N>
__device__ __forceinline__ LineId line_id(int t) {
  constexpr int n = N + 1, nf = n * n;
  LineId q;
  q.d = t / nf; q.ln = t - q.d * nf; q.a = q.ln % n; q.b = q.ln / n;
  q.lsm = q.d == 0 ? 5 : (q.d == 1 ? 2 : 1);
  q.lsp = q.d == 0 ? 3 : (q.d == 1 ? 4 : 6);
  return q;
}

// n SurfElem of an own face point, outward, for the flux: the element's own face metric where the
// library computed the metric terms (the slave's in slaveNS; constant metric terms: from these), else the side's.
template <int N, bool AFF>
__device__ __forceinline__ void outward(const DevMesh& m, const double* je, int d, int s, unsigned own, double* ns) {
  if (AFF && m.ownFaceMetric) {
#pragma unroll
    for (int x = 0; x < 3; ++x) ns[x] = (s ? 1.0 : -1.0) * (d == 0 ? je[x] : (d == 1 ? je[3 + x] : je[6 + x]));
    return;
  }
  const size_t sp = slot_side_point<N>(own);
  if (!slot_is_master<N>(own) && m.slaveNS) {
#pragma unroll
    for (int x = 0; x < 3; ++x) ns[x] = -m.slaveNS[3 * sp + x];
  } else {
    const double f = (slot_is_master<N>(own) ? 1.0 : -1.0) * m.SurfElem[sp];
#pragma unroll
    for (int x = 0; x < 3; ++x) ns[x] = m.NormVec[3 * sp + x] * f;
  }
}

// BR1 jump of u, v, w, T at an own face point, (q_nb - q_own)/2, from the two face states.
__device__ __forceinline__ void jump(const Prim& o, const Prim& b, double* j) {
  j[0] = 0.5 * (b.u - o.u); j[1] = 0.5 * (b.v - o.v); j[2] = 0.5 * (b.w - o.w); j[3] = 0.5 * (b.T - o.T);
}

// The gradients of u, v, w, T at the lane's nodes, p[r][4*x + v], without the factor sJ. In: rows 0..3, the
// jumps of the lane's line; the side's normals in the face rows or (FOLD) folded into the line
// derivatives. Ends with every lane past its reads of rows 0..3.
template <int N, bool GL, bool AFF, bool FOLD>
__device__ __forceinline__ void gradients(const DevMesh& m, const double* basis, const double* je, size_t e0, int t, bool line,
                                          int d, Line<N> lp, const int* place, const double jq[2][4], double* sL,
                                          double (*p)[12]) {
  constexpr int n = S<N>::n, np = S<N>::np, NT = S<N>::NT, RN = S<N>::RN, RS = S<N>::RS;
  using L = LdsW<N, FOLD>;
  const BasisLayout B{n};
  double g[RN][12];
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
        for (int l = 0; l < n; ++l) q[w][l] = lp.at(sL, l)[(2 * h + w) * RS];
#pragma unroll
      for (int i = 0; i < n; ++i)
#pragma unroll
        for (int w = 0; w < 2; ++w) {
          double a = DT[n * i] * q[w][0];
#pragma unroll
          for (int l = 1; l < n; ++l) a += DT[l + n * i] * q[w][l];
          if constexpr (FOLD) {
            if constexpr (GL) {
              if (i == 0) a -= jq[0][2 * h + w] * basis[B.L_HatMinus()];
              if (i == N) a += jq[1][2 * h + w] * basis[B.L_HatPlus() + N];
            } else {
              a += jq[1][2 * h + w] * basis[B.L_HatPlus() + i] - jq[0][2 * h + w] * basis[B.L_HatMinus() + i];
            }
          }
          lp.at(sX, i)[w * RS] = a;
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RN; ++r)
#pragma unroll
      for (int x = 0; x < 3; ++x)
#pragma unroll
        for (int w = 0; w < 2; ++w) g[r][4 * x + 2 * h + w] = sL[(L::X + 2 * x + w) * RS + place[r]];
    __syncthreads();
  }
#pragma unroll
  for (int r = 0; r < RN; ++r) {
    const int nd = t + r * NT < np ? t + r * NT : 0;
    double J[9];
    if constexpr (AFF) {
#pragma unroll
      for (int x = 0; x < 9; ++x) J[x] = je[x];
    } else {
      double sj;
      load_metrics<double>(m, e0 + nd, J, sj);
    }
#pragma unroll
    for (int x = 0; x < 3; ++x)
#pragma unroll
      for (int v = 0; v < 4; ++v) p[r][4 * x + v] = J[x] * g[r][v] + J[3 + x] * g[r][4 + v] + J[6 + x] * g[r][8 + v];
    if constexpr (!FOLD) {
      constexpr int nf = n * n, NF = L::NF;
      const int at[3] = {nd % n, (nd / n) % n, nd / nf};
      const int ln[3] = {nd / n, at[0] + n * at[2], nd % nf};
#pragma unroll
      for (int q = 0; q < 3; ++q)
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const double lh = basis[(s ? B.L_HatPlus() : B.L_HatMinus()) + at[q]];
          const double* F = sL + L::FACE + (2 * q + s) * nf + ln[q];
#pragma unroll
          for (int x = 0; x < 3; ++x) {
            const double ns = F[(4 + x) * NF] * lh;
#pragma unroll
            for (int v = 0; v < 4; ++v) p[r][4 * x + v] += F[v * NF] * ns;
          }
        }
    }
#pragma unroll
    for (int x = 0; x < 12; ++x) now(p[r][x]);
  }
}

// Face states of U into the side slots: prolongation along the lines (Gauss), or the end nodes.
template <int N, bool GL>
__global__ __launch_bounds__(S<N>::NT) void k_weak_faces(const double* __restrict__ U, DevMesh m,
                                                       const double* __restrict__ basis, double* __restrict__ FU) {
  constexpr int n = S<N>::n, nf = S<N>::nf, np = S<N>::np, NL = S<N>::NL, NT = S<N>::NT, RN = S<N>::RN, RS = S<N>::RS;
  __shared__ double sL[5 * RS];  // through LDS: the lines of a wave would read U in pieces of 40 bytes
  const BasisLayout B{n};
  const int e = blockIdx.x, t = threadIdx.x;
  double c[RN][5];
#pragma unroll
  for (int r = 0; r < RN; ++r)
#pragma unroll
    for (int v = 0; v < 5; ++v) c[r][v] = t + r * NT < np ? U[5 * ((size_t)np * e + t + r * NT) + v] : 0.0;
#pragma unroll
  for (int r = 0; r < RN; ++r) {
    const int nd = t + r * NT;
    if (nd < np)
#pragma unroll
      for (int v = 0; v < 5; ++v) sL[v * RS + pos<N>(nd % n, (nd / n) % n, nd / nf)] = c[r][v];
  }
  __syncthreads();
  if (t >= NL) return;
  const LineId q = line_id<N>(t);
  const Line<N> lp(q.d, q.a, q.b);
  double f[2][5] = {{0, 0, 0, 0, 0}, {0, 0, 0, 0, 0}};
#pragma unroll
  for (int l = 0; l < n; ++l) {
    if (GL && l != 0 && l != N) continue;
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      const double x = lp.at(sL, l)[v * RS];
      if constexpr (GL) {
        if (l == 0) f[0][v] = x;
        if (l == N) f[1][v] = x;
      } else {
        f[0][v] += basis[B.L_Minus() + l] * x;
        f[1][v] += basis[B.L_Plus() + l] * x;
      }
    }
  }
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    double* dst = FU + 5 * (size_t)m.slotTab[(size_t)6 * nf * e + ((s ? q.lsp : q.lsm) - 1) * nf + q.ln];
#pragma unroll
    for (int v = 0; v < 5; ++v) dst[v] = f[s][v];
  }
}

// Kernel A.
template <int N, bool GL, bool AFF>
__global__ __launch_bounds__(S<N>::NT) __attribute__((amdgpu_waves_per_eu(N == 7 ? 2 : 3))) void k_weak_visc(
    const double* __restrict__ U, DevMesh m, const double* __restrict__ basis, const double* __restrict__ FU,
    double* __restrict__ FG, Gas gas) {
  constexpr int n = S<N>::n, nf = S<N>::nf, np = S<N>::np, NL = S<N>::NL, NT = S<N>::NT, RN = S<N>::RN, RS = S<N>::RS;
  constexpr bool FOLD = GL || AFF;
  using L = LdsW<N, FOLD>;
  __shared__ double sL[L::SIZE];
  const BasisLayout B{n};
  const int e = blockIdx.x, t = N == 7 ? (threadIdx.x + 64 * (e & 3)) % NT : threadIdx.x;
  const bool line = t < NL;
  const LineId id = line_id<N>(line ? t : 0);
  const unsigned own[2] = {m.slotTab[(size_t)6 * nf * e + (id.lsm - 1) * nf + id.ln],
                           m.slotTab[(size_t)6 * nf * e + (id.lsp - 1) * nf + id.ln]};
  const size_t e0 = (size_t)np * e;
  const double* je = AFF ? m.aff + 10 * (size_t)e : nullptr;
  double c[RN][5];
#pragma unroll
  for (int r = 0; r < RN; ++r)
#pragma unroll
    for (int v = 0; v < 5; ++v) c[r][v] = t + r * NT < np ? U[5 * (e0 + t + r * NT) + v] : 1.0;
  double fo[2][5], fb[2][5];
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      fo[s][v] = FU[5 * (size_t)own[s] + v];
      fb[s][v] = FU[5 * (size_t)slot_nbr<N>(own[s]) + v];
    }
  int place[RN];
#pragma unroll
  for (int r = 0; r < RN; ++r) {
    const int nd = t + r * NT < np ? t + r * NT : 0;
    place[r] = pos<N>(nd % n, (nd / n) % n, nd / nf);
    if (t + r * NT < np) {
      const Prim q = cons_to_prim(c[r], gas);
      double* s = sL + place[r];
      s[0] = q.u; s[RS] = q.v; s[2 * RS] = q.w; s[3 * RS] = q.T;
    }
  }
  double jq[2][4], uf[2][3];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const Prim o = cons_to_prim(fo[s], gas), b = cons_to_prim(fb[s], gas);
    jump(o, b, jq[s]);
    uf[s][0] = o.u; uf[s][1] = o.v; uf[s][2] = o.w;
    if constexpr (!FOLD) {
      if (line) {
        // the lifting takes the side's normal on both sides
        const size_t sp = slot_side_point<N>(own[s]);
        const double f = (slot_is_master<N>(own[s]) ? 1.0 : -1.0) * m.SurfElem[sp];
        double* F = sL + L::FACE + (2 * id.d + s) * nf + id.ln;
#pragma unroll
        for (int v = 0; v < 4; ++v) F[v * L::NF] = jq[s][v];
#pragma unroll
        for (int x = 0; x < 3; ++x) F[(4 + x) * L::NF] = m.NormVec[3 * sp + x] * f;
      }
    }
  }
  Line<N> lp(id.d, id.a, id.b);
  __syncthreads();
  double p[RN][12];
  gradients<N, GL, AFF, FOLD>(m, basis, je, e0, t, line, id.d, lp, place, jq, sL, p);
  // stresses and heat flux at the nodes into rows 0..8, then prolonged to the ends of the lines
#pragma unroll
  for (int r = 0; r < RN; ++r)
    if (t + r * NT < np) {
      const double sj = AFF ? je[9] : m.sJ[e0 + t + r * NT];
      const double mu = gas.mu0 * sj, la = gas.lambda * sj;
      const double* g = p[r];  // [x][u v w T]
      double* s = sL + place[r];
      s[0] = mu * (gas.s43 * g[0] - gas.s23 * g[5] - gas.s23 * g[10]);
      s[RS] = mu * (-gas.s23 * g[0] + gas.s43 * g[5] - gas.s23 * g[10]);
      s[2 * RS] = mu * (-gas.s23 * g[0] - gas.s23 * g[5] + gas.s43 * g[10]);
      s[3 * RS] = mu * (g[4] + g[1]);
      s[4 * RS] = mu * (g[8] + g[2]);
      s[5 * RS] = mu * (g[9] + g[6]);
      s[6 * RS] = la * g[3]; s[7 * RS] = la * g[7]; s[8 * RS] = la * g[11];
    }
  __syncthreads();
  if (!line) return;
  lp.again();
  double f[2][9];
#pragma unroll
  for (int v = 0; v < 9; ++v) {
    f[0][v] = f[1][v] = 0.0;
    if constexpr (GL) {
      f[0][v] = lp.at(sL, 0)[v * RS];
      f[1][v] = lp.at(sL, N)[v * RS];
    } else {
#pragma unroll
      for (int l = 0; l < n; ++l) {
        const double q = lp.at(sL, l)[v * RS];
        f[0][v] += basis[B.L_Minus() + l] * q;
        f[1][v] += basis[B.L_Plus() + l] * q;
      }
    }
  }
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    double ns[3];
    outward<N, AFF>(m, je, id.d, s, own[s], ns);
    const double* T = f[s];  // xx yy zz xy xz yz qx qy qz
    const double a = T[0] * ns[0] + T[3] * ns[1] + T[4] * ns[2], b = T[3] * ns[0] + T[1] * ns[1] + T[5] * ns[2],
                 cc = T[4] * ns[0] + T[5] * ns[1] + T[2] * ns[2];
    double* dst = FG + 4 * (size_t)own[s];
    dst[0] = -a; dst[1] = -b; dst[2] = -cc;
    dst[3] = -(a * uf[s][0] + b * uf[s][1] + cc * uf[s][2]) - (T[6] * ns[0] + T[7] * ns[1] + T[8] * ns[2]);
  }
}

// Kernel B. LAM: the last stage of a step, which also forms CALCTIMESTEP's spectral radii of the new state (a kernel
// of its own over U and the metric terms otherwise, 8 us of a step's 90 at 8^3, N=3).
template <int N, int SOLVER, bool GL, bool AFF, bool LAM>
__global__ __launch_bounds__(S<N>::NT) __attribute__((amdgpu_waves_per_eu(N == 7 ? 2 : 3))) void k_weak_stage(
    const double* U, DevMesh m, const double* __restrict__ basis, const double* __restrict__ FU,
    double* __restrict__ FUnext, const double* __restrict__ FG, Gas gas, double* Ut, RKStage st,
    double* __restrict__ Gout) {
  constexpr int n = S<N>::n, nf = S<N>::nf, np = S<N>::np, NL = S<N>::NL, NT = S<N>::NT, RN = S<N>::RN, RS = S<N>::RS;
  constexpr bool FOLD = GL || AFF;
  using L = LdsW<N, FOLD>;
  __shared__ double sL[L::SIZE];
  const BasisLayout B{n};
  const int e = blockIdx.x, t = N == 7 ? (threadIdx.x + 64 * (e & 3)) % NT : threadIdx.x;
  const bool line = t < NL;
  const LineId id = line_id<N>(line ? t : 0);
  const unsigned own[2] = {m.slotTab[(size_t)6 * nf * e + (id.lsm - 1) * nf + id.ln],
                           m.slotTab[(size_t)6 * nf * e + (id.lsp - 1) * nf + id.ln]};
  const size_t e0 = (size_t)np * e;
  const double* je = AFF ? m.aff + 10 * (size_t)e : nullptr;
  double c[RN][5];
#pragma unroll
  for (int r = 0; r < RN; ++r)
#pragma unroll
    for (int v = 0; v < 5; ++v) c[r][v] = t + r * NT < np ? U[5 * (e0 + t + r * NT) + v] : 1.0;
  double fo[2][5], fb[2][5], gg[2][4];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const size_t o = own[s], b = slot_nbr<N>(own[s]);
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      fo[s][v] = FU[5 * o + v];
      fb[s][v] = FU[5 * b + v];
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) gg[s][v] = 0.5 * (FG[4 * o + v] - FG[4 * b + v]);
  }
  int place[RN];
#pragma unroll
  for (int r = 0; r < RN; ++r) {
    const int nd = t + r * NT < np ? t + r * NT : 0;
    place[r] = pos<N>(nd % n, (nd / n) % n, nd / nf);
    if (t + r * NT < np) {
      const Prim q = cons_to_prim(c[r], gas);
      double* s = sL + place[r];
      s[0] = q.u; s[RS] = q.v; s[2 * RS] = q.w; s[3 * RS] = q.T;
    }
  }
  // the flux through the own face points, outward, times SurfElem: Riemann plus the mean viscous flux
  double jq[2][4], fs[2][5];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const Prim o = cons_to_prim(fo[s], gas), b = cons_to_prim(fb[s], gas);
    jump(o, b, jq[s]);
    const bool master = slot_is_master<N>(own[s]);
    if constexpr (!FOLD) {
      if (line) {
        const size_t sp = slot_side_point<N>(own[s]);
        const double f = (master ? 1.0 : -1.0) * m.SurfElem[sp];
        double* F = sL + L::FACE + (2 * id.d + s) * nf + id.ln;
#pragma unroll
        for (int v = 0; v < 4; ++v) F[v * L::NF] = jq[s][v];
#pragma unroll
        for (int x = 0; x < 3; ++x) F[(4 + x) * L::NF] = m.NormVec[3 * sp + x] * f;
      }
    }
    double ns[3], nv[3];
    outward<N, AFF>(m, je, id.d, s, own[s], ns);
    const double se = sqrt(ns[0] * ns[0] + ns[1] * ns[1] + ns[2] * ns[2]);
    const double ms = master ? 1.0 : -1.0, f = ms / se;
#pragma unroll
    for (int x = 0; x < 3; ++x) nv[x] = ns[x] * f;  // the master's normal
    FaceState l{o.rho, fo[s][4], (fo[s][4] + o.p) * o.srho, o.p, {o.u, o.v, o.w}};
    FaceState r{b.rho, fb[s][4], (fb[s][4] + b.p) * b.srho, b.p, {b.u, b.v, b.w}};
    if (!master) {  // the master's state on the left, so that both elements of a side evaluate the same flux
      const FaceState z = l;
      l = r;
      r = z;
    }
    double F[5];
    riemann_vec<SOLVER, false>(gas, l, r, nv, F);
    fs[s][0] = ms * se * F[0];
#pragma unroll
    for (int v = 0; v < 4; ++v) fs[s][1 + v] = ms * se * F[1 + v] + gg[s][v];
#pragma unroll
    for (int v = 0; v < 5; ++v) now(fs[s][v]);
    __builtin_amdgcn_sched_barrier(0);
  }
  Line<N> lp(id.d, id.a, id.b);
  __syncthreads();
  double p[RN][12];
  gradients<N, GL, AFF, FOLD>(m, basis, je, e0, t, line, id.d, lp, place, jq, sL, p);

  // Euler and viscous fluxes at the nodes, contravariant: f[r][5*d + v]
  double f[RN][15], sj[RN];
  const GasT<double> gt(gas);
#pragma unroll
  for (int r = 0; r < RN; ++r) {
    const int nd = t + r * NT;
    const size_t gid = e0 + (nd < np ? nd : 0);
    double J[9];
    if constexpr (AFF) {
      sj[r] = je[9 + fresh()];
#pragma unroll
      for (int x = 0; x < 9; ++x) J[x] = je[x];
    } else {
      load_metrics<double>(m, gid, J, sj[r]);
    }
#pragma unroll
    for (int x = 0; x < 12; ++x) p[r][x] *= sj[r];
    if (Gout && nd < np) {  // (np, 12, nElems)
#pragma unroll
      for (int x = 0; x < 12; ++x) Gout[nd + (size_t)np * (x + 12 * (size_t)e)] = p[r][x];
    }
    const Prim q = cons_to_prim(c[r], gas);
    double fx[4], fy[4], fz[4];
    diff_flux<double>(gt, q.u, q.v, q.w, p[r], p[r] + 4, p[r] + 8, fx, fy, fz);
    const double Ep = c[r][4] + q.p;
    fx[0] += c[r][1] * q.u + q.p; fx[1] += c[r][1] * q.v; fx[2] += c[r][1] * q.w; fx[3] += Ep * q.u;
    fy[0] += c[r][2] * q.u; fy[1] += c[r][2] * q.v + q.p; fy[2] += c[r][2] * q.w; fy[3] += Ep * q.v;
    fz[0] += c[r][3] * q.u; fz[1] += c[r][3] * q.v; fz[2] += c[r][3] * q.w + q.p; fz[3] += Ep * q.w;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      f[r][5 * d] = J[3 * d] * c[r][1] + J[3 * d + 1] * c[r][2] + J[3 * d + 2] * c[r][3];
#pragma unroll
      for (int v = 0; v < 4; ++v) f[r][5 * d + 1 + v] = J[3 * d] * fx[v] + J[3 * d + 1] * fy[v] + J[3 * d + 2] * fz[v];
    }
#pragma unroll
    for (int x = 0; x < 15; ++x) now(f[r][x]);
  }

  // two variables at a time (the last alone): to the lines, contracted with D_hat, the surface terms added,
  // in place back to the nodes, where the directions are summed
  double sum[RN][5];
#pragma unroll
  for (int h = 0; h < 3; ++h) {
    constexpr int first[3] = {0, 2, 4};
    const int v0 = first[h], nv = h < 2 ? 2 : 1;
#pragma unroll
    for (int r = 0; r < RN; ++r)
      if (t + r * NT < np) {
#pragma unroll
        for (int d = 0; d < 3; ++d)
#pragma unroll
          for (int w = 0; w < nv; ++w) sL[(L::X + 2 * d + w) * RS + place[r]] = f[r][5 * d + v0 + w];
      }
    __syncthreads();
    if (line) {
      const double* DH = basis + B.D_Hat_T() + fresh();
      lp.again();
      double* sX = sL + (L::X + 2 * id.d) * RS;
      double q[2][n];
#pragma unroll
      for (int w = 0; w < nv; ++w)
#pragma unroll
        for (int l = 0; l < n; ++l) q[w][l] = lp.at(sX, l)[w * RS];
#pragma unroll
      for (int i = 0; i < n; ++i)
#pragma unroll
        for (int w = 0; w < nv; ++w) {
          double a = 0.0;
          if constexpr (GL) {
            if (i == 0) a = fs[0][v0 + w] * basis[B.L_HatMinus()];
            if (i == N) a = fs[1][v0 + w] * basis[B.L_HatPlus() + N];
          } else {
            a = fs[0][v0 + w] * basis[B.L_HatMinus() + i] + fs[1][v0 + w] * basis[B.L_HatPlus() + i];
          }
#pragma unroll
          for (int l = 0; l < n; ++l) a += DH[l + n * i] * q[w][l];
          lp.at(sX, i)[w * RS] = a;
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RN; ++r)
#pragma unroll
      for (int w = 0; w < nv; ++w) {
        const double* s = sL + (L::X + w) * RS + place[r];
        sum[r][v0 + w] = s[0] + s[2 * RS] + s[4 * RS];
      }
  }
  double lam[6] = {0, 0, 0, 0, 0, 0};
  int nan_rho = 0;
  // Ut = -Ut*sJ, the register update, and the new state in rows 0..3 and 9 for its face values
#pragma unroll
  for (int r = 0; r < RN; ++r) {
    const int nd = t + r * NT;
    if (nd >= np) continue;
    const size_t o = 5 * (e0 + nd);
    if (st.mode == 0) {
#pragma unroll
      for (int v = 0; v < 5; ++v) Ut[o + v] = -sum[r][v] * sj[r];
      continue;
    }
    double rn[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      const double ut = -sum[r][v] * sj[r];
      rn[v] = st.mode == 1 ? ut : st.R[o + v] * st.minusA + ut;
    }
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      st.R[o + v] = rn[v];
      c[r][v] += rn[v] * st.b_dt;
      st.U[o + v] = c[r][v];
      sL[(v < 4 ? v : 9) * RS + place[r]] = c[r][v];
    }
    if constexpr (LAM) {
      double ln6[6];
      int nr;
      if constexpr (AFF) dt_node_lambda(c[r], gas, je[9], je, je + 3, je + 6, ln6, nr);
      else dt_node_lambda(c[r], gas, sj[r], m.Mf + 3 * (e0 + nd), m.Mg + 3 * (e0 + nd), m.Mh + 3 * (e0 + nd), ln6, nr);
      nan_rho |= nr;
#pragma unroll
      for (int x = 0; x < 6; ++x) lam[x] = (ln6[x] > lam[x] || ln6[x] != ln6[x]) ? ln6[x] : lam[x];
    }
  }
  if (st.mode == 0) return;
  if constexpr (LAM) {
    __shared__ double red[6 * (NT / 64)];
    __shared__ int flag[NT / 64];
    double mx[6];
    int nanr = 0;
    block_lambda_max<NT>(lam, nan_rho, red, flag, threadIdx.x, mx, nanr);
    if (threadIdx.x == 0) {
      st.lamSum[2 * e] = mx[0] + mx[1] + mx[2];
      st.lamSum[2 * e + 1] = mx[3] + mx[4] + mx[5];
      st.lamNan[e] = nanr;
    }
  }
  __syncthreads();
  if (!line) return;
  lp.again();
  double fn[2][5] = {{0, 0, 0, 0, 0}, {0, 0, 0, 0, 0}};
#pragma unroll
  for (int v = 0; v < 5; ++v) {
    const int row = v < 4 ? v : 9;
    if constexpr (GL) {
      fn[0][v] = lp.at(sL, 0)[row * RS];
      fn[1][v] = lp.at(sL, N)[row * RS];
    } else {
#pragma unroll
      for (int l = 0; l < n; ++l) {
        const double q = lp.at(sL, l)[row * RS];
        fn[0][v] += basis[B.L_Minus() + l] * q;
        fn[1][v] += basis[B.L_Plus() + l] * q;
      }
    }
  }
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int v = 0; v < 5; ++v) FUnext[5 * (size_t)own[s] + v] = fn[s][v];
}

struct Scope {
  KernelTimer* t;
  int id;
  hipStream_t s;
  Scope(KernelTimer* t_, int id_, hipStream_t s_) : t(t_), id(id_), s(s_) { if (t) t->mark(id, true, s); }
  ~Scope() { if (t) t->mark(id, false, s); }
};

template <int N, bool GL, bool AFF>
hipError_t weak_n(const DevMesh& m, const FusedWork& w, const Gas& gas, int riemann, const double* U, double* Ut,
                  const RKStage& st, bool faces_fresh, int cur, double* G, hipStream_t s, KernelTimer* tm) {
  const dim3 g(m.nElems), b(S<N>::NT);
  double* FU = w.FU[cur];
  double* FG = (double*)w.FG;
  if (!faces_fresh) {
    Scope sc(tm, K_WEAK_FACES, s);
    hipLaunchKernelGGL((k_weak_faces<N, GL>), g, b, 0, s, U, m, m.basis, FU);
  }
  {
    Scope sc(tm, K_WEAK_VISC, s);
    hipLaunchKernelGGL((k_weak_visc<N, GL, AFF>), g, b, 0, s, U, m, m.basis, FU, FG, gas);
  }
  {
    Scope sc(tm, K_WEAK_STAGE, s);
#define FXG_LAUNCH(SOLV)                                                                                               \
  if (st.lamSum)                                                                                                       \
    hipLaunchKernelGGL((k_weak_stage<N, SOLV, GL, AFF, true>), g, b, 0, s, U, m, m.basis, FU, w.FU[1 - cur], FG, gas, \
                       Ut, st, G);                                                                                     \
  else                                                                                                                 \
    hipLaunchKernelGGL((k_weak_stage<N, SOLV, GL, AFF, false>), g, b, 0, s, U, m, m.basis, FU, w.FU[1 - cur], FG, gas, \
                       Ut, st, G)
    if (riemann == 1) { FXG_LAUNCH(1); }
    else if (riemann == 3) { FXG_LAUNCH(3); }
    else { FXG_LAUNCH(33); }
#undef FXG_LAUNCH
  }
  return hipGetLastError();
}

template <int N>
hipError_t weak_case(const DevMesh& m, const FusedWork& w, const Gas& gas, int nodeType, int riemann, const double* U,
                     double* Ut, const RKStage& st, bool fresh, int cur, double* G, hipStream_t s, KernelTimer* tm) {
  if (nodeType == 2)
    return m.aff ? weak_n<N, true, true>(m, w, gas, riemann, U, Ut, st, fresh, cur, G, s, tm)
                 : weak_n<N, true, false>(m, w, gas, riemann, U, Ut, st, fresh, cur, G, s, tm);
  return m.aff ? weak_n<N, false, true>(m, w, gas, riemann, U, Ut, st, fresh, cur, G, s, tm)
               : weak_n<N, false, false>(m, w, gas, riemann, U, Ut, st, fresh, cur, G, s, tm);
}

}  // namespace

hipError_t launch_rhs_weak(const DevMesh& m, const FusedWork& w, const Gas& gas, int nodeType, int riemann,
                           const double* U, double* Ut, const RKStage& st, bool faces_fresh, int cur, double* G,
                           hipStream_t s, KernelTimer* tm) {
  switch (m.N) {
#define FXG_CASE(NN) \
  case NN: return weak_case<NN>(m, w, gas, nodeType, riemann, U, Ut, st, faces_fresh, cur, G, s, tm);
    FXG_CASE(2) FXG_CASE(3) FXG_CASE(4) FXG_CASE(5) FXG_CASE(6) FXG_CASE(7)
#undef FXG_CASE
    default: return hipErrorInvalidValue;
  }
}

// Side slots are 32-bit, as on the split form's path. N = 1 has too few nodes on a line to gain, FP32-bulk keeps the
// order of its sums, and boundary sides have no form of these kernels yet (fxg_bcface.h holds what one would need).
bool weak_supported(int N, int split, int fp32, int nBC, long long nSides) {
  return !split && !fp32 && nBC == 0 && N >= 2 && N <= 7 && nSides * 2LL * (N + 1) * (N + 1) < (1LL << 32);
}

}  // namespace fxg
