// Kernel A of the fused Gauss-Lobatto split-form stage (the rest is in fxg_fused.hip): for each
// element, the BR1 gradients at its boundary nodes and, for each of its six faces, the viscous
// normal flux f_v . (n SurfElem) seen from that element (4 values per face point, momentum and
// energy) into the side array FG (lifting_br1.t90:48-181, flux.f90:149-241). A translation unit
// of its own, so that its code does not change the register allocation of k_dg_fused.
#include "fxg_bcface.h"
#include "fxg_line.h"

namespace fxg {
namespace {

// FP32-bulk, one lane per boundary node. U is converted from global memory directly and the kernel is
// held to 64 VGPRs (18 KB: four workgroups per CU). On meshes with boundary sides (BC) it also keeps the
// gradients of the boundary face points for k_bc_visc.
// The metric terms are read as the FP32 values that it uses (32^3, N=7: 0.42 ms with FP64 rows, 0.36 now).
// FIRST: no stage has left the face states of U (a right-hand side alone, the first stage of a step on
// a caller's state): the neighbours' states come from their nodes in U and the own face states are
// written to FU for the stage kernel. Replaces a pass of its own over U (k_faces_of, 64 bytes per node at
// N=7 and one launch; right-hand side at 32^3, N=7, FP64: 1.38 -> 1.30 ms).
template <int N, class RF, bool BC, bool FIRST>
__global__ __launch_bounds__(D<N>::NT)
__attribute__((amdgpu_waves_per_eu(N == 7 ? 8 : 6))) void k_visc_faces(
    const double* __restrict__ U, DevMesh m, const RF* __restrict__ Jsoa, double* __restrict__ FU,
    RF* __restrict__ FG, Gas gas, RF* __restrict__ gBC) {
  constexpr int n = D<N>::n, np = D<N>::np, NT = D<N>::NT, NF = D<N>::NF;
  __shared__ RF sP[4 * np];        // u, v, w, T
  __shared__ RF sNb[4 * NF];       // neighbour u, v, w, T per own face point
  __shared__ unsigned sIdx[NF];
  __shared__ double sB[3 * n * n + 4 * n];
  const int e = blockIdx.x, t = threadIdx.x;
  const double* Ue = U + (size_t)5 * np * e;
  constexpr int NB = Bnd<N>::NB;         // boundary nodes
  constexpr int NBAS = 3 * n * n + 4 * n;
  static_assert(NBAS <= NT, "one basis entry per lane");
  constexpr int RS = (NF + NT - 1) / NT;  // own face points per lane
  // Every global load of the staging is issued before the first wait, instead of one wait per
  // loop of loads: the side slots first (the neighbour states depend on them), then U and the basis.
  unsigned own[RS], nbr[RS];
#pragma unroll
  for (int r = 0; r < RS; ++r) {
    const int x = t + r * NT;
    own[r] = x < NF ? face_slot_tab<N>(m, e, x) : 0u;
    nbr[r] = FIRST && x < NF ? m.nbNode[(size_t)NF * e + x] : 0u;
  }
  double ul[5];
#pragma unroll
  for (int r = 0; r < 5; ++r) ul[r] = t < np ? Ue[5 * t + r] : 1.0;
  const double bas = t < NBAS ? m.basis[t] : 0.0;
  double cn[RS][5];
#pragma unroll
  for (int r = 0; r < RS; ++r) {
    const double* c = FIRST ? U + 5 * (size_t)nbr[r] : FU + 5 * (size_t)slot_nbr<N>(own[r]);
#pragma unroll
    for (int v = 0; v < 5; ++v) cn[r][v] = t + r * NT < NF ? c[v] : 1.0;
  }
  if (t < np) {
    const Prim q = cons_to_prim(ul, gas);
    sP[t] = q.u; sP[np + t] = q.v; sP[2 * np + t] = q.w; sP[3 * np + t] = q.T;
  }
  if (t < NBAS) sB[t] = bas;
#pragma unroll
  for (int r = 0; r < RS; ++r) {
    const int x = t + r * NT;
    if (x < NF) {
      sIdx[x] = own[r];
      const Prim q = cons_to_prim(cn[r], gas);
      sNb[x] = q.u; sNb[NF + x] = q.v; sNb[2 * NF + x] = q.w; sNb[3 * NF + x] = q.T;
    }
  }
  __syncthreads();
  if constexpr (FIRST) {
#pragma unroll
    for (int r = 0; r < RS; ++r) {
      const int x = t + r * NT;
      if (x < NF) {
        const int ls = x / (n * n) + 1, ab = x - (ls - 1) * n * n;
        const int id = vidx<N>(ls, ab % n, ab / n);
        const double* c = Ue + 5 * id;
#pragma unroll
        for (int v = 0; v < 5; ++v) FU[5 * (size_t)own[r] + v] = c[v];
      }
    }
  }
  // one lane per boundary node, in boundary-rank order (the Jsoa rows): lanes 0..NB-1, so the
  // waves beyond NB/64 end here instead of idling through the lifting
  if (t >= NB) return;
  int i, j, k;
  bnd_node<N>(t, i, j, k);
  const int nd = i + n * (j + n * k);
  const int sides = node_sides<N>(i, j, k);
  const GasT<RF> gt(gas);
  // metric terms of the boundary nodes only, rows of NB per element (Jsoa layout)
  const RF* Je = Jsoa + (size_t)10 * NB * e;
  RF Ja[9], sj;
#pragma unroll
  for (int r = 0; r < 9; ++r) Ja[r] = Je[r * NB + t];
  sj = Je[9 * NB + t];
  RF g[12];
  lift_node<N, RF>(nd, sP, sB, sNb, Ja, sj, g);
  RF fx[4], fy[4], fz[4];
  diff_flux<RF>(gt, (RF)sP[nd], (RF)sP[np + nd], (RF)sP[2 * np + nd], g, g + 4, g + 8, fx, fy, fz);
#pragma unroll 1
  for (int ls = 1; ls <= 6; ++ls) {
    if (!(sides & (1 << (ls - 1)))) continue;
    const int dir = dir_of(ls);
    const RF s = (RF)normal_sign(ls);
    const RF n0 = Ja[3 * dir] * s, n1 = Ja[3 * dir + 1] * s, n2 = Ja[3 * dir + 2] * s;
    const unsigned own = sIdx[face_point<N>(ls, i, j, k)];
    RF* dst = FG + 4 * (size_t)own;
#pragma unroll
    for (int c = 0; c < 4; ++c) dst[c] = fx[c] * n0 + fy[c] * n1 + fz[c] * n2;
    if constexpr (BC) {
      // a boundary side: keep the gradients at this face point for k_bc_visc
      const int side = (int)(own / (2u * (unsigned)(n * n)));
      if (side < m.nBC) {
        RF* gb = gBC + 12 * slot_side_point<N>(own);
#pragma unroll
        for (int c = 0; c < 12; ++c) gb[c] = g[c];
      }
    }
  }
}

// FP64: the same with one lane per line of nodes (fxg_line.h), as in the stage kernel. The form above, one lane
// per boundary node, reads 120 values per boundary node from LDS and leaves two of five lanes idle; here a
// line is read once per variable, the gradients come together in the node phase, and the ends of the lines are
// the face points. 10 LDS rows: four workgroups of four waves per CU at N=7. Parallelepipeds: 32^3, N=7
// 0.42 -> 0.33 ms (94 bytes per node at 4.8 TB/s, the copy rate), N=5, 24^3 0.108 -> 0.079, N=3, 32^3 0.089 ->
// 0.068; general: N=7, 32^3 0.48 -> 0.44, N=5, 24^3 0.129 -> 0.105.
// LDS rows: 0 u, 1 v, 2 w, 3 T; 4..9 exchange between line and node phases (two variables in three directions).
template <int N, bool BC, bool AFF, bool FIRST>
__global__ __launch_bounds__(S<N>::NT) __attribute__((amdgpu_waves_per_eu(3))) void k_visc_lines(
    const double* __restrict__ U, DevMesh m, const double* __restrict__ basis, const double* __restrict__ Jsoa,
    double* __restrict__ FU, double* __restrict__ FG, Gas gas, double* __restrict__ gBC,
    const double* __restrict__ bcP) {
  constexpr int n = S<N>::n, nf = S<N>::nf, np = S<N>::np, NL = S<N>::NL, NT = S<N>::NT, RN = S<N>::RN, RS = S<N>::RS;
  constexpr int X = 4, NF = 6 * nf;
  __shared__ double sL[10 * RS];
  const BasisLayout B{n};
  const int e = blockIdx.x, t = N == 7 ? (threadIdx.x + 64 * (e & 3)) % NT : threadIdx.x;
  const bool line = t < NL;
  const int tl = line ? t : 0;
  const int d = tl / nf, ln = tl - d * nf, la = ln % n, lb = ln / n;
  const size_t fp0 = (size_t)NF * e + ((d == 0 ? 5 : (d == 1 ? 2 : 1)) - 1) * nf + ln;
  const size_t fp1 = (size_t)NF * e + ((d == 0 ? 3 : (d == 1 ? 4 : 6)) - 1) * nf + ln;
  const unsigned own0 = m.slotTab[fp0], own1 = m.slotTab[fp1];
  const size_t e0 = (size_t)np * e;
  const double* je = AFF ? m.aff + 10 * (size_t)e : nullptr;
  double c[RN][5];
#pragma unroll
  for (int r = 0; r < RN; ++r)
#pragma unroll
    for (int v = 0; v < 5; ++v) c[r][v] = t + r * NT < np ? U[5 * (e0 + t + r * NT) + v] : 1.0;
  double nb[2][5];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const double* b = FIRST ? U + 5 * (size_t)m.nbNode[s ? fp1 : fp0] : FU + 5 * (size_t)slot_nbr<N>(s ? own1 : own0);
#pragma unroll
    for (int v = 0; v < 5; ++v) nb[s][v] = b[v];
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
      if constexpr (FIRST) {  // the state itself, to the ends of the lines
#pragma unroll
        for (int v = 0; v < 5; ++v) s[(X + v) * RS] = c[r][v];
      }
    }
  }
  const Prim q0 = cons_to_prim(nb[0], gas), q1 = cons_to_prim(nb[1], gas);
  Line<N> lp(d, la, lb);
  // the element's boundary sides, one bit per local side: uniform, so that interior elements skip what follows for
  // them (cavity box 32^3, N=7: 0.494 -> 0.457 ms)
  int walls = 0;
  if constexpr (BC) {
#pragma unroll
    for (int ls = 1; ls <= 6; ++ls) walls |= (m.E2S[2 * (ls - 1) + 12 * (size_t)e] <= m.nBC ? 1 : 0) << (ls - 1);
  }
  __syncthreads();
  double jq[2][4];  // BR1 jumps with their sign and weight
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const double* o = lp.at(sL, s ? N : 0);
    const Prim& q = s ? q1 : q0;
    const double h = s ? 0.5 * basis[B.L_HatPlus() + N] : -0.5 * basis[B.L_HatMinus()];
    jq[s][0] = h * (q.u - o[0]); jq[s][1] = h * (q.v - o[RS]); jq[s][2] = h * (q.w - o[2 * RS]);
    jq[s][3] = h * (q.T - o[3 * RS]);
  }
  if constexpr (FIRST) {  // the own face states, for the stage kernel
    if (line) {
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const double* o = lp.at(sL, s ? N : 0) + X * RS;
        double* dst = FU + 5 * (size_t)(s ? own1 : own0);
#pragma unroll
        for (int v = 0; v < 5; ++v) dst[v] = o[v * RS];
      }
    }
    __syncthreads();
  }
  double g[RN][12];  // reference derivatives, then contravariant viscous fluxes: [d][u v w T]
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    if (line) {
      const double* DT = basis + B.D_T() + fresh();
      lp.again();
      double* sX = sL + (X + 2 * d) * RS;
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
        for (int w = 0; w < 2; ++w) g[r][4 * x + 2 * h + w] = sL[(X + 2 * x + w) * RS + place[r]];
    if (h == 0) __syncthreads();
  }
  const GasT<double> gt(gas);
#pragma unroll
  for (int r = 0; r < RN; ++r) {
    const int nd = t + r * NT < np ? t + r * NT : 0;
    double Ja[9], sj;
    if constexpr (AFF) {
      const double* jn = je + fresh();
#pragma unroll
      for (int x = 0; x < 9; ++x) Ja[x] = jn[x];
      sj = jn[9];
    } else {
      // those of the boundary nodes, packed; the interior nodes' fluxes are not needed
      constexpr int NB = Bnd<N>::NB;
      const int i = nd % n, j = (nd / n) % n, k = nd / nf;
      const bool bn = node_sides<N>(i, j, k) != 0;
      const double* Je = Jsoa + (size_t)10 * NB * e + (bn ? bnd_rank<N>(i, j, k) : 0);
#pragma unroll
      for (int x = 0; x < 9; ++x) Ja[x] = bn ? Je[x * NB] : 0.0;
      sj = bn ? Je[9 * NB] : 0.0;
    }
    double p[12];
#pragma unroll
    for (int x = 0; x < 3; ++x)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        p[4 * x + v] = (Ja[x] * g[r][v] + Ja[3 + x] * g[r][4 + v] + Ja[6 + x] * g[r][8 + v]) * sj;
    if constexpr (BC) {
      // boundary sides: the gradients at their face points, for the ends of the lines below
      if (walls && t + r * NT < np) {
        const int i = nd % n, j = (nd / n) % n, k = nd / nf, sides = node_sides<N>(i, j, k) & walls;
#pragma unroll 1
        for (int ls = 1; ls <= 6; ++ls) {
          if (!(sides & (1 << (ls - 1)))) continue;
          const unsigned own = m.slotTab[(size_t)NF * e + face_point<N>(ls, i, j, k)];
          double* gb = gBC + 12 * slot_side_point<N>(own);
#pragma unroll
          for (int x = 0; x < 12; ++x) gb[x] = p[x];
        }
      }
    }
    double fx[4], fy[4], fz[4];
    const double* s = sL + place[r];
    diff_flux<double>(gt, s[0], s[RS], s[2 * RS], p, p + 4, p + 8, fx, fy, fz);
#pragma unroll
    for (int x = 0; x < 3; ++x)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        g[r][4 * x + v] = Ja[3 * x] * fx[v] + Ja[3 * x + 1] * fy[v] + Ja[3 * x + 2] * fz[v];
#pragma unroll
    for (int x = 0; x < 12; ++x) now(g[r][x]);
  }
  // to the ends of the lines: n SurfElem there is NormalSign Ja^d
  double f[2][4];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int r = 0; r < RN; ++r)
      if (t + r * NT < np) {
#pragma unroll
        for (int x = 0; x < 3; ++x)
#pragma unroll
          for (int w = 0; w < 2; ++w) sL[(X + 2 * x + w) * RS + place[r]] = g[r][4 * x + 2 * h + w];
      }
    __syncthreads();
    const double* sX = sL + (X + 2 * d) * RS;
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      f[0][2 * h + w] = -lp.at(const_cast<double*>(sX), 0)[w * RS];
      f[1][2 * h + w] = lp.at(const_cast<double*>(sX), N)[w * RS];
    }
    if (h == 0) __syncthreads();
  }
  if (!line) return;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    FG[4 * (size_t)own0 + v] = f[0][v];
    FG[4 * (size_t)own1 + v] = f[1][v];
  }
  if constexpr (BC) {
    // the outer slots of boundary sides (a kernel of its own over the boundary points otherwise); the gradients
    // were stored by this workgroup, before the barriers above
    if (!walls) return;
#pragma unroll 1
    for (int s = 0; s < 2; ++s) {
      const unsigned own = s ? own1 : own0;
      const int side = (int)(own / (2u * (unsigned)nf));
      if (side >= m.nBC) continue;
      const size_t fp = slot_side_point<N>(own);
      double q[12], fi[4];
#pragma unroll
      for (int x = 0; x < 12; ++x) q[x] = gBC[12 * fp + x];
#pragma unroll
      for (int x = 0; x < 4; ++x) fi[x] = s ? f[1][x] : f[0][x];
      bc_visc_point<double>(m, FU + 5 * (size_t)own, q, fi, FG + 4 * ((size_t)own + nf), bcP, gas, fp, side);
    }
  }
}

// FP32-bulk: one lane per boundary side point, after k_visc_faces (k_visc_lines forms these fluxes itself).
__global__ __launch_bounds__(256) void k_bc_visc(DevMesh m, const double* __restrict__ FU, const float* __restrict__ gBC,
                                               float* __restrict__ FG, const double* __restrict__ bcP, Gas gas, int nf,
                                               int nPts) {
  const int fp = blockIdx.x * blockDim.x + threadIdx.x;
  if (fp >= nPts) return;
  const int side = fp / nf, pq = fp - side * nf;
  const size_t in = ((size_t)side * 2) * nf + pq, out = in + nf;
  float q[12];
#pragma unroll
  for (int c = 0; c < 12; ++c) q[c] = gBC[12 * (size_t)fp + c];
  bc_visc_point<float>(m, FU + 5 * in, q, FG + 4 * in, FG + 4 * out, bcP, gas, fp, side);
}

// One lane per boundary side point: the outer slots from the inner face states (in FP64 a stage leaves those of its
// new state, and this kernel serves the first stage of a state without face states).
__global__ __launch_bounds__(256) void k_bc_ghost(DevMesh m, double* __restrict__ FU, double* __restrict__ bcP,
                                                Gas gas, int nf, int nPts) {
  const int fp = blockIdx.x * blockDim.x + threadIdx.x;
  if (fp >= nPts) return;
  const int side = fp / nf, pq = fp - side * nf;
  const size_t in = ((size_t)side * 2) * nf + pq;
  bc_ghost_point(m, FU + 5 * in, FU + 5 * (in + nf), bcP, gas, fp, side);
}

}  // namespace

hipError_t launch_bc_ghost(const DevMesh& m, double* FU, double* bcP, const Gas& gas, hipStream_t s) {
  const int nf = (m.N + 1) * (m.N + 1), nPts = m.nBC * nf;
  if (nPts == 0) return hipSuccess;
  hipLaunchKernelGGL(k_bc_ghost, dim3((nPts + 255) / 256), dim3(256), 0, s, m, FU, bcP, gas, nf, nPts);
  return hipGetLastError();
}

hipError_t launch_visc_faces(const DevMesh& m, bool fp32, bool faces_fresh, const double* U, const void* Jsoa,
                             double* FU, void* FG, const Gas& gas, void* gBC, const double* bcP, hipStream_t s) {
  const bool bc = m.nBC > 0;
  if (!faces_fresh && !m.nbNode) return hipErrorInvalidValue;
  switch (m.N) {
#define FXG_LAUNCH2(NN, BC, AFF, FIRST)                                                                            \
  do {                                                                                                             \
    if (fp32)                                                                                                      \
      hipLaunchKernelGGL((k_visc_faces<NN, float, BC, FIRST>), dim3(m.nElems), dim3(D<NN>::NT), 0, s, U, m,    \
                         (const float*)Jsoa, FU, (float*)FG, gas, (float*)gBC);                                                  \
    else                                                                                                           \
      hipLaunchKernelGGL((k_visc_lines<NN, BC, AFF, FIRST>), dim3(m.nElems), dim3(S<NN>::NT), 0, s, U, m, m.basis, \
                         (const double*)Jsoa, FU, (double*)FG, gas, (double*)gBC, bcP);                                                      \
  } while (0)
#define FXG_CASE(NN)                                                                                               \
  case NN:                                                                                                         \
    if (bc) { if (m.aff) FXG_LAUNCH2(NN, true, true, false); else FXG_LAUNCH2(NN, true, false, false); }            \
    else if (faces_fresh) { if (m.aff) FXG_LAUNCH2(NN, false, true, false); else FXG_LAUNCH2(NN, false, false, false); } \
    else { if (m.aff) FXG_LAUNCH2(NN, false, true, true); else FXG_LAUNCH2(NN, false, false, true); }              \
    break;
    FXG_CASE(2) FXG_CASE(3) FXG_CASE(4) FXG_CASE(5) FXG_CASE(6) FXG_CASE(7)
#undef FXG_CASE
#undef FXG_LAUNCH2
    default: return hipErrorInvalidValue;
  }
  if (bc && fp32) {
    const int nf = (m.N + 1) * (m.N + 1), nPts = m.nBC * nf;
    hipLaunchKernelGGL(k_bc_visc, dim3((nPts + 255) / 256), dim3(256), 0, s, m, FU, (const float*)gBC, (float*)FG, bcP,
                       gas, nf, nPts);
  }
  return hipGetLastError();
}

}  // namespace fxg
