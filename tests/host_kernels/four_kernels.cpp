// The four-kernel path on one periodic element, one right-hand side and one two-stage step per argument "N": run
// under AddressSanitizer, which reports any access outside an LDS or device array.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>

namespace {  // internal linkage: only then are the LDS arrays of kernel templates given guard zones
#include "fxg_kernels.hip"

namespace fxg {
template <class T>
T* array(size_t n, T v) {  // exactly n entries
  T* p = (T*)std::malloc(n * sizeof(T));
  std::fill(p, p + n, v);
  return p;
}

int run(int N, int nodeType, int split, int fp32) {
  const int n = N + 1, nf = n * n, np = nf * n, S = 3;
  DevMesh m{};
  m.N = N; m.nElems = 1; m.nSides = S;
  // side 1: zeta, 2: eta, 3: xi; the plus sides are the masters
  int* E2S = array<int>(12, 0);
  const int side[6] = {1, 2, 3, 2, 3, 1}, flip[6] = {1, 2, 0, 0, 1, 0};
  for (int ls = 0; ls < 6; ++ls) { E2S[2 * ls] = side[ls]; E2S[2 * ls + 1] = flip[ls]; }
  int* map = array<int>(2 * nf * 30, 0);
  for (int x = 0; x < nf * 30; ++x) { map[2 * x] = x % n; map[2 * x + 1] = x / n % n; }
  m.E2S = E2S; m.s2v2 = map; m.v2s2 = map;
  double *I[3], *NV = array(3 * (size_t)nf * S, 0.0);
  for (int d = 0; d < 3; ++d) {
    I[d] = array(3 * (size_t)np, 0.0);
    for (int x = 0; x < np; ++x) I[d][3 * x + d] = 1.0;
  }
  for (int x = 0; x < nf * S; ++x) NV[3 * x + x / nf] = 1.0;
  m.Mf = I[0]; m.Mg = I[1]; m.Mh = I[2]; m.sJ = array((size_t)np, 1.0);
  m.NormVec = m.TangVec1 = m.TangVec2 = NV;
  m.SurfElem = array((size_t)nf * S, 1.0);
  const BasisLayout B{n};
  m.basis = array((size_t)B.size(), 0.1);
  const size_t g = fp32 ? 4 : 8;
  DevWork w{};
  w.Uf_m = array(5 * (size_t)nf * S, 1.0);
  w.Uf_s = array(5 * (size_t)nf * S, 1.0);
  w.G = std::calloc(12 * (size_t)np, g);
  w.Gf_m = std::calloc(12 * (size_t)nf * S, g);
  w.Gf_s = std::calloc(12 * (size_t)nf * S, g);
  w.Flux = array(5 * (size_t)nf * S, 0.0);
  double *U = array(5 * (size_t)np, 0.0), *R = array(5 * (size_t)np, 0.0), *Ut = array(5 * (size_t)np, 0.0);
  for (int x = 0; x < np; ++x) { U[5 * x] = 1.0; U[5 * x + 4] = 2.5; }
  const Gas gas{1.4, 0.4, 2.5, 1.0, 1.0, 0.0, 0.0, 4.0 / 3.0, 2.0 / 3.0, 1.4 / 0.72};
  hipError_t e = launch_rhs(m, w, gas, nodeType, split, 1, fp32, U, Ut, RKStage{0, 0.0, 0.0, nullptr, nullptr}, false,
                            nullptr, nullptr);
  for (int st = 0; st < 2 && !e; ++st)
    e = launch_rhs(m, w, gas, nodeType, split, 1, fp32, U, nullptr, RKStage{1 + st, 0.0, 0.0, U, R}, st > 0, nullptr, nullptr);
  return e;
}
}  // namespace fxg
}  // namespace

int main(int argc, char** argv) {
  if (argc != 2) return 2;
  const int N = std::atoi(argv[1]);
  for (int fp32 = 0; fp32 < 2; ++fp32)
    for (int form = 0; form < 3; ++form) {  // Gauss weak, Gauss-Lobatto weak, Gauss-Lobatto split
      std::printf("N=%d form %d %s\n", N, form, fp32 ? "float" : "double");
      std::fflush(stdout);
      if (fxg::run(N, form ? 2 : 1, form == 2, fp32)) return 1;
    }
}
