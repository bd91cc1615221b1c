// Just enough of the HIP runtime to compile the element kernels as host code, where the sanitizers see every
// access: a launch runs its workgroups one after the other, each lane a thread, LDS arrays static variables.
#pragma once
#include <algorithm>
#include <barrier>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <memory>
#include <thread>
#include <vector>

using std::sqrt;
using std::fabs;
using std::fmax;
using std::fmin;

typedef int hipError_t;
typedef void* hipStream_t;
constexpr hipError_t hipSuccess = 0, hipErrorInvalidValue = 1;
inline hipError_t hipGetLastError() { return hipSuccess; }

struct dim3 {
  unsigned x, y, z;
  dim3(unsigned a = 1, unsigned b = 1, unsigned c = 1) : x(a), y(b), z(c) {}
};

namespace host {
struct Group {
  std::barrier<> all;
  std::vector<std::unique_ptr<std::barrier<>>> wave;
  std::vector<double> slot;
  explicit Group(int n) : all(n), slot(n) {
    for (int w = 0; w < n; w += 64) wave.emplace_back(new std::barrier<>(std::min(64, n - w)));
  }
};
inline thread_local dim3 tid, bid, bdim, gdim;
inline Group* group;
// the value of lane `from` of the wave
inline double shuffle(double x, unsigned from) {
  auto& b = *group->wave[tid.x / 64];
  group->slot[tid.x] = x;
  b.arrive_and_wait();
  const unsigned base = tid.x / 64 * 64;
  const double y = base + from < std::min(base + 64, bdim.x) ? group->slot[base + from] : x;
  b.arrive_and_wait();
  return y;
}
template <class F>
void launch(dim3 grid, dim3 block, F f) {
  for (unsigned g = 0; g < grid.x; ++g) {
    Group gr((int)block.x);
    group = &gr;
    std::vector<std::thread> lanes;
    for (unsigned t = 0; t < block.x; ++t)
      lanes.emplace_back([=, &gr] {
        tid = dim3(t, 0, 0); bid = dim3(g, 0, 0); bdim = block; gdim = grid;
        f();
        gr.all.arrive_and_drop();  // a lane that has ended is no longer waited for
        gr.wave[t / 64]->arrive_and_drop();
      });
    for (auto& l : lanes) l.join();
  }
}
}  // namespace host

#define threadIdx host::tid
#define blockIdx host::bid
#define blockDim host::bdim
#define gridDim host::gdim
#define __global__
#define __device__
#define __host__
#define __shared__ static
#define __align__(x) alignas(x)
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __builtin_amdgcn_sched_barrier(x)
#define hipLaunchKernelGGL(k, grid, block, lds, stream, ...) host::launch(grid, block, [=] { (k)(__VA_ARGS__); })
inline void __syncthreads() { host::group->all.arrive_and_wait(); }
inline double __shfl_down(double x, int off, int) { return host::shuffle(x, (host::tid.x & 63) + off); }
inline int __shfl_down(int x, int off, int) { return (int)host::shuffle(x, (host::tid.x & 63) + off); }
inline unsigned long long __ballot(int p) {
  unsigned long long m = 0;
  for (unsigned l = 0; l < 64; ++l)
    if ((host::tid.x / 64) * 64 + l < host::bdim.x && host::shuffle(p ? 1.0 : 0.0, l) != 0.0) m |= 1ull << l;
  return m;
}
// register hints of the kernels (empty asm statements) mean nothing here
#define asm
#define volatile(...)
