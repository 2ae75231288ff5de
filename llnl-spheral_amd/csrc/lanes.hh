// Several lanes to a node, for small node sets.
//
// One lane to a node leaves the chip idle on a small node set: 32^3 nodes are
// half a wavefront per SIMD, and a kernel takes as long as one row does.  With L
// consecutive lanes to a node, L entries of a row are evaluated side by side and
// the sums still run in row order, through LDS; a lane past the row's end
// contributes -0, which changes no sum.
#pragma once
#include <cstdint>
#include <type_traits>
#include <hip/hip_runtime.h>

namespace sphgpu {

// LDS traffic between lanes of one wavefront needs no barrier, only the order.
__device__ __forceinline__ void waveLdsOrder() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// acc plus the L terms of the node's lanes, in lane order; `before` is added in
// front of the term of lane `first` (none when first >= L).  Every lane gets the
// result.  buf: one double per lane of the wavefront.
template <int L>
__device__ __forceinline__ double addInOrder(double acc, double term, double* buf, int first = 64, double before = 0.0) {
  const int lane = threadIdx.x & 63;
  buf[lane] = term;
  waveLdsOrder();
  const double2* p = reinterpret_cast<const double2*>(buf + (lane & ~(L - 1)));
#pragma unroll
  for (int e = 0; e < L; e += 2) {
    const double2 v = p[e / 2];
    acc += e == first ? before : -0.0;
    acc += v.x;
    acc += e + 1 == first ? before : -0.0;
    acc += v.y;
  }
  waveLdsOrder();
  return acc;
}
// Place among the node's L lanes of the first one with `c` (64: none).
template <int L> __device__ __forceinline__ int firstLane(bool c) {
  const unsigned long long m = (__ballot(c) >> (threadIdx.x & 63 & ~(L - 1))) & ((1ull << L) - 1ull);
  return m ? __builtin_ctzll(m) : 64;
}

// Lanes to a node.  The lines lie where the measured times cross (reference order
// pair pass, one / 8 / 16 lanes, us; the other passes cross at or above them):
//   3-D  1.7 k nodes 189 / 50 / 30, 14 k 195 / 71 / 72, 33 k 206 / 131 / 132, 64 k 225 / 231 / 251
//   2-D  1 k 47 / 16 / 11, 10 k 48 / 20 / 17, 22 k 50 / 26 / 30, 48 k 53 / 49 / 53, 102 k 84 / 102 / 108
//   1-D  2 k 14 / 8 / 8, 20 k 15 / 11 / 17, 100 k 23 / 29 / 53 (rows of 6 entries)
// beyond them the lanes' extra instructions cost more than idle SIMDs gain.
inline int rowLanes(int dim, int64_t nodes) {
  if (dim == 1) return nodes <= 32768 ? 8 : 1;
  return nodes <= 16384 ? 16 : (nodes <= 49152 ? 8 : 1);
}
// Mixed pair pass: a lane takes a block of kSumBlock entries, two blocks in a 2-D
// row and eight in a 3-D one.
inline int mixedLanes(int dim, int64_t nodes) {
  if (dim == 1) return 1;
  return dim == 2 ? (nodes <= 131072 ? 2 : 1) : (nodes <= 49152 ? 8 : 1);
}
// f(std::integral_constant) with the lanes this dimension is built for.
template <int D, class F> void withLanes(int lanes, F&& f) {
  if constexpr (D > 1) {
    if (lanes == 16) { f(std::integral_constant<int, 16>{}); return; }
  }
  if (lanes == 8) f(std::integral_constant<int, 8>{});
  else f(std::integral_constant<int, 1>{});
}

}  // namespace sphgpu
