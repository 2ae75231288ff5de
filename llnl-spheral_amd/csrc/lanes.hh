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

// Lanes to a node, by pass: the lines lie where the measured times cross (one / 8
// lanes, us; 16 lanes where 8 would leave SIMDs idle).  Beyond them the lanes'
// extra instructions cost more than idle SIMDs gain.
//   pairs (reference order)
//     3-D 1.7 k nodes 189 / 50 (16: 30), 14 k 195 / 71 (72), 27 k 206 / 123, 64 k 224 / 224,
//         104 k 380 / 363, 141 k 565 / 503, 195 k 647 / 690
//     2-D 1 k 47 / 16 (11), 10 k 48 / 20 (17), 32 k 54 / 34, 68 k 83 / 65, 102 k 87 / 90
//     1-D 2 k 14 / 8, 20 k 15 / 11, 100 k 23 / 29 (rows of 6 entries)
//   pairs (search order, FP64)
//     3-D 64 k 151 / 205; 2-D 32 k 44 / 34, 68 k 56 / 57
//   sum density
//     3-D 27 k 87 / 30, 64 k 91 / 61, 104 k 111 / 98, 141 k 133 / 136, 195 k 151 / 190
//     2-D 32 k 29 / 11, 102 k 34 / 26, 250 k 70 / 56
//     mixed: 3-D 64 k 65 / 35, 141 k 87 / 81; 2-D 102 k 28 / 18, 250 k 41 / 35
//   grad-h correction
//     3-D 27 k 70 / 39, 64 k 74 / 74, 104 k 103 / 119; 2-D 68 k 28 / 22, 102 k 30 / 28, 250 k 62 / 58
//   ideal H
//     3-D 27 k 88 / 41, 64 k 87 / 75, 104 k 102 / 107; 2-D 32 k 29 / 23, 68 k 41 / 43
//   compatible energy (two or three dimensions: 8 lanes at every size)
//     3-D 27 k 117 / 30, 104 k 259 / 127, 373 k 958 / 409; 2-D 32 k 26 / 10, 250 k 78 / 49
enum class RowPass { kPairs, kIsoPairs, kDensity, kOmega, kIdealH, kCompat };
inline int rowLanes(RowPass pass, int dim, int64_t nodes) {
  if (dim == 1) return nodes <= 32768 ? 8 : 1;
  if (nodes <= 16384) return 16;
  int64_t most2 = 0, most3 = 0;
  switch (pass) {
    case RowPass::kPairs: most2 = 81920; most3 = 163840; break;
    case RowPass::kIsoPairs: most2 = 65536; most3 = 49152; break;
    case RowPass::kDensity: most2 = 262144; most3 = 131072; break;
    case RowPass::kOmega: most2 = 262144; most3 = 65536; break;
    case RowPass::kIdealH: most2 = 49152; most3 = 81920; break;
    case RowPass::kCompat: return 8;
  }
  return nodes <= (dim == 2 ? most2 : most3) ? 8 : 1;
}
// Mixed pair pass: a lane takes a block of kSumBlock entries, two blocks in a 2-D
// row and eight in a 3-D one.
inline int mixedLanes(int dim, int64_t nodes) {
  if (dim == 1) return 1;
  return dim == 2 ? (nodes <= 131072 ? 2 : 1) : (nodes <= 49152 ? 8 : 1);
}
// f(std::integral_constant) with the lanes this dimension is built for (ONE: one
// lane too).
template <int D, bool ONE = true, class F> void withLanes(int lanes, F&& f) {
  if constexpr (D > 1) {
    if (lanes == 16) { f(std::integral_constant<int, 16>{}); return; }
  }
  if constexpr (ONE) {
    if (lanes == 1) { f(std::integral_constant<int, 1>{}); return; }
  }
  f(std::integral_constant<int, 8>{});
}

}  // namespace sphgpu
