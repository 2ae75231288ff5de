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

// Lanes to a node, by pass.  One lane to a node takes as long for one row as for 65536,
// a wavefront on each of the 1024 SIMDs, and steps up at every further 65536; with
// several lanes the time grows with the rows.  So the line between them lies anew in
// every step.  Below 16 Ki nodes 16 lanes, where 8 would leave SIMDs idle (16641 nodes
// in 2-D, 17576 in 3-D, us, 8 / 16: pairs 25.1 / 26.6 and 82.7 / 76.1, density 8.7 / 8.2
// and 21.9 / 19.8, grad-h 19.5 / 18.8 and 38.4 / 35.8).  One lane / 8 lanes, us:
//   pairs (reference order)
//     3-D 1.7 k nodes 189 / 50 (16: 30), 27 k 189 / 115, 51 k 198 / 181, 59 k 203 / 203,
//         64 k 206 / 209; 69 k 299 / 228, 91 k 304 / 292, 104 k 310 / 321, 125 k 320 / 387;
//         133 k 439 / 400, 141 k 447 / 451, 149 k 443 / 459, 166 k 468 / 500
//     2-D 1 k 47 / 16 (11), 17 k 48 / 25, 48 k 54 / 45, 58 k 55 / 55, 66 k 56 / 57;
//         66 k 75 / 61, 82 k 76 / 69, 102 k 80 / 88
//     1-D 2 k 14 / 8, 20 k 15 / 11, 100 k 23 / 29 (rows of 6 entries)
//   pairs, any H
//     3-D 27 k 265 / 147, 51 k 280 / 249, 64 k 280 / 285; 69 k 528 / 317, 104 k 521 / 449,
//         118 k 546 / 515, 125 k 528 / 546; 133 k 771 / 570, 166 k 772 / 707
//     2-D 48 k 67 / 56, 58 k 67 / 69, 66 k 68 / 71; 66 k 95 / 76, 82 k 95 / 86, 102 k 99 / 111
//   pairs, pair accelerations stored (five whole steps with the grad-h correction, ms)
//     3-D 59 k 8.67 / 8.63; 80 k 9.79 / 9.17, 104 k 11.55 / 11.24, 118 k 12.26 / 12.17,
//         125 k 12.66 / 12.74; 133 k 15.4 / 14.2, 149 k 16.3 / 15.5, 166 k 16.95 / 16.60
//     2-D (one pass) 58 k 59 / 56, 66 k 60 / 58; 66 k 80 / 63, 82 k 81 / 69, 102 k 83 / 85
//   pairs (search order, FP64)
//     3-D 27 k 133 / 97, 39 k 139 / 133, 47 k 140 / 152
//     2-D (tuned) 17 k 37 / 21, 48 k 43 / 40, 58 k 46 / 52
//   sum density
//     3-D 27 k 80 / 26, 64 k 84 / 53, 104 k 97 / 79, 125 k 97 / 94, 149 k 114 / 108, 166 k 115 / 121
//     2-D 32 k 24 / 10, 102 k 33 / 24, 250 k 61 / 50
//     mixed: 3-D 64 k 63 / 31, 85 k 65 / 46, 141 k 87 / 81; 2-D 65 k 24 / 12, 250 k 37 / 34
//   sum density, any H
//     3-D 51 k 91 / 76, 111 k 150 / 146, 118 k 151 / 154, 125 k 153 / 163
//     2-D 102 k 38 / 35, 116 k 39 / 40, 131 k 41 / 43; 144 k 57 / 48, 250 k 90 / 76
//   grad-h correction
//     3-D 27 k 72 / 45, 59 k 80 / 79, 64 k 79 / 81, 91 k 101 / 107
//     2-D 32 k 30 / 21, 102 k 37 / 36, 116 k 39 / 41, 131 k 40 / 43; 144 k 44 / 46, 194 k 45 / 56
//   grad-h correction, any H
//     3-D 51 k 93 / 74, 64 k 94 / 82
//     2-D 102 k 43 / 41, 116 k 45 / 46, 131 k 46 / 49; 144 k 56 / 54, 194 k 67 / 65, 250 k 94 / 79
//   ideal H
//     3-D 27 k 88 / 41, 64 k 87 / 75, 104 k 102 / 107; 2-D 32 k 29 / 23, 68 k 41 / 43
//   compatible energy (two or three dimensions: 8 lanes at every size)
//     3-D 27 k 117 / 30, 104 k 259 / 127, 373 k 958 / 409; 2-D 32 k 26 / 10, 250 k 78 / 49
enum class RowPass { kPairs, kPairsAnyH, kPairsStored, kIsoPairs, kDensity, kDensityAnyH, kOmega, kOmegaAnyH, kIdealH,
                     kCompat };
inline int rowLanes(RowPass pass, int dim, int64_t nodes) {
  if (dim == 1) return nodes <= 32768 ? 8 : 1;
  if (nodes <= 16384) return 16;
  if (pass == RowPass::kCompat) return 8;
  // the most nodes that take 8 lanes in each step of 65536, in 1024s, 2-D and 3-D
  constexpr int kSteps = 4;
  constexpr int kMost[][2][kSteps] = {
      {{56, 80, 0, 0}, {56, 92, 136, 0}},         // kPairs
      {{56, 80, 0, 0}, {56, 116, 160, 0}},        // kPairsAnyH
      {{64, 80, 0, 0}, {64, 116, 160, 0}},        // kPairsStored
      {{48, 0, 0, 0}, {40, 0, 0, 0}},             // kIsoPairs
      {{64, 128, 192, 256}, {64, 128, 0, 0}},     // kDensity
      {{64, 112, 192, 256}, {64, 112, 0, 0}},     // kDensityAnyH
      {{64, 104, 0, 0}, {60, 0, 0, 0}},           // kOmega
      {{64, 104, 192, 256}, {64, 0, 0, 0}},       // kOmegaAnyH
      {{48, 0, 0, 0}, {64, 80, 0, 0}},            // kIdealH
  };
  const int64_t step = (nodes - 1) / 65536;
  return step < kSteps && nodes <= int64_t(kMost[int(pass)][dim - 2][step]) * 1024 ? 8 : 1;
}
// Mixed pair pass: a lane takes a block of kSumBlock entries, two blocks in a 2-D
// row and eight in a 3-D one.  One lane (2-D: the tuned launch) / several, us:
//   3-D 27 k 115 / 64, 47 k 123 / 96, 51 k 124 / 116, 64 k 127 / 126, 69 k 140 / 145, 85 k 142 / 174
//   2-D 4 k 31 / 22, 32 k 33 / 23, 65 k 39 / 31, 90 k 43 / 39, 116 k 46 / 48, 131 k 47 / 51
inline int mixedLanes(int dim, int64_t nodes) {
  if (dim == 1) return 1;
  return dim == 2 ? (nodes <= 98304 ? 2 : 1) : (nodes <= 49152 ? 8 : 1);
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
