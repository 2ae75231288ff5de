// Order-preserving scans with their producer and consumer in the kernel.
//
// An operation F gives a count per item and takes the exclusive prefix of
// these counts in item order:
//   int32_t value(int64_t i) const            count of item i (pure)
//   void emit(int64_t i, int32_t prefix, int32_t v) const
//   void total(int32_t t) const               once, by one thread
//   kCompact                                  counts are 0 or 1 and only the ones emit
// The emitted data must not feed value().  With kCompact a tile's ones are
// gathered in LDS first and emitted by consecutive lanes, so that a costly
// emit runs once a lane, not up to four times in the lanes that hold them.
//
// Up to kScanOnce items one launch does all: a workgroup sums the counts of
// the tiles before its own by itself, at most 12 extra values a lane.  Beyond,
// a first launch writes the tiles' sums and the second adds up those before its
// tile.  Measured: 4.5 us for one launch of 8 k items; at 30 k 8 us for the two,
// where one launch took 14-28 us (its last tile counts 28 k items again) and a
// scan in one workgroup 11 us without the producer and the consumer.  What the
// second launch adds up grows with the square of the tiles, so from kScanPrefix
// tiles on (the cells of a sparse grid) one workgroup sums them up between the two.
#pragma once
#include <cstdint>
#include <type_traits>
#include <hip/hip_runtime.h>

namespace sphgpu {

constexpr int kScanBlock = 512;
constexpr int64_t kScanOnce = 8192;
// Items a lane.  A GhostPlane's ones lie together (a face of a lattice), so a tile
// may emit all of its items, four rounds of dependent loads at four a lane: 11.0 us
// for the second launch at 82 k rows, 6.4 us at one a lane, where its tiles fill the
// chip as well.  Beyond half a million items each workgroup's pass over the tile
// sums before it costs more than that gives (2.4 M rows: 31 us at four, 38 at two,
// 63 at one).
constexpr int64_t kScanOnePer = 524288;
// Tiles up to which each workgroup adds up the sums before its own.  A whole neighbour
// build of 90 k nodes in two clumps, without and with the launch between: 37 M cells
// (18 k tiles) 0.29 and 0.26 ms, 100 M 0.88 and 0.56, 0.9 G 23.2 and 3.9.
constexpr int64_t kScanPrefix = 16384;

// The workgroup's tile, given each thread's part of the sum before the tile.
template <int PER, class F>
__device__ __forceinline__ void scanTile(const F& f, int64_t n, int32_t before) {
  constexpr int kTile = kScanBlock * PER;
  __shared__ int32_t waveSum[kScanBlock / 64], waveBefore[kScanBlock / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t base = blockIdx.x * int64_t(kTile) + int64_t(threadIdx.x) * PER;
  int32_t v[PER], local = 0;
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    v[q] = base + q < n ? f.value(base + q) : 0;
    local += v[q];
  }
  int32_t incl = local;
#pragma unroll
  for (int s = 1; s < 64; s <<= 1) {
    const int32_t t = __shfl_up(incl, s);
    if (lane >= s) incl += t;
  }
#pragma unroll
  for (int s = 32; s > 0; s >>= 1) before += __shfl_xor(before, s);
  if (lane == 63) {
    waveSum[wave] = incl;
    waveBefore[wave] = before;
  }
  __syncthreads();
  int32_t first = 0, run = incl - local;          // prefix of the tile, and of the thread in it
#pragma unroll
  for (int w = 0; w < kScanBlock / 64; ++w) {
    first += waveBefore[w];
    run += w < wave ? waveSum[w] : 0;
  }
  if constexpr (F::kCompact) {
    __shared__ int32_t ones[kTile];
    int32_t at = run;
#pragma unroll
    for (int q = 0; q < PER; ++q)
      if (v[q]) ones[at++] = threadIdx.x * PER + q;
    int32_t count = 0;
#pragma unroll
    for (int w = 0; w < kScanBlock / 64; ++w) count += waveSum[w];
    __syncthreads();
    for (int32_t t = threadIdx.x; t < count; t += kScanBlock)
      f.emit(blockIdx.x * int64_t(kTile) + ones[t], first + t, 1);
  } else {
    int32_t at = first + run;
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      if (base + q < n) f.emit(base + q, at, v[q]);
      at += v[q];
    }
  }
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == kScanBlock - 1) f.total(first + run + local);
}

template <class F>
__global__ void __launch_bounds__(kScanBlock) k_scan_once(F f, int64_t n) {
  const int64_t tile0 = blockIdx.x * int64_t(kScanBlock * 4);   // <= n: the grid covers n items
  int32_t before = 0;
#pragma unroll 4
  for (int64_t i = threadIdx.x; i < tile0; i += kScanBlock) before += f.value(i);
  scanTile<4>(f, n, before);
}

template <int PER, class F>
__global__ void __launch_bounds__(kScanBlock) k_scan_sums(F f, int64_t n, int32_t* __restrict__ tileSums) {
  __shared__ int32_t waveSum[kScanBlock / 64];
  const int64_t base = blockIdx.x * int64_t(kScanBlock * PER) + threadIdx.x;
  int32_t sum = 0;
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int64_t i = base + int64_t(q) * kScanBlock;
    if (i < n) sum += f.value(i);
  }
  for (int s = 32; s > 0; s >>= 1) sum += __shfl_xor(sum, s);
  if ((threadIdx.x & 63) == 0) waveSum[threadIdx.x >> 6] = sum;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kScanBlock / 64; ++w) sum += waveSum[w];
    tileSums[blockIdx.x] = sum;
  }
}

// The tiles' sums become the sums before each tile (one workgroup).
constexpr int kPrefixBlock = 1024, kPrefixPer = 4;
static __global__ void __launch_bounds__(kPrefixBlock) k_scan_prefix(int32_t* __restrict__ tileSums, int64_t tiles) {
  __shared__ int32_t waveSum[kPrefixBlock / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int32_t carry = 0;
  for (int64_t t0 = 0; t0 < tiles; t0 += kPrefixBlock * kPrefixPer) {
    const int64_t base = t0 + int64_t(threadIdx.x) * kPrefixPer;
    int32_t v[kPrefixPer], local = 0;
#pragma unroll
    for (int q = 0; q < kPrefixPer; ++q) {
      v[q] = base + q < tiles ? tileSums[base + q] : 0;
      local += v[q];
    }
    int32_t incl = local;
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) {
      const int32_t t = __shfl_up(incl, s);
      if (lane >= s) incl += t;
    }
    if (lane == 63) waveSum[wave] = incl;
    __syncthreads();
    int32_t run = carry + incl - local;
#pragma unroll
    for (int w = 0; w < kPrefixBlock / 64; ++w) {
      run += w < wave ? waveSum[w] : 0;
      carry += waveSum[w];
    }
#pragma unroll
    for (int q = 0; q < kPrefixPer; ++q) {
      if (base + q < tiles) tileSums[base + q] = run;
      run += v[q];
    }
    __syncthreads();                               // waveSum is written again
  }
}

// PREFIX: tileSums holds the sums before each tile.
template <int PER, bool PREFIX, class F>
__global__ void __launch_bounds__(kScanBlock) k_scan_emit(F f, int64_t n, const int32_t* __restrict__ tileSums) {
  int32_t before = 0;
  if constexpr (PREFIX) {
    if (threadIdx.x == 0) before = tileSums[blockIdx.x];
  } else {
    for (int64_t t = threadIdx.x; t < blockIdx.x; t += kScanBlock) before += tileSums[t];
  }
  scanTile<PER>(f, n, before);
}

// Runs F over n items (n = 0 still calls total(0)); `tmp` holds the tile sums.
template <class F> void scanItems(const F& f, int64_t n, DBuf& tmp, hipStream_t st) {
  auto tilesOf = [n](int per) { return n > 0 ? (n + kScanBlock * per - 1) / (kScanBlock * per) : 1; };
  auto two = [&](auto per) {
    constexpr int PER = decltype(per)::value;
    const int64_t tiles = tilesOf(PER);
    tmp.ensure(sizeof(int32_t) * size_t(tiles));
    hipLaunchKernelGGL((k_scan_sums<PER, F>), dim3(unsigned(tiles)), dim3(kScanBlock), 0, st, f, n, tmp.as<int32_t>());
    if constexpr (PER > 1) {
      if (tiles > kScanPrefix) {
        hipLaunchKernelGGL(k_scan_prefix, dim3(1), dim3(kPrefixBlock), 0, st, tmp.as<int32_t>(), tiles);
        hipLaunchKernelGGL((k_scan_emit<PER, true, F>), dim3(unsigned(tiles)), dim3(kScanBlock), 0, st, f, n,
                           tmp.as<int32_t>());
        return;
      }
    }
    hipLaunchKernelGGL((k_scan_emit<PER, false, F>), dim3(unsigned(tiles)), dim3(kScanBlock), 0, st, f, n,
                       tmp.as<int32_t>());
  };
  if (n <= kScanOnce) hipLaunchKernelGGL(k_scan_once<F>, dim3(unsigned(tilesOf(4))), dim3(kScanBlock), 0, st, f, n);
  else if (n <= kScanOnePer) two(std::integral_constant<int, 1>{});
  else two(std::integral_constant<int, 4>{});
  SG_CHECK_HIP(hipGetLastError());
}

}  // namespace sphgpu
