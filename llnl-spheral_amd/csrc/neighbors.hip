// Device ConnectivityMap build.
//
// Contract (src/Neighbor/ConnectivityMap.cc:630-749): for an internal node i, j
// is a neighbour iff |H_i r_ij|^2 <= ext^2 or |H_j r_ij|^2 <= ext^2 (FP64,
// r_ij = r_i - r_j, SymTensor.Vector and magnitude2 summed left to right), j != i.
// The reference orders each row by node index (:735-738); that order is kept on
// request (SPHGPU_ROW_ORDER_REFERENCE, needed for reference-order FP64 sums),
// otherwise rows keep the deterministic search order.  How candidates are found
// is free (the reference's NestedGridNeighbor only has to return a superset):
//
//  1. bounds: min/max position, the smallest Gershgorin lower bound of
//     lambda_min(H) over all nodes, and whether every H is h I.  |H r| <= ext
//     implies |r| <= R = ext/min(lambda) (plus a 1e-6 relative margin).
//  2. counting sort of nodes by cell (rank by comparison inside a cell).  Cells are numbered brick by brick
//     (4^nu cells per brick, Z-order inside) so a brick's nodes are contiguous;
//     each cell is then ordered by node index (the order depends only on
//     positions and indices).  Records of all nodes are packed in this order.
//  3. rows, one thread per internal node, into a blocked-transposed ELL: entry
//     w of slot k at nbr[((w/4)*n + k)*4 + w%4], so four entries are one int4
//     and a wavefront's int4s are contiguous (coalesced writes here, coalesced
//     int4 reads in the passes):
//      - 3-D with isotropic H: cells of edge R/2, one workgroup per brick
//        stages the 8^3 cells around it in LDS (FP32 offsets from the brick
//        origin), each node scans its 5^3 cells; the FP32 estimate of h^2|r|^2
//        decides every pair farther than 1e-5 (relative) from the threshold,
//        the rest take the exact FP64 reference test;
//      - otherwise: cells of edge R, 3^nu stencil read from global memory.
//     Rows longer than the ELL capacity are counted, the build grows the
//     capacity and repeats the row pass.
//  4. optionally, rows sorted by node index (one wavefront per row, bitonic
//     sort in registers).
// Ensembles: bounds and grid per member (each member's grid is the one it
// would get alone); a member's cells are numbered after those of the members
// before it, so the sort groups slots by member, and a row only looks at its
// own member's cells.
#include "internal.hh"
#include "dgeom.hh"
#include "records.hh"
#include "ell.hh"
#include "pack.hh"
#include "scan.hh"
#include <cstring>

namespace sphgpu {

namespace {

constexpr int kBlock = 256;

inline int nblocks(int64_t n, int bs = kBlock) { return int(std::max<int64_t>(1, (n + bs - 1) / bs)); }

// Gershgorin lower bound of the smallest eigenvalue of a SymTensor.
template <int D> __device__ double gershgorinMin(const double* h) {
  if constexpr (D == 1) return h[0];
  else if constexpr (D == 2) return dmin(h[0] - fabs(h[1]), h[2] - fabs(h[1]));
  else return dmin(h[0] - fabs(h[1]) - fabs(h[2]), dmin(h[3] - fabs(h[1]) - fabs(h[4]), h[5] - fabs(h[2]) - fabs(h[4])));
}
template <int D> __device__ bool isIsotropic(const double* h) {
  if constexpr (D == 1) return true;
  else if constexpr (D == 2) return h[1] == 0.0 && h[2] == h[0];
  else return h[1] == 0.0 && h[2] == 0.0 && h[4] == 0.0 && h[3] == h[0] && h[5] == h[0];
}

// reduced values: lo[3] hi[3] min Gershgorin bound, isotropic flag, max diagonal
// of H, max Gershgorin bound, non-finite flag (1 when a position or H entry is
// NaN or infinite: min and max would pass a NaN over)
constexpr int kNB = 11;
constexpr int kNonFinite = 10;
__host__ __device__ __forceinline__ bool isMaxSlot(int k) { return (k >= 3 && k < 6) || k >= 8; }
#define SG_BOUNDS_IDENT {1e300, 1e300, 1e300, -1e300, -1e300, -1e300, 1e300, 1.0, -1e300, -1e300, 0.0}

// Bounds a grid can be made from: finite positions and H, and a positive
// Gershgorin bound (1: ok; 0: a non-finite entry; -1: no positive bound).
int boundsUsable(const double* hb) {
  if (hb[kNonFinite] > 0.5) return 0;
  return (hb[6] > 0.0 && std::isfinite(hb[6]) && hb[9] > 0.0 && std::isfinite(hb[9])) ? 1 : -1;
}
void requireUsableBounds(const double* hb) {
  const int u = boundsUsable(hb);
  SG_REQUIRE(u != 0, SPHGPU_ERR_ARG, "non-finite node position or H");
  SG_REQUIRE(u > 0, SPHGPU_ERR_UNSUPPORTED, "neighbour search needs H with a positive Gershgorin bound on every node");
}

template <int D> __device__ __forceinline__ bool rowFinite(const double* x, const double* h) {
  bool ok = true;
  for (int k = 0; k < D; ++k) ok = ok && isfinite(x[k]);
  for (int k = 0; k < NSym<D>::value; ++k) ok = ok && isfinite(h[k]);
  return ok;
}

template <int D> __device__ double maxDiag(const double* h) {
  double m = h[0];
  for (int a = 1; a < D; ++a) m = dmax(m, h[sdiag<D>(a)]);
  return m;
}

// n rows, or with nDev the rows the ghost generation has left on the device.  The
// workgroups' bounds of up to kBoundsHost of them go to pinned memory, with the
// generation's counts (genOut), and the host, which waits for them anyway, takes the
// last step: 22 KB at most in 3 us, where a launch of one workgroup took 5 us and
// 4 us of the host.  Beyond, k_bounds_final reduces them.
constexpr int kBoundsHost = 256;
template <int D>
__global__ void k_bounds(const double* __restrict__ pos, const double* __restrict__ H, int64_t n,
                         const int64_t* __restrict__ nDev, double* partials, const int64_t* __restrict__ gen, int nGen,
                         int64_t* __restrict__ genOut) {
  if (nDev) n = *nDev;
  if (genOut && blockIdx.x == 0)
    for (int q = threadIdx.x; q < nGen; q += blockDim.x) genOut[q] = gen[q];
  __shared__ double sh[kNB][kBlock];
  double r[kNB] = SG_BOUNDS_IDENT;
  for (int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x) {
    for (int k = 0; k < D; ++k) { const double x = pos[i * D + k]; r[k] = dmin(r[k], x); r[3 + k] = dmax(r[3 + k], x); }
    const double* h = H + i * NSym<D>::value;
    const double gm = gershgorinMin<D>(h);
    r[6] = dmin(r[6], gm);
    if (!isIsotropic<D>(h)) r[7] = 0.0;
    r[8] = dmax(r[8], maxDiag<D>(h));
    r[9] = dmax(r[9], gm);
    if (!rowFinite<D>(pos + i * D, h)) r[kNonFinite] = 1.0;
  }
  for (int k = 0; k < kNB; ++k) sh[k][threadIdx.x] = r[k];
  __syncthreads();
  for (int s = kBlock / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s)
      for (int k = 0; k < kNB; ++k) {
        const double a = sh[k][threadIdx.x], b = sh[k][threadIdx.x + s];
        sh[k][threadIdx.x] = isMaxSlot(k) ? dmax(a, b) : dmin(a, b);
      }
    __syncthreads();
  }
  if (threadIdx.x < kNB) partials[blockIdx.x * kNB + threadIdx.x] = sh[threadIdx.x][0];
}

// The bounds, and the ghost generation's counts, straight to pinned memory.
__global__ void k_bounds_final(const double* partials, int nb, double* __restrict__ out, const int64_t* __restrict__ gen,
                               int nGen, int64_t* __restrict__ genOut) {
  for (int q = threadIdx.x; q < nGen; q += blockDim.x) genOut[q] = gen[q];
  __shared__ double sh[kNB][kBlock];
  double r[kNB] = SG_BOUNDS_IDENT;
  for (int b = threadIdx.x; b < nb; b += blockDim.x)
    for (int k = 0; k < kNB; ++k) {
      const double v = partials[b * kNB + k];
      r[k] = isMaxSlot(k) ? dmax(r[k], v) : dmin(r[k], v);
    }
  for (int k = 0; k < kNB; ++k) sh[k][threadIdx.x] = r[k];
  __syncthreads();
  for (int s = kBlock / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s)
      for (int k = 0; k < kNB; ++k) {
        const double a = sh[k][threadIdx.x], b = sh[k][threadIdx.x + s];
        sh[k][threadIdx.x] = isMaxSlot(k) ? dmax(a, b) : dmin(a, b);
      }
    __syncthreads();
  }
  if (threadIdx.x < kNB) out[threadIdx.x] = sh[threadIdx.x][0];
}

struct DGrid {
  double lo[3];
  double cell;
  double invCell;
  int nc[3];
  int nb[3];
};

// Grid lists.  Grids [first[m], first[m+1]) serve ensemble member m (m = 0
// without an ensemble), in increasing cell size: the levels of a node set
// whose search radii span more than a factor 2.  A node lives in the first of
// its member's grids whose cell is at least its search radius bound
// ext/gershgorin(H)(1 + 1e-6).  g == null: one grid, passed by value.
struct SegGrids {
  const double* seg;        // member index per caller row, or null
  const DGrid* g;
  const int64_t* base;      // first global cell of each grid
  const int32_t* first;     // grids of each member, +1 entry
  double ext;
};

template <int D> __device__ __forceinline__ double searchRadius(const double* h, double ext) {
  return ext / gershgorinMin<D>(h) * (1.0 + 1.0e-6);
}

// Order-preserving map of a double onto uint64 (for atomic min/max).
__device__ __forceinline__ unsigned long long orderedBits(double x) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(x);
  return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}
inline double fromOrderedBits(unsigned long long o) {
  const unsigned long long b = (o >> 63) ? (o & 0x7FFFFFFFFFFFFFFFull) : ~o;
  double x;
  std::memcpy(&x, &b, sizeof(x));
  return x;
}

// The bounds of k_bounds per member, as ordered bits: a max slot keeps its
// bits, a min slot their complement, so that every slot is an atomic maximum
// that starts at zero.  A wavefront walks `groups` consecutive groups of 64 rows
// (members are contiguous runs of internal rows) and keeps a running reduction
// in registers while its groups stay in one member; in a group that spans members
// (ghost rows, whose planes mix them) each run of a member's rows is reduced to its
// first lane.  Either way a slot that already holds as much is left alone: 10
// contended atomics a lane were 105 us of a 30 k row batch (a plain read may be
// stale, then the atomic decides).  Max is order-free, so the result does not
// depend on the grouping.  A lane enters one slot of a uniform wavefront, where
// lane 0 entered all eleven, a read and an atomic each: 33 -> 15 us for six 2-D
// members (39 k rows), 18 -> 8 us for 24 tubes.  `clear` is the next build's table.
constexpr int kSegGroups = 16;
template <int D>
__global__ void __launch_bounds__(kBlock) k_seg_bounds(const double* __restrict__ pos, const double* __restrict__ H,
                                                       const double* __restrict__ seg, int64_t n,
                                                       const int64_t* __restrict__ nDev, int groups,
                                                       unsigned long long* __restrict__ bits,
                                                       unsigned long long* __restrict__ clear, int words) {
  if (nDev) n = *nDev;
  const int64_t tid = blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
  for (int64_t q = tid; q < words; q += int64_t(gridDim.x) * blockDim.x) clear[q] = 0ull;
  const int lane = threadIdx.x & 63;
  const int64_t base = (tid >> 6) * int64_t(64 * groups);
  const double ident[kNB] = SG_BOUNDS_IDENT;
  double acc[kNB];
  for (int k = 0; k < kNB; ++k) acc[k] = ident[k];
  int mAcc = -1;                           // member of the running reduction (wave-uniform)
  auto entry = [&](int k, double v) { return isMaxSlot(k) ? orderedBits(v) : ~orderedBits(v); };
  auto flush = [&]() {                     // called by the whole wavefront
    // lane k enters slot k: one read and one atomic in a row instead of kNB
    unsigned long long mine = 0;
    for (int k = 0; k < kNB; ++k) {
      double v = acc[k];
      for (int sh = 32; sh > 0; sh >>= 1) {
        const double o = __shfl_xor(v, sh);
        v = isMaxSlot(k) ? dmax(v, o) : dmin(v, o);
      }
      mine = lane == k ? entry(k, v) : mine;
      acc[k] = ident[k];
    }
    if (lane < kNB) {
      unsigned long long* p = bits + int64_t(mAcc) * kNB + lane;
      if (mine > *static_cast<volatile unsigned long long*>(p)) atomicMax(p, mine);
    }
  };
  for (int it = 0; it < groups; ++it) {
    const int64_t i = base + int64_t(it) * 64 + lane;
    double r[kNB];
    for (int k = 0; k < kNB; ++k) r[k] = ident[k];
    int m = -1;
    if (i < n) {
      m = int(seg[i]);
      for (int k = 0; k < D; ++k) { const double x = pos[i * D + k]; r[k] = x; r[3 + k] = x; }
      const double* h = H + i * NSym<D>::value;
      r[6] = gershgorinMin<D>(h);
      r[7] = isIsotropic<D>(h) ? 1.0 : 0.0;
      r[8] = maxDiag<D>(h);
      r[9] = r[6];
      r[kNonFinite] = rowFinite<D>(pos + i * D, h) ? 0.0 : 1.0;
    }
    const int m0 = __shfl(m, 0);
    if (m0 < 0) break;                     // lane 0 holds the group's first row: the rest are past n too
    if (__all(m == m0 || m < 0)) {
      if (m0 != mAcc) {
        if (mAcc >= 0) flush();
        mAcc = m0;
      }
      for (int k = 0; k < kNB; ++k) acc[k] = isMaxSlot(k) ? dmax(acc[k], r[k]) : dmin(acc[k], r[k]);
    } else {
      if (mAcc >= 0) flush();
      mAcc = -1;
      // a run of one member's rows is reduced to its first lane
      for (int sh = 1; sh < 64; sh <<= 1) {
        const int mo = __shfl_down(m, sh);
        const bool same = lane + sh < 64 && mo == m;
        for (int k = 0; k < kNB; ++k) {
          const double o = __shfl_down(r[k], sh);
          const double v = isMaxSlot(k) ? dmax(r[k], o) : dmin(r[k], o);
          r[k] = same ? v : r[k];
        }
      }
      const int before = __shfl_up(m, 1);
      if (m >= 0 && (lane == 0 || before != m)) {
        unsigned long long* p = bits + int64_t(m) * kNB;
        unsigned long long held[kNB];      // all reads before the first wait
#pragma unroll
        for (int k = 0; k < kNB; ++k) held[k] = static_cast<volatile unsigned long long*>(p)[k];
#pragma unroll
        for (int k = 0; k < kNB; ++k) {
          const unsigned long long o = entry(k, r[k]);
          if (o > held[k]) atomicMax(p + k, o);
        }
      }
    }
  }
  if (mAcc >= 0) flush();
}

// Member bounds and generation counts to pinned memory.
__global__ void k_report(const unsigned long long* __restrict__ bits, int words, unsigned long long* __restrict__ out,
                         const int64_t* __restrict__ gen, int nGen, int64_t* __restrict__ genOut) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < words) out[t] = bits[t];
  if (t < nGen) genOut[t] = gen[t];
}

template <int D> __device__ __forceinline__ void cellCoords(const DGrid& g, const double* x, int* c) {
  c[0] = c[1] = c[2] = 0;
  for (int k = 0; k < D; ++k) {
    int ck = int((x[k] - g.lo[k]) * g.invCell);
    ck = ck < 0 ? 0 : (ck >= g.nc[k] ? g.nc[k] - 1 : ck);
    c[k] = ck;
  }
}

// Brick-ordered cell id: bricks of 4^nu cells in row-major order, Z-order inside.
template <int D> __device__ __forceinline__ int64_t cellId(const DGrid& g, int cx, int cy, int cz) {
  if constexpr (D == 1) {
    return cx;
  } else if constexpr (D == 2) {
    const int64_t b = int64_t(cy >> 2) * g.nb[0] + (cx >> 2);
    const int lx = cx & 3, ly = cy & 3;
    const int z = (lx & 1) | ((ly & 1) << 1) | ((lx & 2) << 1) | ((ly & 2) << 2);
    return b * 16 + z;
  } else {
    const int64_t b = (int64_t(cz >> 2) * g.nb[1] + (cy >> 2)) * g.nb[0] + (cx >> 2);
    const int lx = cx & 3, ly = cy & 3, lz = cz & 3;
    const int z = (lx & 1) | ((ly & 1) << 1) | ((lz & 1) << 2) | ((lx & 2) << 2) | ((ly & 2) << 3) | ((lz & 2) << 4);
    return b * 64 + z;
  }
}

template <int D>
__global__ void k_cell_count(const double* __restrict__ pos, const double* __restrict__ H, int64_t n, DGrid g,
                             SegGrids sg, int32_t* __restrict__ cellOf, int32_t* __restrict__ cellCount,
                             int32_t* __restrict__ cellRank) {
  const int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
  if (i >= n) return;
  int64_t base = 0;
  if (sg.g) {
    const int m = sg.seg ? int(sg.seg[i]) : 0;
    int q = sg.first[m];
    const int e = sg.first[m + 1];
    if (e - q > 1) {
      const double R = searchRadius<D>(H + i * NSym<D>::value, sg.ext);
      while (q < e - 1 && R > sg.g[q].cell) ++q;
    }
    g = sg.g[q];
    base = sg.base[q];
  }
  int c[3];
  cellCoords<D>(g, pos + i * D, c);
  const int32_t id = int32_t(base + cellId<D>(g, c[0], c[1], c[2]));
  cellOf[i] = id;
  cellRank[i] = atomicAdd(&cellCount[id], 1);
}

// cellStart from cellCount (scan.hh)
struct CellScan {
  static constexpr bool kCompact = false;
  const int32_t* count;
  int32_t* start;
  int64_t n;
  __device__ int32_t value(int64_t i) const { return count[i]; }
  __device__ void emit(int64_t i, int32_t prefix, int32_t) const { start[i] = prefix; }
  __device__ void total(int32_t t) const { start[n] = t; }
};

// Each cell's members together, in the order the count met them; with `keys`
// also their x (pos[i * stride]), which the ordering then reads contiguously.
__global__ void k_cell_scatter(const int32_t* __restrict__ cellOf, const int32_t* __restrict__ cellStart,
                               const int32_t* __restrict__ cellRank, int32_t* __restrict__ members, int64_t n,
                               const double* __restrict__ pos, int stride, double* __restrict__ keys) {
  const int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
  if (i >= n) return;
  const int32_t q = cellStart[cellOf[i]] + cellRank[i];
  members[q] = int32_t(i);
  if (keys) keys[q] = pos[i * stride];
}

// The slot of every row: its rank in its cell by node index, or, XKEY, by x and
// then node index, so that the members of a row of cells are in x order; then
// the maps both ways and the row's records.  One lane per row compares it with
// the members of its cell: independent reads of lines the neighbouring lanes
// share, where one lane per cell sorting by insertion ran a dependent chain
// over global memory (40 us in a batch of blasts, whose cells hold ~9 nodes,
// against 9 us for this kernel with the pack in it).  Rows are walked in
// caller order, so the fields are read contiguously and each record is written
// whole.
template <int D, bool ISO, int SEC, bool XKEY>
__global__ void __launch_bounds__(kBlock) k_cell_order(const int32_t* __restrict__ cellOf,
                                                       const int32_t* __restrict__ cellStart,
                                                       const int32_t* __restrict__ members,
                                                       const double* __restrict__ keys, int64_t n,
                                                       int32_t* __restrict__ perm,
                                                       int32_t* __restrict__ iperm, PackIn in, PackOut o) {
  const int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
  if (i >= n) return;
  const int32_t c = cellOf[i];
  const int32_t b = cellStart[c], e = cellStart[c + 1];
  int32_t rank = 0;
  const double x = XKEY ? in.pos[i * D] : 0.0;
  // four members at a time: their reads are in flight together
  for (int32_t q0 = b; q0 < e; q0 += 4) {
    int32_t u[4];
    double xu[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int32_t at = q0 + q < e ? q0 + q : e - 1;
      u[q] = members[at];
      if constexpr (XKEY) xu[q] = keys[at];
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      bool before = u[q] < int32_t(i);
      if constexpr (XKEY) before = xu[q] < x || (xu[q] == x && before);
      rank += (before && q0 + q < e) ? 1 : 0;
    }
  }
  const int32_t k = b + rank;
  perm[k] = int32_t(i);
  iperm[i] = k;
  packRow<D, ISO, SEC>(k, i, loadPackRow<D, ISO>(i, in), o);
}

// Row writer of one lane: keeps up to four entries in registers and stores them as
// one int4.  Each entry is shifted in at w and a marker goes in below them, so the
// buffer itself tells when the next entry fills it, and only whole chunks are
// counted; the last partial chunk is aligned once per row, zeros after its
// entries.  `at` walks the row's chunks (ellChunk(c, n, k) = c n + k).  Capacities
// are multiples of 4.
struct ChunkWriter {
  int4 buf;
  int chunks, room;
  int64_t n;
  int4* at;
  __device__ __forceinline__ ChunkWriter(int4* o, int64_t n_, int64_t k_, int cap)
      : buf{0, 0, 0, -1}, chunks(0), room(cap / 4), n(n_), at(o + ellChunk(0, n_, k_)) {}
  // append v when acc, shifted in by selects
  __device__ __forceinline__ void pushIf(bool acc, int32_t v) {
    const bool full = acc && buf.x == -1;
    buf.x = acc ? buf.y : buf.x;
    buf.y = acc ? buf.z : buf.y;
    buf.z = acc ? buf.w : buf.z;
    buf.w = acc ? v : buf.w;
    if (full) {
      if (chunks < room) *at = buf;
      at += n;
      ++chunks;
      buf.w = -1;
    }
  }
  // the last chunk, and the row's length (which may pass its capacity)
  __device__ __forceinline__ int32_t finish() {
    const int r = buf.w == -1 ? 0 : (buf.z == -1 ? 1 : (buf.y == -1 ? 2 : 3));
    if (r != 0 && chunks < room)
      *at = r == 1 ? make_int4(buf.w, 0, 0, 0)
                   : (r == 2 ? make_int4(buf.z, buf.w, 0, 0) : make_int4(buf.y, buf.z, buf.w, 0));
    return 4 * chunks + r;
  }
};

// Entries and the longest row of a search: summed in the workgroup, one pair
// of atomics each, in the workgroup's bin of the flags.
template <int BS = kBlock> struct RowStats {
  uint32_t sum = 0;
  int32_t most = 0;
  __device__ __forceinline__ void add(int32_t c) {
    sum += uint32_t(c);
    most = c > most ? c : most;
  }
  // called by every thread of the workgroup
  __device__ __forceinline__ void store(int32_t* __restrict__ flags) {
    __shared__ uint32_t ws[BS / 64];
    __shared__ int32_t wm[BS / 64];
    for (int sh = 32; sh > 0; sh >>= 1) {
      sum += __shfl_xor(sum, sh);
      const int32_t m = __shfl_xor(most, sh);
      most = m > most ? m : most;
    }
    if ((threadIdx.x & 63) == 0) {
      ws[threadIdx.x >> 6] = sum;
      wm[threadIdx.x >> 6] = most;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int w = 1; w < BS / 64; ++w) {
        sum += ws[w];
        most = wm[w] > most ? wm[w] : most;
      }
      if (sum) {
        int32_t* bin = flags + kRowBinStride * (1 + blockIdx.x % kRowBins);
        atomicAdd(reinterpret_cast<unsigned long long*>(bin + 2), (unsigned long long)sum);
        if (most > *static_cast<volatile int32_t*>(bin)) atomicMax(bin, most);
      }
    }
  }
};

// ---------------------------------------------------------------------------
// Staged brick search, 3-D, isotropic H.
// ---------------------------------------------------------------------------
constexpr int kStageEdge = 8;                       // 4-cell brick + 2 cells each side
constexpr int kStaged = kStageEdge * kStageEdge * kStageEdge;
// Candidates a brick stages.  A 4 R wide halo of a lattice at nPerh = 1.51 is 12
// or 13 planes wide on each axis: 13^3 = 2197 where all three axes catch one
// more, and such a brick must not fall back to reading every candidate from
// global memory: a few dozen of 13 k bricks held a whole 128^3 search up (1.84 ms
// with room for 2048 candidates, 1.58 ms with 2240).  2240 is what three
// workgroups per CU leave room for.
constexpr int kCandCap = 2240;
// A brick's outer layers hold 7 x 7 x 6 or 7^3 nodes with the ghosts, more than
// 256 lanes, and a second round of the walk is as long as the first.  While every
// brick has a place on the chip at two workgroups of 512 lanes to a CU, one round
// does (343 bricks: 170 us with 256 lanes, 96 with 512; 500 bricks: 143 and 107);
// beyond, three workgroups of 256 hide each other's rounds (729 bricks: 190 and
// 195 us).
constexpr int kWideBlock = 512;
constexpr int64_t kWideBricks = 512;
constexpr int kRunRows = 6;      // one z slab: 5 runs and the sentinel

struct SearchArgs {
  DGrid g;
  double ext, ext2;
  float mid32, half32;      // ext2 and half the band around it that the exact test decides (FP32)
  float prune2, cell32, invCell32;   // staged path: (search radius (1 + 1e-4))^2, cell edge and its inverse (FP32)
  int64_t n, nInt;
  int cap;
  int32_t* keepSlot;        // optional: set to 1 for every ghost slot some row holds
};

// Exact reference test for isotropic H: eta = h r componentwise (the SymTensor
// product with zero off-diagonals), magnitude2 left to right.
__device__ __forceinline__ bool exactIso(double rx, double ry, double rz, double hi, double hj, double ext2) {
  const double ax = hi * rx, ay = hi * ry, az = hi * rz;
  const double bx = hj * rx, by = hj * ry, bz = hj * rz;
  const double e2i = ax * ax + ay * ay + az * az;
  const double e2j = bx * bx + by * by + bz * bz;
  return (e2i <= ext2 || e2j <= ext2);
}

template <int BS>
__global__ void __launch_bounds__(BS) k_search_staged(const double* __restrict__ rec, const int32_t* __restrict__ cellStart,
                                                         SearchArgs a, int32_t* __restrict__ rowCount,
                                                         int4* __restrict__ nbr, int32_t* __restrict__ flags) {
  using R = RL<true>;
  __shared__ int32_t sOff[kStaged + 1];
  __shared__ float4 sCand[kCandCap];               // x,y,z offsets from the brick origin, (1/h)^2 (FP32)
  __shared__ int32_t sSlot[kCandCap];
  // per lane: the runs of one z slab of its stencil (t0 | t1 << 16),
  // lane-strided; up to 5 runs and the sentinel the reader stays on past them.
  // Before the runs are formed the same memory holds each staged cell's first
  // slot and the scan's partial sums (52 KB in all: three workgroups per CU)
  __shared__ uint32_t sRun[kRunRows * BS];
  __shared__ int32_t sMembers;                     // bits of the staged cells' member counts
  static_assert(kRunRows * BS >= kStaged + BS / 64, "sStart and sc alias the run table");
  int32_t* const sStart = reinterpret_cast<int32_t*>(sRun);
  int32_t* const sc = sStart + kStaged;
  const DGrid& g = a.g;
  const int b = int(xcdBlock(int64_t(g.nb[0]) * g.nb[1] * g.nb[2]));
  if (b >= g.nb[0] * g.nb[1] * g.nb[2]) return;   // uniform over the block
  const int bx = b % g.nb[0], by = (b / g.nb[0]) % g.nb[1], bz = b / (g.nb[0] * g.nb[1]);
  const int64_t h0 = cellStart[int64_t(b) * 64], h1 = cellStart[int64_t(b) * 64 + 64];
  if (h0 == h1) return;                           // uniform over the block
  RowStats<BS> stats;
  const int cx0 = bx * 4 - 2, cy0 = by * 4 - 2, cz0 = bz * 4 - 2;
  const double ox = g.lo[0] + (bx * 4) * g.cell, oy = g.lo[1] + (by * 4) * g.cell, oz = g.lo[2] + (bz * 4) * g.cell;
  // staged cell table (x fastest)
  for (int t = threadIdx.x; t < kStaged; t += BS) {
    const int sx = t % kStageEdge, sy = (t / kStageEdge) % kStageEdge, sz = t / (kStageEdge * kStageEdge);
    const int cx = cx0 + sx, cy = cy0 + sy, cz = cz0 + sz;
    int32_t st = 0, cnt = 0;
    if (cx >= 0 && cx < g.nc[0] && cy >= 0 && cy < g.nc[1] && cz >= 0 && cz < g.nc[2]) {
      const int64_t id = cellId<3>(g, cx, cy, cz);
      st = cellStart[id];
      cnt = cellStart[id + 1] - st;
    }
    sStart[t] = st;
    sOff[t + 1] = cnt;
  }
  if (threadIdx.x == 0) {
    sOff[0] = 0;
    sMembers = 0;
  }
  __syncthreads();
  // inclusive scan of sOff[1..512], kStaged / BS elements a thread: within the
  // wavefront, then over the wavefronts' sums
  {
    constexpr int PER = kStaged / BS;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int32_t v[PER], own = 0;
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      v[q] = sOff[PER * threadIdx.x + 1 + q];
      own += v[q];
      if (v[q]) atomicOr(&sMembers, v[q]);
    }
    int32_t incl = own;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int32_t up = __shfl_up(incl, d);
      if (lane >= d) incl += up;
    }
    if (lane == 63) sc[wave] = incl;
    __syncthreads();
    int32_t run = incl - own;
#pragma unroll
    for (int w = 0; w < BS / 64; ++w) run += w < wave ? sc[w] : 0;
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      run += v[q];
      sOff[PER * threadIdx.x + 1 + q] = run;
    }
  }
  __syncthreads();
  const int32_t total = sOff[kStaged];
  const bool staged = total < kCandCap;           // and one more: the candidate that no node takes
  int ghosts = 0;
  if (staged) {
    for (int t = threadIdx.x; t < kStaged; t += BS) {
      const int32_t o = sOff[t], cnt = sOff[t + 1] - o, st = sStart[t];
      for (int q = 0; q < cnt; ++q) {
        const double4 r = *reinterpret_cast<const double4*>(rec + int64_t(st + q) * R::STRIDE);
        sCand[o + q] = make_float4(float(r.x - ox), float(r.y - oy), float(r.z - oz), float(r.w) * float(r.w));
        // bit 31 flags a ghost (slots stay below 2^31)
        const bool ghost = rec[int64_t(st + q) * R::STRIDE + R::ORIG] >= double(a.nInt);
        ghosts |= ghost ? 1 : 0;
        sSlot[o + q] = int32_t(uint32_t(st + q) | (ghost ? 0x80000000u : 0u));
      }
    }
    if (threadIdx.x == 0) {
      sCand[total] = make_float4(1.0e30f, 0.0f, 0.0f, 1.0f);
      sSlot[total] = 0;
    }
  } else if (threadIdx.x == 0) {
    atomicAdd(&flags[1], 1);                      // bricks that read candidates from global memory
  }
  __syncthreads();
  // ghost marks only where the staged candidates hold a ghost (the outer
  // bricks): a scalar flag, so interior bricks skip the mark code per candidate
  const bool marks =
      __builtin_amdgcn_readfirstlane(__syncthreads_or(ghosts)) != 0 && a.keepSlot != nullptr;

  const int steps = 32 - __builtin_clz(__builtin_amdgcn_readfirstlane(sMembers) | 1);   // bisections of a cell
  // One lane per node; the node's 25 (dz, dy) runs of up to 5 staged cells
  // are contiguous candidate ranges in LDS.  Rows leave as int4 chunks, one
  // per lane, contiguous across a wavefront's slots.  Bricks whose candidates
  // exceed the stage read them from the records in global memory.
  // the cell table's first slots are read again only by bricks that are not
  // staged, which write no runs
  for (int64_t k = h0 + threadIdx.x; k < h1; k += BS) {
    const double* ri = rec + k * R::STRIDE;
    if (int64_t(ri[R::ORIG]) >= a.nInt) { rowCount[k] = 0; continue; }
    const double xi = ri[R::X], yi = ri[R::X + 1], zi = ri[R::X + 2], hi = ri[R::HINV];
    const float fx = float(xi - ox), fy = float(yi - oy), fz = float(zi - oz);
    const int32_t hi2 = __float_as_int(float(hi) * float(hi));
    int c[3];
    const double xv[3] = {xi, yi, zi};
    cellCoords<3>(g, xv, c);
    const int sx = c[0] - cx0, sy = c[1] - cy0, sz = c[2] - cz0;   // in [2, 5]
    ChunkWriter row(nbr, a.n, k, a.cap);
    if (staged) {
      for (int dz = -2; dz <= 2; ++dz) {
        // 1. the node's non-empty runs of this z slab, in dy order, into its
        //    column of the run table: the candidates of each (dz, dy) row of
        //    staged cells inside the x chord of a sphere of the search radius
        //    (with a 1e-4 margin) around the node.  The members of a cell are in
        //    x order, so the chord's ends inside the end cells are bisections, and
        //    the slab's ten run side by side, as many steps as the largest staged
        //    cell needs: one after the other, each with its own loop, they took a
        //    fifth of the kernel waiting for LDS.
        int32_t lo[10], up[10];
        float key[5], rem[5];
        // distance from the node to the cell slab along z (staged cell t spans
        // [(t - 2) c, (t - 1) c) in brick-origin offsets)
        const float zlo = float(sz + dz - 2) * a.cell32, zhi = zlo + a.cell32;
        const float dzm = fz < zlo ? zlo - fz : (fz > zhi ? fz - zhi : 0.f);
#pragma unroll
        for (int y = 0; y < 5; ++y) {
          const int dy = y - 2;
          const float ylo = float(sy + dy - 2) * a.cell32, yhi = ylo + a.cell32;
          const float dym = fy < ylo ? ylo - fy : (fy > yhi ? fy - yhi : 0.f);
          const float rem2 = a.prune2 - (dzm * dzm + dym * dym);
          rem[y] = __builtin_sqrtf(rem2 < 0.f ? 0.f : rem2);
          int x0 = int(floorf((fx - rem[y]) * a.invCell32)) + 2, x1 = int(floorf((fx + rem[y]) * a.invCell32)) + 2;
          x0 = x0 < sx - 2 ? sx - 2 : x0;
          x1 = x1 > sx + 2 ? sx + 2 : x1;
          const bool any = rem2 >= 0.f && x0 <= x1;
          const int rowb = ((sz + dz) * kStageEdge + (sy + dy)) * kStageEdge;
          const int c0 = any ? rowb + x0 : 0, c1 = any ? rowb + x1 : 0;
          lo[y] = sOff[c0];
          up[y] = sOff[c0 + 1];
          lo[5 + y] = sOff[c1];
          up[5 + y] = any ? sOff[c1 + 1] : -1;     // (-1: no run)
          key[y] = fx - rem[y];
        }
        for (int st = 0; st < steps; ++st) {
          float x[10];
          int32_t mid[10];
#pragma unroll
          for (int q = 0; q < 10; ++q) {
            mid[q] = (lo[q] + up[q]) >> 1;
            x[q] = sCand[mid[q] < 0 ? 0 : mid[q]].x;
          }
#pragma unroll
          for (int q = 0; q < 10; ++q) {
            const bool before = q < 5 ? x[q] < key[q] : x[q] <= fx + rem[q - 5];
            const bool open = lo[q] < up[q];
            lo[q] = open && before ? mid[q] + 1 : lo[q];
            up[q] = open && !before ? mid[q] : up[q];
          }
        }
        int nr = 0, nCand = 0;
#pragma unroll
        for (int y = 0; y < 5; ++y) {
          const int32_t t0 = lo[y], t1 = up[5 + y] < 0 ? -1 : lo[5 + y];
          if (t1 > t0) {
            sRun[nr++ * BS + threadIdx.x] = uint32_t(4 * t0) | (uint32_t(4 * t1) << 16);
            nCand += t1 - t0;
          }
        }
        sRun[nr * BS + threadIdx.x] = uint32_t(4 * total);
        // 2. one walk over the slab's candidates: a wavefront iterates as often
        //    as its longest candidate list in the slab, not its longest run in
        //    every (dz, dy) row.  Candidates are read two ahead of their test (three
        //    register sets in rotation); the reader steps through the runs with
        //    no branch and, past the last one, stays on the sentinel run, the
        //    candidate that no node takes: a lane that has finished its list
        //    needs no test and no branch of its own.  (Runs hold 4 t: the byte
        //    offsets of the slots.)  Two thirds of the kernel's time issue VALU
        //    instructions, so the walk counts them: the row's state is one marker
        //    in its chunk buffer.  With the bisections side by side: 1.58 -> 1.50 ms
        //    at 128^3.  The rare paths (the exact FP64 test, ghost marks) are
        //    entered only when some lane of the wavefront needs them.
        // one instance of the walk with ghost marks and one without, chosen by
        // the block-uniform flag; another pair for the slab that holds the node
        auto walk = [&](auto marksOn, auto selfOn) {
          const uint32_t first = sRun[threadIdx.x];
          int32_t t = int32_t(first & 0xffffu), tEnd = int32_t(first >> 16);
          const int last = nr * BS + int(threadIdx.x);      // the sentinel
          int at = nr > 0 ? BS + int(threadIdx.x) : last;   // where nxt came from
          uint32_t nxt = sRun[at];
          auto advance = [&]() {
            const bool same = t + 4 < tEnd;
            const int next = at + BS < last ? at + BS : last;
            t = same ? t + 4 : int32_t(nxt & 0xffffu);
            tEnd = same ? tEnd : int32_t(nxt >> 16);
            at = same ? at : next;
            nxt = sRun[at];
          };
          auto read = [&](float4& c, int32_t& raw) {
            c = *static_cast<const float4*>(
                __builtin_assume_aligned(reinterpret_cast<const char*>(sCand) + 4 * t, 16));
            raw = *reinterpret_cast<const int32_t*>(reinterpret_cast<const char*>(sSlot) + t);
          };
          auto test = [&](const float4 cj, const int32_t raw) {
            const float rx = fx - cj.x, ry = fy - cj.y, rz = fz - cj.z;
            // FP32 estimate of min(h_i^2, h_j^2) |r|^2: fused products (any
            // rounding change stays inside the band that takes the exact test);
            // q min(a, b) = min(q a, q b) exactly for q >= 0, and positive floats
            // compare as their bits
            const float q = __builtin_fmaf(rz, rz, __builtin_fmaf(ry, ry, rx * rx));
            const int32_t wj = __float_as_int(cj.w);
            const float d = q * __int_as_float(wj < hi2 ? wj : hi2) - a.mid32;
            bool in = d < -a.half32;
            const bool band = fabsf(d) <= a.half32;
            const int32_t sj = raw & 0x7fffffff;
            if (__any(band)) {
              if (band) {
                const double* rj = rec + int64_t(sj) * R::STRIDE;
                in = exactIso(xi - rj[R::X], yi - rj[R::X + 1], zi - rj[R::X + 2], hi, rj[R::HINV], a.ext2);
              }
            }
            const bool acc = decltype(selfOn)::value ? in && sj != int32_t(k) : in;
            row.pushIf(acc, sj);
            if constexpr (decltype(marksOn)::value) {
              if (acc && raw < 0) a.keepSlot[sj] = 1;
            }
          };
          float4 c0, c1, c2;
          int32_t s0, s1, s2;
          read(c0, s0);
          advance();
          read(c1, s1);
          advance();
          for (int done = 3;; done += 3) {
            read(c2, s2);
            advance();
            test(c0, s0);
            read(c0, s0);
            advance();
            test(c1, s1);
            read(c1, s1);
            advance();
            test(c2, s2);
            if (!__any(done < nCand)) break;
          }
        };
        if (__any(nr > 0)) {
          if (marks) {
            if (dz != 0) walk(std::true_type{}, std::false_type{});
            else walk(std::true_type{}, std::true_type{});
          } else {
            if (dz != 0) walk(std::false_type{}, std::false_type{});
            else walk(std::false_type{}, std::true_type{});
          }
        }
      }
    } else {
      for (int dz = -2; dz <= 2; ++dz) {
        for (int dy = -2; dy <= 2; ++dy) {
          const int base = ((sz + dz) * kStageEdge + (sy + dy)) * kStageEdge + (sx - 2);
          for (int dx = 0; dx < 5; ++dx) {
            const int cidx = base + dx;
            const int32_t st = sStart[cidx], ncell = sOff[cidx + 1] - sOff[cidx];
            for (int32_t q2 = 0; q2 < ncell; ++q2) {
              const int32_t sj = st + q2;
              if (sj == int32_t(k)) continue;
              const double* rj = rec + int64_t(sj) * R::STRIDE;
              if (exactIso(xi - rj[R::X], yi - rj[R::X + 1], zi - rj[R::X + 2], hi, rj[R::HINV], a.ext2)) {
                row.pushIf(true, sj);
                if (a.keepSlot && rj[R::ORIG] >= double(a.nInt)) a.keepSlot[sj] = 1;
              }
            }
          }
        }
      }
    }
    const int32_t cnt = row.finish();
    rowCount[k] = cnt;
    stats.add(cnt);
  }
  stats.store(flags);
}

// ---------------------------------------------------------------------------
// Global search: any dimension, any H (cell edge = R, 3^nu stencil).
//
// Bound by the latency of its candidates' records: one after the other, a row took
// 50 us in 2-D and 400 us in 3-D however few rows there were.  L consecutive lanes
// walk a node's candidates in order, L at a time: the lanes that accept theirs
// append them at once, each at its place among them, so the row is the one that a
// single lane writes.  One lane to a node takes four candidates of a cell at a
// time and writes its row in chunks, which is less work where there are rows
// enough to fill the chip.
// ---------------------------------------------------------------------------
// Lanes to a node, by slots: the lines lie where the measured times cross (one by
// one as before / 1 / 4 / 16 lanes, us).
//   1-D 200 7.2 / 6.6 / 5.8 / 4.9, 2 k 9.4 / 8.6 / 4.3 / 3.4, 20 k 10.3 / 8.5 / 6.0 / 8.5,
//       100 k 21 / 12 / 16 / 30, 1 M 276 / 104 / 125 / 267
//   2-D 1 k 50 / 38 / 20 / 9, 10 k 54 / 42 / 19 / 14, 48 k 54 / 43 / 36 / 44,
//       250 k 128 / 92 / 142 / 171
//   3-D 1.7 k 432 / 313 / 132 / 48, 14 k 403 / 299 / 164 / 127, 33 k 405 / 303 / 279 / 219,
//       111 k 653 / 606 / 723 / 725
inline int searchLanes(int dim, int64_t slots) {
  if (slots > 65536) return 1;
  if (dim == 2) return slots <= 16384 ? 16 : 4;
  return dim == 1 ? 4 : 16;
}
template <int D, bool ISO, int L>
__device__ __forceinline__ int32_t searchRow(int64_t k, int sub, const double* __restrict__ rec,
                                             const int32_t* __restrict__ cellStart, const SearchArgs& a,
                                             const SegGrids& sg, int32_t* __restrict__ nbr) {
  using R = RL<ISO>;
  const double* ri_ = rec + k * R::STRIDE;
  const int64_t oi = int64_t(ri_[R::ORIG]);
  if (oi >= a.nInt) return 0;
  int ga = 0, gb = 1;
  if (sg.g) {
    const int m = sg.seg ? int(sg.seg[oi]) : 0;
    ga = sg.first[m];
    gb = sg.first[m + 1];
  }
  constexpr int NS = NSym<D>::value;
  auto loadH = [](const double* r) {
    S<D> H;
    if constexpr (ISO) {
      for (int c = 0; c < NS; ++c) H.c[c] = 0.0;
      for (int c = 0; c < D; ++c) H.c[sdiag<D>(c)] = r[RL<true>::HINV];
    } else {
      for (int c = 0; c < NS; ++c) H.c[c] = r[RL<false>::H + c];
    }
    return H;
  };
  V<D> ri;
  for (int c = 0; c < D; ++c) ri.c[c] = ri_[R::X + c];
  const S<D> Hi = loadH(ri_);
  // own search radius bound (only needed with several levels)
  double Ri = 0.0;
  if (gb - ga > 1) {
    if constexpr (ISO) Ri = a.ext / ri_[RL<true>::HINV] * (1.0 + 1.0e-6);
    else Ri = a.ext / gershgorinMin<D>(Hi.c) * (1.0 + 1.0e-6);
  }
  ChunkWriter row(reinterpret_cast<int4*>(nbr), a.n, k, a.cap);     // L = 1
  int32_t cnt = 0;
  const unsigned long long below = ((1ull << sub) - 1ull) << (threadIdx.x & 63 & ~(L - 1));
  const unsigned long long group = ((1ull << L) - 1ull) << (threadIdx.x & 63 & ~(L - 1));
  auto hit = [&](int32_t j) {
    const double* rj_ = rec + int64_t(j) * R::STRIDE;
    V<D> rij;
    for (int c = 0; c < D; ++c) rij.c[c] = ri.c[c] - rj_[R::X + c];
    double eta2i, eta2j;
    if constexpr (ISO) {
      // the products with zeros left out: the same sums for finite positions
      const double hi = Hi.c[0], hj = rj_[RL<true>::HINV];
      V<D> ei, ej;
      for (int c = 0; c < D; ++c) {
        ei.c[c] = hi * rij.c[c];
        ej.c[c] = hj * rij.c[c];
      }
      eta2i = vmag2(ei);
      eta2j = vmag2(ej);
    } else {
      eta2i = vmag2(sdot(Hi, rij));
      eta2j = vmag2(sdot(loadH(rj_), rij));
    }
    return (eta2i <= a.ext2) | (eta2j <= a.ext2);
  };
  auto append = [&](bool in, int32_t j) {
    const unsigned long long m = __ballot(in);
    if (in) {
      const int32_t at = cnt + __popcll(m & below);
      if (at < a.cap) nbr[ellIndex(at, a.n, k)] = j;
      if (a.keepSlot && rec[int64_t(j) * R::STRIDE + R::ORIG] >= double(a.nInt)) a.keepSlot[j] = 1;
    }
    cnt += __popcll(m & group);
  };
  for (int q = ga; q < gb; ++q) {
    const DGrid g = sg.g ? sg.g[q] : a.g;
    const int64_t base = sg.g ? sg.base[q] : 0;
    // cells that can hold a neighbour: the 3^nu stencil when the grid's cell
    // covers both radii (nodes of a grid have radius <= its cell), else every
    // cell within Ri
    int c0[3] = {0, 0, 0}, nc[3] = {1, 1, 1};
    {
      int cc[3];
      cellCoords<D>(g, ri.c, cc);
      for (int d = 0; d < D; ++d) {
        int c1;
        if (Ri <= g.cell) {
          c0[d] = cc[d] - 1 < 0 ? 0 : cc[d] - 1;
          c1 = cc[d] + 1 >= g.nc[d] ? g.nc[d] - 1 : cc[d] + 1;
        } else {
          const double t0 = floor((ri.c[d] - Ri - g.lo[d]) * g.invCell), t1 = floor((ri.c[d] + Ri - g.lo[d]) * g.invCell);
          c0[d] = t0 < 0.0 ? 0 : (t0 > double(g.nc[d] - 1) ? g.nc[d] - 1 : int(t0));
          c1 = t1 < 0.0 ? 0 : (t1 > double(g.nc[d] - 1) ? g.nc[d] - 1 : int(t1));
        }
        nc[d] = c1 - c0[d] + 1;
      }
    }
    if constexpr (L == 1) {
      // four candidates of a cell in flight together
      for (int z = 0; z < nc[2]; ++z)
        for (int y = 0; y < nc[1]; ++y)
          for (int x = 0; x < (D == 1 ? 1 : nc[0]); ++x) {
            const int64_t id = base + cellId<D>(g, c0[0] + x, c0[1] + y, c0[2] + z);
            const int32_t b = cellStart[id], e = cellStart[id + (D == 1 ? nc[0] : 1)];
            for (int32_t j = b; j < e; j += 4) {
              bool in[4];
#pragma unroll
              for (int t = 0; t < 4; ++t) {
                const bool is = j + t < e && j + t != k;
                const bool h = hit(is ? j + t : int32_t(k));
                in[t] = is && h;
              }
#pragma unroll
              for (int t = 0; t < 4; ++t) {
                row.pushIf(in[t], j + t);
                if (a.keepSlot && in[t] && rec[int64_t(j + t) * R::STRIDE + R::ORIG] >= double(a.nInt))
                  a.keepSlot[j + t] = 1;
              }
            }
          }
      continue;
    }
    // 1-D cells follow each other in slot order: one range.  Else the lanes load
    // the bounds of L cells (x fastest) and take them three at a time, the first
    // L candidates of each in flight together.
    const uint32_t cells = D == 1 ? 1u : uint32_t(nc[0]) * uint32_t(nc[1]) * uint32_t(nc[2]);   // below 2^31
    for (uint32_t m0 = 0; m0 < cells; m0 += L) {
      const uint32_t m = m0 + sub;
      int32_t b = 0, e = 0;
      if (m < cells) {
        const uint32_t row = D == 1 ? 0u : m / uint32_t(nc[0]), mx = D == 1 ? 0u : m - row * uint32_t(nc[0]);
        const uint32_t mz = D == 3 ? row / uint32_t(nc[1]) : 0u, my = row - mz * uint32_t(nc[1]);
        const int64_t id = base + cellId<D>(g, c0[0] + int(mx), c0[1] + int(my), c0[2] + int(mz));
        b = cellStart[id];
        e = cellStart[id + (D == 1 ? nc[0] : 1)];
      }
      const int here = cells - m0 < L ? int(cells - m0) : L;
      constexpr int T = D == 1 ? 1 : 3;
      for (int c = 0; c < here; c += T) {
        int32_t j[T], end[T];
        bool in[T];
#pragma unroll
        for (int t = 0; t < T; ++t) {
          const bool cell = c + t < here;
          j[t] = __shfl(b, cell ? c + t : c, L) + sub;
          end[t] = cell ? __shfl(e, cell ? c + t : c, L) : 0;
          const bool is = j[t] < end[t] && j[t] != k;
          const bool h = hit(is ? j[t] : int32_t(k));
          in[t] = is && h;
        }
#pragma unroll
        for (int t = 0; t < T; ++t) {
          append(in[t], j[t]);
          for (int32_t j0 = j[t] - sub + L; j0 < end[t]; j0 += L) {
            const int32_t jn = j0 + sub;
            const bool is = jn < end[t] && jn != k;
            const bool h = hit(is ? jn : int32_t(k));
            append(is && h, jn);
          }
        }
      }
    }
  }
  if constexpr (L == 1) return row.finish();
  // the rest of the last chunk
  if (sub < (-cnt & 3) && cnt + sub < a.cap) nbr[ellIndex(cnt + sub, a.n, k)] = 0;
  return cnt;
}
template <int D, bool ISO, int L>
__global__ void __launch_bounds__(kBlock) k_search_global(const double* __restrict__ rec,
                                                          const int32_t* __restrict__ cellStart, SearchArgs a,
                                                          SegGrids sg, int32_t* __restrict__ rowCount,
                                                          int32_t* __restrict__ nbr, int32_t* __restrict__ flags) {
  const int64_t k = (xcdBlock((a.n * L + kBlock - 1) / kBlock) * kBlock + threadIdx.x) / L;
  const int sub = threadIdx.x % L;
  RowStats<> stats;
  if (k < a.n) {
    const int32_t c = searchRow<D, ISO, L>(k, sub, rec, cellStart, a, sg, nbr);
    if (sub == 0) {
      rowCount[k] = c;
      stats.add(c);
    }
  }
  stats.store(flags);
}

// Internal slots in slot order: the work list of the density and pair passes
// (scan.hh).
struct WorkScan {
  static constexpr bool kCompact = true;
  const int32_t* perm;
  int32_t* work;
  int64_t nInt;
  __device__ int32_t value(int64_t k) const {
    const int32_t i = perm[k];
    return i >= 0 && i < nInt ? 1 : 0;
  }
  __device__ void emit(int64_t k, int32_t prefix, int32_t) const { work[prefix] = int32_t(k); }
  __device__ void total(int32_t) const {}
};

// ---------------------------------------------------------------------------
// Reference row order: sort each row by caller index.  One wavefront per row,
// K keys per lane (rows up to 256 entries), bitonic network in registers;
// longer rows are sorted by a single lane.
// ---------------------------------------------------------------------------
// The value of lane ^ M: a DPP move within rows of 16 lanes, an LDS swizzle within
// 32, else a permute.
template <int M> __device__ __forceinline__ int32_t xorLane(int32_t v) {
  if constexpr (M == 1) return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xf, 0xf, true);          // quad_perm 1 0 3 2
  else if constexpr (M == 2) return __builtin_amdgcn_mov_dpp(v, 0x4E, 0xf, 0xf, true);     // quad_perm 2 3 0 1
  else if constexpr (M == 3) return __builtin_amdgcn_mov_dpp(v, 0x1B, 0xf, 0xf, true);     // quad_perm 3 2 1 0
  else if constexpr (M == 7) return __builtin_amdgcn_mov_dpp(v, 0x141, 0xf, 0xf, true);    // row_half_mirror
  else if constexpr (M == 8) return __builtin_amdgcn_mov_dpp(v, 0x128, 0xf, 0xf, true);    // row_ror 8
  else if constexpr (M == 15) return __builtin_amdgcn_mov_dpp(v, 0x140, 0xf, 0xf, true);   // row_mirror
  else if constexpr (M < 32) return __builtin_amdgcn_ds_swizzle(v, (M << 10) | 0x1f);
  else return __shfl_xor(v, M);
}
template <int M> __device__ __forceinline__ int64_t xorLane(int64_t v) {
  const int32_t lo = xorLane<M>(int32_t(v)), hi = xorLane<M>(int32_t(v >> 32));
  return (int64_t(hi) << 32) | int64_t(uint32_t(lo));
}
// Sorts the K keys a lane of the wavefront, element q * 64 + lane, ascending.  Every
// merge starts with the mirrored partner, so all exchanges keep the smaller key
// below and a step is a lane move, min, max and one select on one of six masks; the
// directions of the textbook network, formed again at each step, and its permutes
// took twice the instructions (what is left is the gather of the callers and slots:
// 82 k rows of 115 entries 49 -> 40 us).
template <int K, int M, typename T>
__device__ __forceinline__ void exchange(T (&key)[K], bool lower) {
#pragma unroll
  for (int q = 0; q < K; ++q) {
    const T other = xorLane<M>(key[q]);
    const T mn = key[q] < other ? key[q] : other, mx = key[q] < other ? other : key[q];
    key[q] = lower ? mn : mx;
  }
}
template <int K, typename T>
__device__ __forceinline__ void waveBitonic(T (&key)[K], int lane) {
  const bool l1 = (lane & 1) == 0, l2 = (lane & 2) == 0, l4 = (lane & 4) == 0, l8 = (lane & 8) == 0,
             l16 = (lane & 16) == 0, l32 = (lane & 32) == 0;
  auto from1 = [&] { exchange<K, 1>(key, l1); };
  auto from2 = [&] { exchange<K, 2>(key, l2); from1(); };
  auto from4 = [&] { exchange<K, 4>(key, l4); from2(); };
  auto from8 = [&] { exchange<K, 8>(key, l8); from4(); };
  auto from16 = [&] { exchange<K, 16>(key, l16); from8(); };
  auto from32 = [&] { exchange<K, 32>(key, l32); from16(); };
  exchange<K, 1>(key, l1);
  exchange<K, 3>(key, l2);
  from1();
  exchange<K, 7>(key, l4);
  from2();
  exchange<K, 15>(key, l8);
  from4();
  exchange<K, 31>(key, l16);
  from8();
  exchange<K, 63>(key, l32);
  from16();
#pragma unroll
  for (int half = 1; half < K; half <<= 1) {      // merges of 2 half x 64 elements
    T mirror[K];
#pragma unroll
    for (int q = 0; q < K; ++q) mirror[q] = xorLane<63>(key[q]);
#pragma unroll
    for (int q = 0; q < K; ++q) {
      const T other = mirror[q ^ (2 * half - 1)];
      const bool less = key[q] < other;
      key[q] = ((q & half) == 0) == less ? key[q] : other;
    }
#pragma unroll
    for (int d = half >> 1; d > 0; d >>= 1)
#pragma unroll
      for (int q = 0; q < K; ++q)
        if ((q & d) == 0) {
          const T a = key[q], b = key[q ^ d];
          key[q] = a < b ? a : b;
          key[q ^ d] = a < b ? b : a;
        }
    from32();
  }
}

template <int K>
__device__ void sortRowWave(int32_t* __restrict__ nbr, int64_t n, int64_t k, int len, const int32_t* __restrict__ perm,
                            const int32_t* __restrict__ iperm, int lane) {
  int32_t key[K];
#pragma unroll
  for (int q = 0; q < K; ++q) {
    const int e = q * 64 + lane;
    key[q] = e < len ? perm[nbr[ellIndex(e, n, k)]] : 0x7fffffff;
  }
  waveBitonic<K>(key, lane);
#pragma unroll
  for (int q = 0; q < K; ++q) {
    const int e = q * 64 + lane;
    if (e < len) nbr[ellIndex(e, n, k)] = iperm[key[q]];
  }
}

// Several NodeLists: the order in which the reference's scatter delivers node
// x's pair terms (calculatePairInteraction, ConnectivityMapInline.hh:169-186):
// first the internal neighbours that own their pair (lower caller index, in
// that order), then x's own pairs in ConnectivityMap order, by (NodeList,
// index within the NodeList), a NodeList's ghosts after its internal nodes.
// With one NodeList this is ascending caller index.
// mapOrder: ConnectivityMap's own order, by (NodeList, index within the
// NodeList), for the loops that walk a node's full connectivity
// (iterateIdealH.cc:164-205) rather than receive from owners.
__device__ __forceinline__ int64_t receiveKey(int32_t c, int32_t x, const double* __restrict__ seg, int64_t nInt,
                                              bool mapOrder) {
  if (!mapOrder && c < nInt && c < x) return int64_t(c);
  const int64_t local = c < nInt ? int64_t(c) : (int64_t(1) << 31) + c;
  return (int64_t(1) << 62) | (int64_t(seg[c]) << 32) | local;
}
__device__ __forceinline__ int32_t callerOfKey(int64_t key) {
  if (key < (int64_t(1) << 62)) return int32_t(key);
  const int64_t low = key & 0xffffffffll;
  return int32_t(low >= (int64_t(1) << 31) ? low - (int64_t(1) << 31) : low);
}
template <int K>
__device__ void sortRowWaveLists(int32_t* __restrict__ nbr, int64_t n, int64_t k, int len,
                                 const int32_t* __restrict__ perm, const int32_t* __restrict__ iperm,
                                 const double* __restrict__ seg, int64_t nInt, bool mapOrder, int lane) {
  const int32_t x = perm[k];
  int64_t key[K];
#pragma unroll
  for (int q = 0; q < K; ++q) {
    const int e = q * 64 + lane;
    key[q] = e < len ? receiveKey(perm[nbr[ellIndex(e, n, k)]], x, seg, nInt, mapOrder) : INT64_MAX;
  }
  waveBitonic<K>(key, lane);
#pragma unroll
  for (int q = 0; q < K; ++q) {
    const int e = q * 64 + lane;
    if (e < len) nbr[ellIndex(e, n, k)] = iperm[callerOfKey(key[q])];
  }
}

__global__ void __launch_bounds__(kBlock) k_row_sort(const int32_t* __restrict__ rowCount, int32_t* __restrict__ nbr,
                                                    int64_t n, const int32_t* __restrict__ perm,
                                                    const int32_t* __restrict__ iperm,
                                                    const double* __restrict__ seg, int64_t nInt, int mapOrder) {
  const int lane = threadIdx.x & 63;
  const int64_t k = (blockIdx.x * int64_t(blockDim.x) + threadIdx.x) >> 6;
  if (k >= n) return;                              // uniform per wavefront
  const int len = rowCount[k];
  if (len <= 1) return;
  if (seg) {
    const bool mo = mapOrder != 0;
    if (len <= 64) sortRowWaveLists<1>(nbr, n, k, len, perm, iperm, seg, nInt, mo, lane);
    else if (len <= 128) sortRowWaveLists<2>(nbr, n, k, len, perm, iperm, seg, nInt, mo, lane);
    else if (len <= 256) sortRowWaveLists<4>(nbr, n, k, len, perm, iperm, seg, nInt, mo, lane);
    else if (lane == 0) {
      const int32_t x = perm[k];
      for (int a2 = 1; a2 < len; ++a2) {
        const int32_t v = nbr[ellIndex(a2, n, k)];
        const int64_t pv = receiveKey(perm[v], x, seg, nInt, mo);
        int q = a2 - 1;
        while (q >= 0 && receiveKey(perm[nbr[ellIndex(q, n, k)]], x, seg, nInt, mo) > pv) {
          nbr[ellIndex(q + 1, n, k)] = nbr[ellIndex(q, n, k)];
          --q;
        }
        nbr[ellIndex(q + 1, n, k)] = v;
      }
    }
    return;
  }
  if (len <= 64) sortRowWave<1>(nbr, n, k, len, perm, iperm, lane);
  else if (len <= 128) sortRowWave<2>(nbr, n, k, len, perm, iperm, lane);
  else if (len <= 256) sortRowWave<4>(nbr, n, k, len, perm, iperm, lane);
  else if (lane == 0) {
    for (int a2 = 1; a2 < len; ++a2) {
      const int32_t v = nbr[ellIndex(a2, n, k)];
      const int32_t pv = perm[v];
      int q = a2 - 1;
      while (q >= 0 && perm[nbr[ellIndex(q, n, k)]] > pv) { nbr[ellIndex(q + 1, n, k)] = nbr[ellIndex(q, n, k)]; --q; }
      nbr[ellIndex(q + 1, n, k)] = v;
    }
  }
}

// ---- zeroing several int32 buffers in one dispatch ------------------------
__global__ void k_zero_many(ZeroSet z) {
  const int64_t stride = int64_t(gridDim.x) * blockDim.x;
  for (int q = 0; q < z.m; ++q)
    for (int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < z.n[q]; i += stride) z.p[q][i] = 0;
  for (int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < z.words; i += stride)
    z.to[i] = __hip_atomic_load(z.from + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);   // host memory, written anew
}

// A grid of cell edge `cell` over the bounds hb: cells per axis, bricks, cell count.
template <int D>
void gridWithCell(const double* hb, double cell, Grid& G, DGrid& dg, int64_t& bricks) {
  G.cell = cell;
  dg = DGrid{};
  dg.cell = cell;
  dg.invCell = 1.0 / cell;
  bricks = 1;
  const int bw = (D == 1) ? 1 : 4;
  for (int k = 0; k < 3; ++k) {
    G.lo[k] = k < D ? hb[k] : 0.0;
    G.nc[k] = k < D ? int(std::floor((hb[3 + k] - hb[k]) / cell)) + 1 : 1;
    G.nb[k] = k < D ? (G.nc[k] + bw - 1) / bw : 1;
    dg.lo[k] = G.lo[k]; dg.nc[k] = G.nc[k]; dg.nb[k] = G.nb[k];
    if (k < D) bricks *= G.nb[k];
  }
  G.ncells = (D == 1) ? int64_t(G.nc[0]) : bricks * (D == 2 ? 16 : 64);
  SG_REQUIRE(G.ncells < (int64_t(1) << 31) - 2, SPHGPU_ERR_CAPACITY, "neighbour grid too large");
}

// Search grid from the bounds hb (k_bounds layout).  Staged path: cells of
// edge R/2 (5^3 stencil).  Global path: cells of edge >= R (3^nu stencil),
// enlarged if the grid would be too fine.
template <int D>
void gridFromBounds(const double* hb, double ext, bool allowStaged, Grid& G, DGrid& dg, int64_t& bricks,
                    bool& stagedPath) {
  requireUsableBounds(hb);
  const double R = ext / hb[6] * (1.0 + 1.0e-6);
  double spanX = 0.0;
  for (int k = 0; k < D; ++k) spanX = std::max(spanX, hb[3 + k] - hb[k]);
  const int maxCells = D == 3 ? 1024 : (D == 2 ? 32768 : (1 << 26));
  stagedPath = (D == 3) && allowStaged;
  double cell = 0.5 * R * (1.0 + 1.0e-9);
  if (stagedPath && spanX / cell > maxCells - 2) stagedPath = false;
  if (!stagedPath) {
    cell = R * (1.0 + 1.0e-9);
    if (spanX / cell > maxCells - 2) cell = spanX / (maxCells - 2);
  }
  G.span = stagedPath ? 2 : 1;
  G.R2 = R * R;
  gridWithCell<D>(hb, cell, G, dg, bricks);
}

// Levels of a node set whose search radii span more than a factor 2: cells
// of edge Rmin 2^L (>= R at the top level), each grid enlarged if too fine.
// One grid when the radii are within a factor 2.
template <int D>
void levelGrids(const double* hb, double ext, std::vector<DGrid>& out, std::vector<int64_t>& cells) {
  requireUsableBounds(hb);
  const double R = ext / hb[6] * (1.0 + 1.0e-6);
  const double Rmin = ext / hb[9] * (1.0 + 1.0e-6);
  Grid G;
  DGrid dg;
  int64_t bricks;
  if (!(R > 2.0 * Rmin)) {
    bool staged;
    gridFromBounds<D>(hb, ext, false, G, dg, bricks, staged);
    out.push_back(dg);
    cells.push_back(G.ncells);
    return;
  }
  double spanX = 0.0;
  for (int k = 0; k < D; ++k) spanX = std::max(spanX, hb[3 + k] - hb[k]);
  const int maxCells = D == 3 ? 1024 : (D == 2 ? 32768 : (1 << 26));
  double c = Rmin * (1.0 + 1.0e-9);
  for (int L = 0; L < 40; ++L) {
    const bool top = c >= R * (1.0 + 1.0e-9);
    double cell = c;
    if (spanX / cell > maxCells - 2) cell = spanX / (maxCells - 2);
    gridWithCell<D>(hb, cell, G, dg, bricks);
    out.push_back(dg);
    cells.push_back(G.ncells);
    if (top) break;
    c *= 2.0;
  }
}

// Grid lists to the device, with the kernel that runs z; returns the total cell
// count.
int64_t uploadGrids(Sim& s, const std::vector<DGrid>& grids, const std::vector<int64_t>& cells,
                    const std::vector<int32_t>& first, ZeroSet& z) {
  const size_t ng = grids.size();
  std::vector<int64_t> base(ng + 1, 0);
  for (size_t q = 0; q < ng; ++q) base[q + 1] = base[q] + cells[q];
  SG_REQUIRE(base.back() < (int64_t(1) << 31) - 2, SPHGPU_ERR_CAPACITY, "neighbour grid too large");
  // the grids, their first global cells and each member's first grid in one
  // buffer, staged in pinned memory at the same offsets and read from there by the
  // zeroing kernel: a copy of a few KB and the event behind it were 15 us of a step
  // that takes 200.  The build's own wait frees the staging.
  const size_t bG = sizeof(DGrid) * ng, bB = sizeof(int64_t) * (ng + 1), bF = sizeof(int32_t) * first.size();
  const size_t oB = (bG + 63) / 64 * 64, oF = oB + (bB + 63) / 64 * 64;
  const size_t bytes = (oF + bF + 3) / 4 * 4;
  s.segGrid.ensure(bytes);
  char* d = static_cast<char*>(s.segGrid.p);
  s.gridList = d;
  s.gridCellBase = reinterpret_cast<int64_t*>(d + oB);
  s.gridFirst = reinterpret_cast<int32_t*>(d + oF);
  char* h = static_cast<char*>(hostStaging(s, 1, bytes));
  std::memcpy(h, grids.data(), bG);
  std::memcpy(h + oB, base.data(), bB);
  std::memcpy(h + oF, first.data(), bF);
  z.from = reinterpret_cast<const uint32_t*>(h);
  z.to = reinterpret_cast<uint32_t*>(d);
  z.words = int64_t(bytes / 4);
  s.pinnedInBusy = true;
  return base.back();
}

template <int D, bool XKEY>
void cellOrder(Sim& s, int64_t n) {
  // the records the next kernel reads, written with the FP64 record: the
  // caller's hint, else the density sum's
  const int sec = s.isotropic ? (s.buildRecHint >= 0 ? s.buildRecHint : densityRecordSec(s)) : 0;
  PackOut o = packOutputs(s, sec);
  if (s.buildVel) {
    s.velS.ensure(sizeof(double) * size_t(velStride(D)) * size_t(n));
    o.vel = s.velS.as<double>();
  }
  const PackIn in = packInputs(s);
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(nblocks(n)), dim3(kBlock), 0, s.stream, s.cellOf.as<int32_t>(),
                       s.cellStart.as<int32_t>(), s.cellMembers.as<int32_t>(), s.xs.as<double>(), n,
                       s.perm.as<int32_t>(), s.iperm.as<int32_t>(), in, o);
  };
  if (!s.isotropic) {
    go(k_cell_order<D, false, 0, XKEY>);
  } else {
    switch (sec) {
      case 0: go(k_cell_order<D, true, 0, XKEY>); break;
      case 1: go(k_cell_order<D, true, 1, XKEY>); break;
      case 2: go(k_cell_order<D, true, 2, XKEY>); break;
      case 4: go(k_cell_order<D, true, 4, XKEY>); break;
      case 8: go(k_cell_order<D, true, 8, XKEY>); break;
      default: SG_REQUIRE(false, SPHGPU_ERR_STATE, "unsupported record kinds for the neighbour build");
    }
  }
  SG_CHECK_HIP(hipGetLastError());
  s.recValid = true;
}

template <int D>
void buildNeighborsD(Sim& s, double ext) {
  hipStream_t st = s.stream;
  SG_CHECK_HIP(hipEventRecord(s.ev[0], st));
  // rows: those the caller set, or a ghost generation's whose count is still
  // on the device (read back with the bounds)
  ZeroSet z{};
  const bool pending = s.genPending;
  s.genPending = false;
  const int64_t rows = pending ? s.genCap : s.nTot;
  const int nGen = pending ? int(s.subs.size()) + 2 : 0;
  const int64_t* gen = pending ? s.genDev.as<int64_t>() : nullptr;
  const int64_t* nDev = pending ? gen + nGen - 1 : nullptr;

  // 1. bounds
  Grid& G = s.grid;
  DGrid dg{};
  int64_t bricks = 1;
  bool stagedPath = false;
  double hb[kNB];
  SegGrids sgr{nullptr, nullptr, nullptr, nullptr, ext};
  if (s.nSeg > 0) {
    const int ns = s.nSeg;
    const size_t nbits = size_t(ns) * kNB;
    unsigned long long* next = nullptr;
    unsigned long long* bits = s.segBoundsBits.take(nbits, st, next);
    // one group a wavefront until every SIMD has one
    const int groups = int(std::min<int64_t>(kSegGroups, std::max<int64_t>(1, rows / (64 * 1024))));
    hipLaunchKernelGGL((k_seg_bounds<D>), dim3(nblocks((rows + groups - 1) / groups)), dim3(kBlock), 0, st,
                       s.pos.as<double>(), s.H.as<double>(), s.seg.as<double>(), rows, nDev, groups, bits, next,
                       int(nbits));
    unsigned long long* hbits = static_cast<unsigned long long*>(
        hostStaging(s, 0, (nbits + size_t(nGen)) * sizeof(unsigned long long)));
    int64_t* hgen = reinterpret_cast<int64_t*>(hbits + nbits);
    hipLaunchKernelGGL(k_report, dim3(nblocks(std::max<int64_t>(int64_t(nbits), nGen))), dim3(kBlock), 0, st, bits,
                       int(nbits), hbits, gen, nGen, hgen);
    SG_CHECK_HIP(hipGetLastError());
    SG_CHECK_HIP(hipStreamSynchronize(st));
    if (pending) finishGeneration(s, hgen);
    // back to min slots as such
    for (size_t q = 0; q < nbits; ++q)
      if (!isMaxSlot(int(q % kNB))) hbits[q] = ~hbits[q];
    std::vector<DGrid> grids;
    std::vector<int64_t> cells;
    std::vector<int32_t> first(size_t(ns) + 1, 0);
    // a member with a non-finite position or H (or no positive bound of its
    // H) fails alone: the step is abandoned before anything of it is kept,
    // and the caller evicts the member and steps the others
    MemberFailure bad;
    for (int m = 0; m < ns; ++m) {
      double hm[kNB];
      for (int k = 0; k < kNB; ++k) hm[k] = fromOrderedBits(hbits[size_t(m) * kNB + k]);
      const int u = boundsUsable(hm);
      if (u <= 0) bad.add(m, u == 0 ? SPHGPU_MEMBER_NONFINITE : SPHGPU_MEMBER_BAD_H);
    }
    if (!bad.members.empty()) throw bad;
    bool iso = true;
    double absMax = 0.0;
    for (int m = 0; m < ns; ++m) {
      double hm[kNB];
      for (int k = 0; k < kNB; ++k) hm[k] = fromOrderedBits(hbits[size_t(m) * kNB + k]);
      for (int k = 0; k < D; ++k) absMax = std::max(absMax, std::max(std::fabs(hm[k]), std::fabs(hm[3 + k])));
      iso = iso && hm[7] > 0.5;
      levelGrids<D>(hm, ext, grids, cells);
      first[size_t(m) + 1] = int32_t(grids.size());
      if (m == 0) for (int k = 0; k < kNB; ++k) hb[k] = hm[k];
      hb[6] = std::min(hb[6], hm[6]);
      hb[8] = std::max(hb[8], hm[8]);
    }
    s.isotropic = iso && !s.hasMultipliers;
    s.rMax = ext / hb[6];
    s.posAbsMax = absMax;
    G = Grid{};
    G.ncells = uploadGrids(s, grids, cells, first, z);
    sgr = SegGrids{s.seg.as<double>(), static_cast<const DGrid*>(s.gridList), s.gridCellBase, s.gridFirst, ext};
  } else {
    const int nbB = int(std::min<int64_t>(1024, nblocks(rows)));
    s.reduceTmp.ensure(sizeof(double) * (size_t(nbB) * kNB + 16));
    const bool onHost = nbB <= kBoundsHost;
    const int parts = onHost ? std::max(nbB, 1) : 1;
    double* hbp = static_cast<double*>(
        hostStaging(s, 0, sizeof(double) * kNB * size_t(parts) + sizeof(int64_t) * size_t(nGen)));
    int64_t* hgen = reinterpret_cast<int64_t*>(hbp + kNB * parts);
    double* partials = onHost ? hbp : s.reduceTmp.as<double>();
    hipLaunchKernelGGL((k_bounds<D>), dim3(nbB), dim3(kBlock), 0, st, s.pos.as<double>(), s.H.as<double>(), rows, nDev,
                       partials, gen, nGen, onHost ? hgen : nullptr);
    if (!onHost)
      hipLaunchKernelGGL(k_bounds_final, dim3(1), dim3(kBlock), 0, st, partials, nbB, hbp, gen, nGen, hgen);
    SG_CHECK_HIP(hipGetLastError());
    SG_CHECK_HIP(hipStreamSynchronize(st));
    if (pending) finishGeneration(s, hgen);
    std::memcpy(hb, hbp, sizeof(hb));
    for (int b = 1; b < parts; ++b)
      for (int k = 0; k < kNB; ++k) {
        const double v = hbp[b * kNB + k];
        hb[k] = isMaxSlot(k) ? std::max(hb[k], v) : std::min(hb[k], v);
      }
    requireUsableBounds(hb);
    s.isotropic = hb[7] > 0.5 && !s.hasMultipliers;
    s.rMax = ext / hb[6];
    s.posAbsMax = 0.0;
    for (int k = 0; k < D; ++k) s.posAbsMax = std::max(s.posAbsMax, std::max(std::fabs(hb[k]), std::fabs(hb[3 + k])));
    std::vector<DGrid> grids;
    std::vector<int64_t> cells;
    levelGrids<D>(hb, ext, grids, cells);
    if (grids.size() == 1) {
      gridFromBounds<D>(hb, ext, s.isotropic, G, dg, bricks, stagedPath);
    } else {
      // smoothing scales spanning more than a factor 2: levels
      std::vector<int32_t> first = {0, int32_t(grids.size())};
      G = Grid{};
      G.ncells = uploadGrids(s, grids, cells, first, z);
      sgr = SegGrids{nullptr, static_cast<const DGrid*>(s.gridList), s.gridCellBase, s.gridFirst, ext};
    }
  }

  const int64_t n = s.nTot;
  // 2. counting sort by cell, then by node index (staged search: by x) inside a cell
  s.cellOf.ensure(sizeof(int32_t) * size_t(n));
  s.cellCount.ensure(sizeof(int32_t) * size_t(G.ncells + 1));
  s.cellRank.ensure(sizeof(int32_t) * size_t(n));
  s.cellMembers.ensure(sizeof(int32_t) * size_t(n));
  if (stagedPath) s.xs.ensure(sizeof(double) * size_t(n));
  s.cellStart.ensure(sizeof(int32_t) * size_t(G.ncells + 2));
  s.perm.ensure(sizeof(int32_t) * size_t(n));
  s.iperm.ensure(sizeof(int32_t) * size_t(n));
  // zero the cell counters, the search flags and the ghost-use marks in one dispatch
  const bool markUse = s.markGhostUse && s.nTot > s.nInt;
  if (markUse) s.slotKeep.ensure(sizeof(int32_t) * size_t(n + 1));
  s.flags.ensure(sizeof(int32_t) * kSearchFlags);
  z.add(s.cellCount.as<int32_t>(), G.ncells + 1);
  z.add(s.flags.as<int32_t>(), kSearchFlags);
  if (markUse) z.add(s.slotKeep.as<int32_t>(), n);
  zeroMany(z, s.stream);
  hipLaunchKernelGGL((k_cell_count<D>), dim3(nblocks(n)), dim3(kBlock), 0, st, s.pos.as<double>(), s.H.as<double>(),
                     n, dg, sgr, s.cellOf.as<int32_t>(), s.cellCount.as<int32_t>(), s.cellRank.as<int32_t>());
  scanItems(CellScan{s.cellCount.as<int32_t>(), s.cellStart.as<int32_t>(), G.ncells}, G.ncells, s.scanTmp, st);
  hipLaunchKernelGGL(k_cell_scatter, dim3(nblocks(n)), dim3(kBlock), 0, st, s.cellOf.as<int32_t>(),
                     s.cellStart.as<int32_t>(), s.cellRank.as<int32_t>(), s.cellMembers.as<int32_t>(), n,
                     s.pos.as<double>(), D, stagedPath ? s.xs.as<double>() : nullptr);
  SG_CHECK_HIP(hipGetLastError());
  s.nSlots = n;
  // the staged search cuts each row of cells to the chord of its sphere by x
  if constexpr (D == 3) {
    if (stagedPath) cellOrder<D, true>(s, n);
    else cellOrder<D, false>(s, n);
  } else {
    cellOrder<D, false>(s, n);
  }

  // 3. rows
  SearchArgs sa{};
  sa.g = dg;
  sa.ext = ext;
  sa.ext2 = ext * ext;
  // FP32 classification band.  Offsets from the brick origin are at most 3R, so
  // |r| carries an absolute error below 7.2e-7 R; near the threshold of the
  // smallest smoothing scale (|r| = ext/hmax_inv >= R*hinv_min/hinv_max) that is
  // a relative error of 1.44e-6*ratio in |r|^2, plus ~5e-7 from the FP32
  // products.  The band is four times that, and never narrower than 1e-5.
  const double ratio = hb[8] / hb[6];
  const double band = std::max(1.0e-5, 4.0 * (1.44e-6 * ratio + 5.0e-7));
  sa.mid32 = float(sa.ext2);
  sa.half32 = float(sa.ext2 * band);
  {
    const double Rm = ext / hb[6] * (1.0 + 1.0e-6) * (1.0 + 1.0e-4);
    sa.prune2 = float(Rm * Rm);
    sa.cell32 = float(dg.cell);
    sa.invCell32 = float(1.0 / dg.cell);
  }
  sa.n = n;
  sa.nInt = s.nInt;
  sa.keepSlot = nullptr;
  if (markUse) sa.keepSlot = s.slotKeep.as<int32_t>();
  if (s.ellCap <= 0) s.ellCap = D == 3 ? 160 : (D == 2 ? 48 : 16);
  s.rowCount.ensure(sizeof(int32_t) * size_t(n));
  for (int attempt = 0; attempt < 2; ++attempt) {
    sa.cap = s.ellCap;
    s.nbr.ensure(ellBytes(n, s.ellCap));
    if (attempt > 0) {
      // the first attempt's flags were zeroed with the cell counters; ghost
      // marks of the first attempt are a subset of the second's
      ZeroSet again{};
      again.add(s.flags.as<int32_t>(), kSearchFlags);
      zeroMany(again, s.stream);
    }
    if (stagedPath) {
      auto staged = [&](auto kern, int bs) {
        hipLaunchKernelGGL(kern, dim3(int(xcdGrid(bricks))), dim3(bs), 0, st, s.rec.as<double>(),
                           s.cellStart.as<int32_t>(), sa, s.rowCount.as<int32_t>(), s.nbr.as<int4>(),
                           s.flags.as<int32_t>());
      };
      if (bricks <= kWideBricks) staged(k_search_staged<kWideBlock>, kWideBlock);
      else staged(k_search_staged<kBlock>, kBlock);
    } else {
      auto global = [&](auto kern, int L) {
        hipLaunchKernelGGL(kern, dim3(int(xcdGrid(nblocks(n * L)))), dim3(kBlock), 0, st, s.rec.as<double>(),
                           s.cellStart.as<int32_t>(), sa, sgr, s.rowCount.as<int32_t>(), s.nbr.as<int32_t>(),
                           s.flags.as<int32_t>());
      };
      auto lanes = [&](auto ln) {
        constexpr int L = decltype(ln)::value;
        if (s.isotropic) global(k_search_global<D, true, L>, L);
        else global(k_search_global<D, false, L>, L);
      };
      const int L = searchLanes(D, n);
      if (L == 1) lanes(std::integral_constant<int, 1>{});
      else if (D < 3 && L == 4) lanes(std::integral_constant<int, (D < 3 ? 4 : 16)>{});
      else lanes(std::integral_constant<int, (D > 1 ? 16 : 4)>{});
    }
    SG_CHECK_HIP(hipGetLastError());
    // pinned: the folded flags, the cull's starts; or the flags as they are
    const size_t raw = sizeof(int32_t) * kSearchFlags;
    char* hp = static_cast<char*>(
        hostStaging(s, 0, std::max(raw, sizeof(SearchFlags) + sizeof(int32_t) * (s.subs.size() + 1))));
    int32_t* hcull = reinterpret_cast<int32_t*>(hp + sizeof(SearchFlags));
    // the ghost cull's first half rides on the same wait and brings the flags along
    if (markUse) cullLaunch(s, reinterpret_cast<SearchFlags*>(hp), hcull);
    else SG_CHECK_HIP(hipMemcpyAsync(hp, s.flags.p, raw, hipMemcpyDeviceToHost, st));
    SG_CHECK_HIP(hipStreamSynchronize(st));
    s.pinnedInBusy = false;
    const SearchFlags hf = markUse ? *reinterpret_cast<const SearchFlags*>(hp)
                                   : foldFlags(reinterpret_cast<const int32_t*>(hp));
    if (markUse) {
      s.cullStarts.assign(hcull, hcull + s.subs.size() + 1);
      s.cullStartsReady = true;
    }
    s.maxRow = hf.longest;
    s.stagedFallbacks = hf.fallbacks;
    s.nEntries = int64_t(hf.entries);
    if (s.maxRow <= s.ellCap) break;
    SG_REQUIRE(attempt == 0, SPHGPU_ERR_CAPACITY, "neighbour row capacity exceeded twice");
    s.ellCap = ((s.maxRow + 15) / 16) * 16 + 16;
  }
  // 4. reference row order
  if (s.rowOrder == SPHGPU_ROW_ORDER_REFERENCE && n > 0)
    hipLaunchKernelGGL(k_row_sort, dim3(nblocks(n * 64)), dim3(kBlock), 0, st, s.rowCount.as<int32_t>(),
                       s.nbr.as<int32_t>(), n, s.perm.as<int32_t>(), s.iperm.as<int32_t>(),
                       s.nLists > 1 ? s.seg.as<double>() : nullptr, s.nInt, s.rowsMapOrder ? 1 : 0);
  // 5. work list of internal slots
  s.work.ensure(sizeof(int32_t) * size_t(std::max<int64_t>(s.nInt, 1)));
  scanItems(WorkScan{s.perm.as<int32_t>(), s.work.as<int32_t>(), s.nInt}, n, s.scanTmp, st);
  SG_CHECK_HIP(hipGetLastError());
  SG_CHECK_HIP(hipEventRecord(s.ev[1], st));
}

}  // namespace

void* hostStaging(Sim& s, int which, size_t bytes) {
  void*& p = which ? s.pinnedIn : s.pinnedOut;
  size_t& cap = which ? s.pinnedInBytes : s.pinnedOutBytes;
  // uploads: the kernel of the previous use must have read the buffer (a build that
  // ended early leaves it unknown)
  if (which && s.pinnedInBusy) {
    SG_CHECK_HIP(hipStreamSynchronize(s.stream));
    s.pinnedInBusy = false;
  }
  if (bytes > cap) {
    SG_CHECK_HIP(hipStreamSynchronize(s.stream));   // no copy still uses the old buffer
    if (p) SG_CHECK_HIP(hipHostFree(p));
    p = nullptr;
    cap = 0;
    const size_t want = std::max<size_t>(4096, ((bytes + 4095) / 4096) * 4096);
    // uploads are read by a kernel: coherent, so none of it stays in a cache
    SG_CHECK_HIP(hipHostMalloc(&p, want, which ? hipHostMallocCoherent : hipHostMallocDefault));
    cap = want;
  }
  return p;
}

void zeroMany(const ZeroSet& z, hipStream_t st) {
  int64_t most = z.words;
  for (int q = 0; q < z.m; ++q) most = std::max(most, z.n[q]);
  if (most == 0) return;
  hipLaunchKernelGGL(k_zero_many, dim3(std::min(nblocks(most), 1024)), dim3(kBlock), 0, st, z);
  SG_CHECK_HIP(hipGetLastError());
}

void buildNeighbors(Sim& s, double ext) {
  s.cullStartsReady = false;
  SG_REQUIRE(s.nTot > 0, SPHGPU_ERR_STATE, "no nodes");
  SG_REQUIRE(ext > 0.0, SPHGPU_ERR_ARG, "kernel extent must be positive");
  s.kernelExtent = ext;
  s.neighborsValid = false;
  s.pairsValid = false;
  s.derivsValid = false;
  if (s.dim == 1) buildNeighborsD<1>(s, ext);
  else if (s.dim == 2) buildNeighborsD<2>(s, ext);
  else buildNeighborsD<3>(s, ext);
  s.timingPending |= 1u;
  s.neighborsValid = true;
}

}  // namespace sphgpu
