// Planar ghost boundaries on the device.
//
// The reference (src/Integrator/Integrator.cc:443-595) rebuilds its ghosts once
// per step: every boundary, in order, looks at all nodes that exist when it
// runs (internal nodes and the ghosts of the boundaries before it), selects
// its control nodes and appends one ghost per control
// (src/Boundary/PlanarBoundary.cc:112-182, 329-400):
//   hmax     = max over nodes i with min(|d_exit(x_i)|, |d_enter(x_i)|) < ext*h_i
//              of h_i = 1/lambda_min(H_i)
//   controls = nodes with 0 <= d_exit(x_i)/hmax <= ext, in index order
//   ghost    = mapPositionThroughPlanes(x_c, exit, enter); H, v by R = I - 2nn
//              (reflecting) or copied (periodic); scalars copied.
// After the connectivity is built, ghosts that no internal node sees and that
// control no other ghost are culled, the rest keep their order
// (src/Integrator/Integrator.cc:491-570, src/Boundary/Boundary.cc:182-233).
//
// Device form: one launch over the internal rows enters h into the hmax of every plane
// they are near (wavefront maximum, one 64-bit atomic max on the bit pattern of a
// non-negative double); then per plane one launch (two for large node sets) flags the
// controls, scans and appends their ghosts, which enter themselves for the planes
// after their own (scan.hh).  The row counts stay on the device and the launches cover
// a capacity; the neighbour build reads the counts back with its bounds.  Ghost fields
// are filled by one launch, each ghost from its internal node through the maps of the
// planes between.
// Culling: the row search marks every ghost slot it puts in a row; a scan of the keep
// flags over the ghosts gives the old -> new index map; the controls, the planes and the
// caller <-> slot maps are renumbered and the kept ghosts' rows filled again at their
// new place.  Slots themselves stay where they are (culled ghosts become dead slots that
// no row holds), so the rows, their entries and their order are untouched and no second
// build is needed.
//
// Floating-point order follows the reference exactly: plane distances
// n.(x - p), closest points x + ((p - x).n) n (3-D), the 2-D and 1-D special
// cases, and the closed-form eigenvalues of SymTensor::eigenValues
// (src/Geometry/GeomSymmetricTensorInline_default.hh:2053-2110).  The 3-D
// eigenvalues call atan2, cos and sin; their device and host results may
// differ in the last bit, which moves hmax by far less than one ulp except in
// rare rounding ties.
#include "internal.hh"
#include "dgeom.hh"
#include "records.hh"
#include "ell.hh"
#include "eigen.hh"
#include "pack.hh"
#include "scan.hh"
#include <cmath>
#include <algorithm>

namespace sphgpu {

namespace {

constexpr int kBlock = 256;
inline int nblocks(int64_t n, int bs = kBlock) { return int(std::max<int64_t>(1, (n + bs - 1) / bs)); }

struct DSub {
  double enterP[3], enterN[3], exitP[3], exitN[3];
  int reflect;
  int periodicSecond;
  double R[9];
};

DSub toDevice(const SubBoundary& b) {
  DSub d;
  for (int k = 0; k < 3; ++k) {
    d.enterP[k] = b.enterP[k]; d.enterN[k] = b.enterN[k]; d.exitP[k] = b.exitP[k]; d.exitN[k] = b.exitN[k];
  }
  d.reflect = b.reflect;
  d.periodicSecond = b.periodicSecond;
  for (int k = 0; k < 9; ++k) d.R[k] = b.R[k];
  return d;
}

template <int D> __device__ __forceinline__ V<D> loadV(const double* __restrict__ a, int64_t i) {
  V<D> v;
  for (int k = 0; k < D; ++k) v.c[k] = a[i * D + k];
  return v;
}
template <int D> __device__ __forceinline__ V<D> arr(const double* a) {
  V<D> v;
  for (int k = 0; k < D; ++k) v.c[k] = a[k];
  return v;
}
// GeomPlane::signedDistance: normal.dot(point - mPoint)
template <int D> __device__ __forceinline__ double signedDist(const double* P, const double* N, const V<D>& x) {
  return vdot(arr<D>(N), vsub(x, arr<D>(P)));
}
// GeomPlane::closestPointOnPlane (GeomPlane.cc:237-259, pointDistances.hh:53-57)
template <int D> __device__ __forceinline__ V<D> closestPoint(const double* P, const double* N, const V<D>& x) {
  if constexpr (D == 1) {
    return arr<1>(P);
  } else if constexpr (D == 2) {
    const V<2> a0p = vsub(x, arr<2>(P));
    V<2> dir;
    dir.c[0] = -N[1]; dir.c[1] = N[0];
    const double s = vdot(a0p, dir);
    V<2> o;
    for (int k = 0; k < 2; ++k) o.c[k] = P[k] + dir.c[k] * s;
    return o;
  } else {
    const double s = vdot(vsub(arr<3>(P), x), arr<3>(N));
    V<3> o;
    for (int k = 0; k < 3; ++k) o.c[k] = x.c[k] + N[k] * s;
    return o;
  }
}
// PlanarBoundary::updateGhostNodes: mapPositionThroughPlanes(x, exitPlane, enterPlane)
//   = closestPoint(enter, x) - signedDistance(exit, x) * enter.normal
template <int D> __device__ __forceinline__ V<D> ghostPosition(const DSub& b, const V<D>& x) {
  const V<D> p0 = closestPoint<D>(b.enterP, b.enterN, x);
  const double s = signedDist<D>(b.exitP, b.exitN, x);
  V<D> o;
  for (int k = 0; k < D; ++k) o.c[k] = p0.c[k] - b.enterN[k] * s;
  return o;
}

// R.v, rows left to right (GeomTensorInline_default.hh:1918-1922)
template <int D> __device__ __forceinline__ V<D> reflectV(const double* R, const V<D>& v) {
  V<D> o;
  for (int i = 0; i < D; ++i) {
    double s = R[i * D] * v.c[0];
    for (int k = 1; k < D; ++k) s = s + R[i * D + k] * v.c[k];
    o.c[i] = s;
  }
  return o;
}
// (R*(H*R)).Symmetric() (ReflectingBoundary.cc:155-175)
template <int D> __device__ __forceinline__ void reflectH(const double* R, const double* h, double* out) {
  double full[D * D], t1[D * D], t2[D * D];
  int c = 0;
  for (int i = 0; i < D; ++i)
    for (int j = i; j < D; ++j, ++c) { full[i * D + j] = h[c]; full[j * D + i] = h[c]; }
  for (int i = 0; i < D; ++i)
    for (int j = 0; j < D; ++j) {
      double s = full[i * D] * R[j];
      for (int k = 1; k < D; ++k) s = s + full[i * D + k] * R[k * D + j];
      t1[i * D + j] = s;
    }
  for (int i = 0; i < D; ++i)
    for (int j = 0; j < D; ++j) {
      double s = R[i * D] * t1[j];
      for (int k = 1; k < D; ++k) s = s + R[i * D + k] * t1[k * D + j];
      t2[i * D + j] = s;
    }
  c = 0;
  for (int i = 0; i < D; ++i)
    for (int j = i; j < D; ++j, ++c) out[c] = (i == j) ? t2[i * D + i] : 0.5 * (t2[i * D + j] + t2[j * D + i]);
}

// Ghost generation, device-held counts: gen[0] is set when a ghost fell beyond
// the capacity, gen[1 + b] holds the rows before plane b's ghosts (gen[1] =
// nInt), gen[1 + nSubs] all rows.
//
// A plane's hmax is the maximum of h = 1/lambda_min(H) over the rows near it:
// the internal nodes of a member or NodeList are entered for all planes by one
// launch, and each ghost enters itself for the planes after its own when it is
// made, so a plane needs no pass of its own for it.
struct HmaxBits {
  unsigned long long* bits;   // [plane][group], zero before the generation
  int groups;
};
// A non-negative double's bits order as the double: the maximum is an atomic
// max of the bits, skipped where the slot already holds as much (a plain read
// may be stale, then the atomic decides).
__device__ __forceinline__ void enterBits(unsigned long long* p, double h) {
  const unsigned long long v = (unsigned long long)__double_as_longlong(h);
  if (v > *static_cast<volatile unsigned long long*>(p)) atomicMax(p, v);
}
template <int D> __device__ __forceinline__ bool nearPlane(const DSub& b, const V<D>& x, double h, double ext) {
  const double d = dmin(dabs(signedDist<D>(b.exitP, b.exitN, x)), dabs(signedDist<D>(b.enterP, b.enterN, x)));
  return h > 0.0 && d < ext * h;
}

// h and hmax of the internal rows, the first counts, and the next generation's
// hmax table cleared.  A wavefront walks `rows64` consecutive groups of 64 rows
// once per plane (its rows stay in L1) and enters one maximum per plane, or,
// when its rows span members, one per lane: with an entry per row, 2.1 M rows
// took 534 us, all of it contention for the six words.
template <int D>
__global__ void k_gen_start(const double* __restrict__ pos, const double* __restrict__ H,
                            const double* __restrict__ seg, int64_t nInt, const DSub* __restrict__ subs, int nSubs,
                            double ext, HmaxBits hb, double* hmaxOf, int64_t* __restrict__ gen,
                            unsigned long long* __restrict__ clear, int rows64) {
  const int64_t tid = blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
  if (tid == 0) {
    gen[0] = 0;
    gen[1] = nInt;
  }
  for (int64_t q = tid; q < int64_t(nSubs) * hb.groups; q += int64_t(gridDim.x) * blockDim.x) clear[q] = 0ull;
  const int lane = threadIdx.x & 63;
  const int64_t base = (tid >> 6) * int64_t(64 * rows64) + lane;
  if (base - lane >= nInt) return;                 // uniform over the wavefront
  int group = 0;
  bool one = true;                                 // every row of the walk in one group
  for (int it = 0; it < rows64; ++it) {
    const int64_t i = base + int64_t(it) * 64;
    if (i < nInt) hmaxOf[i] = 1.0 / minEigen<D>(H + i * NSym<D>::value);
    if (seg) {
      const int g = i < nInt ? int(seg[i]) : -1, g0 = __shfl(g, 0);
      if (it == 0) group = g0;
      one = one && __all(g == group || g < 0) != 0;
    }
  }
  for (int b = 0; b < nSubs; ++b) {
    double v = 0.0;
    for (int it = 0; it < rows64; ++it) {
      const int64_t i = base + int64_t(it) * 64;
      if (i >= nInt) break;
      const double h = hmaxOf[i];
      if (!nearPlane<D>(subs[b], loadV<D>(pos, i), h, ext)) continue;
      if (one) v = dmax(v, h);
      else enterBits(hb.bits + int64_t(b) * hb.groups + int(seg[i]), h);
    }
    if (!one || __ballot(v > 0.0) == 0) continue;
    for (int sh = 32; sh > 0; sh >>= 1) v = dmax(v, __shfl_xor(v, sh));
    if (lane == 0) enterBits(hb.bits + int64_t(b) * hb.groups + group, v);
  }
}

// One plane's ghosts (scan.hh): the rows that are its controls, in index order,
// each appended after the rows that were there.  Flag, scan, compaction and the
// new row count in one launch (two for large node sets), where they were five.
template <int D> struct GhostPlane {
  static constexpr bool kCompact = true;
  double *pos, *H, *seg;
  int64_t cap, nInt;
  const DSub* subs;
  int plane, nSubs;
  double ext;
  HmaxBits hb;
  double* hmaxOf;
  int32_t *control, *subOf, *isControl;
  int64_t* gen;
  __device__ __forceinline__ int64_t live() const { return gen[1 + plane]; }
  __device__ int32_t value(int64_t i) const {
    if (i >= live()) return 0;
    const int group = seg ? int(seg[i]) : 0;
    const double hmax = __longlong_as_double((long long)hb.bits[int64_t(plane) * hb.groups + group]);
    if (!(hmax > 0.0)) return 0;
    const DSub& b = subs[plane];
    const double d = signedDist<D>(b.exitP, b.exitN, loadV<D>(pos, i)) / hmax;
    return d >= 0.0 && d <= ext ? 1 : 0;
  }
  __device__ void emit(int64_t i, int32_t prefix, int32_t) const {
    constexpr int NS = NSym<D>::value;
    const DSub& b = subs[plane];
    const int64_t g = live() + prefix;
    if (g >= cap) { gen[0] = 1; return; }          // the capacity was short: the caller generates again
    const V<D> xc = loadV<D>(pos, i), x = ghostPosition<D>(b, xc);
    for (int k = 0; k < D; ++k) pos[g * D + k] = x.c[k];
    // the control's h, unless the reflection changed H (an h I stays itself
    // under an axis plane): the eigenvalue is a function of these values alone
    const double hc = hmaxOf[i];
    double h = hc;
    if (b.reflect) {
      double hg[NS];
      bool same = true;
      reflectH<D>(b.R, H + i * NS, hg);
      for (int k = 0; k < NS; ++k) {
        same = same && hg[k] == H[i * NS + k];
        H[g * NS + k] = hg[k];
      }
      if (!same) h = 1.0 / minEigen<D>(hg);
    } else {
      for (int k = 0; k < NS; ++k) H[g * NS + k] = H[i * NS + k];
    }
    hmaxOf[g] = h;
    control[g - nInt] = int32_t(i);
    subOf[g - nInt] = plane;
    isControl[g - nInt] = 0;
    if (i >= nInt) isControl[i - nInt] = 1;
    if (seg) seg[g] = seg[i];
    const int group = seg ? int(seg[i]) : 0;
    // nothing to enter where the control, near the plane itself, has entered as much
    for (int q = plane + 1; q < nSubs; ++q)
      if (nearPlane<D>(subs[q], x, h, ext) && !(hc >= h && nearPlane<D>(subs[q], xc, hc, ext)))
        enterBits(hb.bits + int64_t(q) * hb.groups + group, h);
  }
  __device__ void total(int32_t t) const {
    const int64_t next = live() + t;
    if (next > cap) gen[0] = 1;
    gen[2 + plane] = next > cap ? cap : next;
  }
};

struct FieldPtrs {
  double *pos, *H, *vel, *mass, *rho, *eps, *P, *cs, *omega, *fCl, *fCq, *fsh, *seg;
};

// Where a ghost's values come from: its control may be a ghost of an earlier
// plane (edges and corners of a box), so a ghost is reached from an internal
// node by `depth` plane maps.  Every kernel below gives one lane to a ghost of
// any plane and applies those maps in order from the internal node, the same
// operations on the same values as filling plane after plane from the stored
// ghosts, so one launch serves all planes: a 2-D box step went from 12 + 4
// launches of 4.3 us (ghost fields, densities) to 4.
struct GhostMap {
  const int32_t* control;
  const int32_t* subOf;
  const DSub* subs;
  int64_t nInt;
};
// The internal node a ghost descends from, and the number of maps.
__device__ __forceinline__ int64_t ghostRoot(const GhostMap& m, int64_t g, int& depth) {
  depth = 0;
  while (g >= m.nInt) {
    g = m.control[g - m.nInt];
    ++depth;
  }
  return g;
}
// The plane of the map `step` controls below ghost g (step 0: g's own).
__device__ __forceinline__ const DSub& ghostPlane(const GhostMap& m, int64_t g, int step) {
  for (int q = 0; q < step; ++q) g = m.control[g - m.nInt];
  return m.subs[m.subOf[g - m.nInt]];
}

// All ghost rows [nInt, nTot) from their internal nodes.  REC >= 0: also their
// slots' records (pack sec bits, isotropic layout) from the values just stored.
template <int D, int REC>
__global__ void k_ghost_fields(FieldPtrs f, GhostMap m, int64_t nTot, const int64_t* __restrict__ nDev, int geometry,
                               const int32_t* __restrict__ iperm, PackOut pout) {
  constexpr int NS = NSym<D>::value;
  if (nDev) nTot = *nDev;                          // a generation's count, still on the device
  const int64_t g = m.nInt + blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
  if (g >= nTot) return;
  int depth;
  const int64_t r = ghostRoot(m, g, depth);
  V<D> x = vzero<D>(), v = loadV<D>(f.vel, r);
  double h[NS] = {};
  if (geometry) {
    x = loadV<D>(f.pos, r);
    for (int k = 0; k < NS; ++k) h[k] = f.H[r * NS + k];
  }
  for (int step = depth - 1; step >= 0; --step) {
    const DSub& b = ghostPlane(m, g, step);
    if (geometry) x = ghostPosition<D>(b, x);
    if (b.reflect) {
      v = reflectV<D>(b.R, v);
      if (geometry) {
        double hg[NS];
        reflectH<D>(b.R, h, hg);
        for (int k = 0; k < NS; ++k) h[k] = hg[k];
      }
    }
  }
  if (geometry) {
    for (int k = 0; k < D; ++k) f.pos[g * D + k] = x.c[k];
    for (int k = 0; k < NS; ++k) f.H[g * NS + k] = h[k];
  }
  for (int k = 0; k < D; ++k) f.vel[g * D + k] = v.c[k];
  PackRow<D> w;
  w.m = f.mass[r]; w.rho = f.rho[r]; w.P = f.P[r]; w.cs = f.cs[r]; w.omega = f.omega[r];
  f.eps[g] = f.eps[r];
  f.mass[g] = w.m;
  f.rho[g] = w.rho;
  f.P[g] = w.P;
  f.cs[g] = w.cs;
  f.omega[g] = w.omega;
  if (f.fCl) { f.fCl[g] = f.fCl[r]; f.fCq[g] = f.fCq[r]; f.fsh[g] = f.fsh[r]; }
  if (f.seg) f.seg[g] = f.seg[r];
  if constexpr (REC >= 0) {                        // always with the geometry
    w.x = x;
    w.v = v;
    for (int k = 0; k < NS; ++k) w.h.c[k] = h[k];
    packRow<D, true, REC>(iperm[g], g, w, pout);
  }
}

__global__ void k_ghost_scalar(double* __restrict__ a, GhostMap m, int64_t nTot) {
  const int64_t g = m.nInt + blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
  int depth;
  if (g < nTot) a[g] = a[ghostRoot(m, g, depth)];
}

// A Vector field on the ghost rows: R.a for every reflecting map, a copy for a
// periodic one (ReflectingBoundary.cc:106-125).
template <int D>
__global__ void k_ghost_vector(double* __restrict__ a, GhostMap m, int64_t nTot) {
  const int64_t g = m.nInt + blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
  if (g >= nTot) return;
  int depth;
  V<D> v = loadV<D>(a, ghostRoot(m, g, depth));
  for (int step = depth - 1; step >= 0; --step) {
    const DSub& b = ghostPlane(m, g, step);
    if (b.reflect) v = reflectV<D>(b.R, v);
  }
  for (int k = 0; k < D; ++k) a[g * D + k] = v.c[k];
}

// Ghost densities and records after sum density: the density of the internal
// node, and the same expressions as the internal update.
template <bool ISO>
__global__ void k_ghost_records(double* __restrict__ rec, const int32_t* __restrict__ iperm, double* __restrict__ rho,
                                GhostMap map, int64_t nTot) {
  using R = RL<ISO>;
  const int64_t g = map.nInt + blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
  if (g >= nTot) return;
  int depth;
  const double acc = rho[ghostRoot(map, g, depth)];
  rho[g] = acc;
  double* r = rec + int64_t(iperm[g]) * R::STRIDE;
  const double som = r[R::SOM], p = r[R::P], m = r[R::M];
  r[R::RHO] = acc;
  r[R::PRHO] = som * p / (acc * acc);
  r[R::MOR] = m / acc;
}

// ---- boundary enforcement ---------------------------------------------------
// position < plane (GeomPlane::compare == 1): n.(x - p) < 0 and not within
// fuzzyEqual of 0 (src/Geometry/GeomPlane.cc:306-341).
template <int D> __device__ __forceinline__ bool behind(const double* P, const double* N, const V<D>& x) {
  const double d = signedDist<D>(P, N, x);
  return !fuzzyEqual(d, 0.0) && !(d > 0.0);
}

// PlanarBoundary::setViolationNodes / updateViolationNodes over the internal
// nodes, with ReflectingBoundary::enforceBoundary of v and H
// ((R*H)*R).Symmetric(), src/Boundary/ReflectingBoundary.cc:240-282).
template <int D>
__device__ __forceinline__ bool enforcePlane(const DSub& b, V<D>& x, double* __restrict__ vel, double* __restrict__ H,
                                             int64_t i) {
  constexpr int NS = NSym<D>::value;
  if (!behind<D>(b.enterP, b.enterN, x)) return false;
  // mapPosition(x, enterPlane, exitPlane)
  const V<D> p0 = closestPoint<D>(b.exitP, b.exitN, x);
  const double sd = signedDist<D>(b.enterP, b.enterN, x);
  for (int k = 0; k < D; ++k) x.c[k] = p0.c[k] - b.exitN[k] * sd;
  if (b.reflect) {
    const V<D> v = reflectV<D>(b.R, loadV<D>(vel, i));
    for (int k = 0; k < D; ++k) vel[i * D + k] = v.c[k];
    double full[D * D], t1[D * D], t2[D * D];
    int c = 0;
    for (int a = 0; a < D; ++a)
      for (int q = a; q < D; ++q, ++c) { full[a * D + q] = H[i * NS + c]; full[q * D + a] = H[i * NS + c]; }
    for (int a = 0; a < D; ++a)
      for (int q = 0; q < D; ++q) {
        double sum = b.R[a * D] * full[q];
        for (int k = 1; k < D; ++k) sum = sum + b.R[a * D + k] * full[k * D + q];
        t1[a * D + q] = sum;
      }
    for (int a = 0; a < D; ++a)
      for (int q = 0; q < D; ++q) {
        double sum = t1[a * D] * b.R[q];
        for (int k = 1; k < D; ++k) sum = sum + t1[a * D + k] * b.R[k * D + q];
        t2[a * D + q] = sum;
      }
    c = 0;
    for (int a = 0; a < D; ++a)
      for (int q = a; q < D; ++q, ++c) H[i * NS + c] = (a == q) ? t2[a * D + a] : 0.5 * (t2[a * D + q] + t2[q * D + a]);
  }
  return true;
}

// PeriodicBoundary::updateViolationNodes: nodes still outside either plane
// are wrapped by the fmod rule (src/Boundary/PeriodicBoundary.cc:176-207).
// b: the first half of the pair (plane1 = enter, plane2 = exit).
template <int D> __device__ __forceinline__ bool wrapPair(const DSub& b, V<D>& x) {
  if (!(behind<D>(b.enterP, b.enterN, x) || behind<D>(b.exitP, b.exitN, x))) return false;
  const V<D> p2 = arr<D>(b.exitP);
  const double L = dabs(signedDist<D>(b.enterP, b.enterN, p2));
  const double s = vdot(vsub(arr<D>(b.enterP), x), arr<D>(b.enterN));
  const double f = dmax(-1.0, dmin(1.0, fmod(signedDist<D>(b.enterP, b.enterN, x) / L, 1.0)));
  for (int k = 0; k < D; ++k) x.c[k] = (x.c[k] + b.enterN[k] * s) + b.enterN[k] * (f * L);
  return true;
}

// Every plane in order on one node per lane (a node's enforcement reads no
// other node): one launch instead of one per plane and periodic pair.
template <int D>
__global__ void k_enforce(double* __restrict__ pos, double* __restrict__ vel, double* __restrict__ H, int64_t nInt,
                          const DSub* __restrict__ subs, int nSubs) {
  const int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
  if (i >= nInt) return;
  V<D> x = loadV<D>(pos, i);
  bool moved = false;
  for (int q = 0; q < nSubs; ++q) {
    moved |= enforcePlane<D>(subs[q], x, vel, H, i);
    // the second half of a periodic pair closes it: wrap what is still outside
    if (subs[q].periodicSecond) moved |= wrapPair<D>(subs[q - 1], x);
  }
  if (moved)
    for (int k = 0; k < D; ++k) pos[i * D + k] = x.c[k];
}

// ---- culling ---------------------------------------------------------------
// Which ghosts stay (scan.hh, over the ghosts): those some row holds (marked by
// the search in slot space) and those that control another ghost (marked when
// that one was made).  keep and scan are by ghost; the new first ghost of every
// plane, the new ghost count and the search's flags go to pinned memory.
struct KeepScan {
  static constexpr bool kCompact = false;
  const int32_t *slotKeep, *iperm, *isControl;
  int32_t *keep, *scan;
  int64_t nInt, ng;
  const int64_t* gen;       // gen[1 + b]: the rows before plane b's ghosts
  int nSubs;
  const int32_t* flags;
  SearchFlags* flagsOut;
  int32_t* starts;
  __device__ int32_t value(int64_t g) const { return slotKeep[iperm[nInt + g]] != 0 || isControl[g] != 0 ? 1 : 0; }
  __device__ void emit(int64_t g, int32_t prefix, int32_t v) const {
    keep[g] = v;
    scan[g] = prefix;
    for (int b = 0; b < nSubs; ++b)
      if (gen[1 + b] - nInt == g) starts[b] = prefix;
  }
  __device__ void total(int32_t t) const {
    for (int b = 0; b < nSubs; ++b)
      if (gen[1 + b] - nInt >= ng) starts[b] = t;
    starts[nSubs] = t;
    *flagsOut = foldFlags(flags);
  }
};

// Renumbering after the cull, one lane per caller row and slot: the kept
// ghosts' controls and planes, the caller -> slot map, and the slots' caller
// index (slots keep their place, culled ones die).  The records (when current)
// take the new caller index; nothing else in a record depends on the
// numbering, so they stay valid.  The ghosts' state rows are not moved but
// filled again at their new place: two launches in place of two per field and
// three more (22 in 2-D).
__global__ void k_cull(const int32_t* __restrict__ control, const int32_t* __restrict__ subOf,
                       int32_t* __restrict__ newControl, int32_t* __restrict__ newSubOf,
                       const int32_t* __restrict__ iperm, int32_t* __restrict__ newIperm, int32_t* __restrict__ perm,
                       const int32_t* __restrict__ keep, const int32_t* __restrict__ scan, int64_t nInt, int64_t nTot,
                       int64_t nSlots, double* __restrict__ rec, int stride, int origOff) {
  const int64_t t = blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
  if (t < nInt) {
    newIperm[t] = iperm[t];
  } else if (t < nTot && keep[t - nInt]) {
    const int64_t o = scan[t - nInt];
    const int32_t c = control[t - nInt];
    newIperm[nInt + o] = iperm[t];
    newControl[o] = c < nInt ? c : int32_t(nInt) + scan[c - nInt];
    newSubOf[o] = subOf[t - nInt];
  }
  if (t < nSlots) {
    const int32_t c = perm[t];
    if (c < nInt) return;
    const int32_t nc = keep[c - nInt] ? int32_t(nInt) + scan[c - nInt] : -1;
    perm[t] = nc;
    if (rec) rec[t * stride + origOff] = nc >= 0 ? double(nc) : 2147483648.0;
  }
}

std::vector<DBuf*> stateBufs(Sim& s) {
  return {&s.pos, &s.vel, &s.H, &s.mass, &s.rho, &s.eps, &s.P, &s.cs, &s.omega, &s.fCl, &s.fCq, &s.fshear, &s.seg};
}
// fields 9-11 exist with Q multipliers, field 12 in an ensemble
bool stateUsed(const Sim& s, int which) {
  if (which >= 9 && which < 12) return s.hasMultipliers;
  if (which == 12) return s.ensemble || s.nLists > 1;
  return true;
}
int stateComps(const Sim& s, int which) {
  const int D = s.dim, NS = nsymOf(D);
  return which == 0 || which == 1 ? D : (which == 2 ? NS : 1);
}

// Make room for `rows` rows in every caller-order field, keeping nTot rows.
void ensureRows(Sim& s, int64_t rows) {
  auto bufs = stateBufs(s);
  for (int w = 0; w < int(bufs.size()); ++w) {
    if (!stateUsed(s, w)) continue;
    const size_t per = sizeof(double) * size_t(stateComps(s, w));
    if (bufs[size_t(w)]->bytes >= per * size_t(rows)) continue;
    bufs[size_t(w)]->grow(per * size_t(rows + rows / 4), per * size_t(s.nTot), s.stream);
  }
}

FieldPtrs fieldPtrs(Sim& s) {
  FieldPtrs f;
  f.pos = s.pos.as<double>(); f.H = s.H.as<double>(); f.vel = s.vel.as<double>(); f.mass = s.mass.as<double>();
  f.rho = s.rho.as<double>(); f.eps = s.eps.as<double>(); f.P = s.P.as<double>(); f.cs = s.cs.as<double>();
  f.omega = s.omega.as<double>();
  f.fCl = s.hasMultipliers ? s.fCl.as<double>() : nullptr;
  f.fCq = s.hasMultipliers ? s.fCq.as<double>() : nullptr;
  f.fsh = s.hasMultipliers ? s.fshear.as<double>() : nullptr;
  f.seg = s.ensemble || s.nLists > 1 ? s.seg.as<double>() : nullptr;
  return f;
}

GhostMap ghostMap(const Sim& s) {
  return GhostMap{s.ghostControl.as<int32_t>(), s.ghostSub.as<int32_t>(), s.subDev.as<DSub>(), s.nInt};
}

// Rows [nInt, nTot), or those of a generation whose count is on the device.
template <int D> void applyFieldsD(Sim& s, bool geometry, int rec) {
  const int64_t rows = s.genPending ? s.genCap : s.nTot, ng = rows - s.nInt;
  const int64_t* nDev = s.genPending ? s.genDev.as<int64_t>() + s.subs.size() + 1 : nullptr;
  if (ng <= 0) {
    if (rec >= 0) (void)packOutputs(s, rec);
    return;
  }
  const FieldPtrs f = fieldPtrs(s);
  const GhostMap m = ghostMap(s);
  SG_REQUIRE(rec < 0 || geometry, SPHGPU_ERR_STATE, "ghost records take the refreshed geometry");
  const PackOut pout = rec >= 0 ? packOutputs(s, rec) : PackOut{};
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(nblocks(ng)), dim3(kBlock), 0, s.stream, f, m, rows, nDev, geometry ? 1 : 0,
                       s.iperm.as<int32_t>(), pout);
  };
  switch (rec) {
    case -1: go(k_ghost_fields<D, -1>); break;
    case 0: go(k_ghost_fields<D, 0>); break;
    case 1: go(k_ghost_fields<D, 1>); break;
    case 2: go(k_ghost_fields<D, 2>); break;
    case 4: go(k_ghost_fields<D, 4>); break;
    case 8: go(k_ghost_fields<D, 8>); break;
    default: SG_REQUIRE(false, SPHGPU_ERR_STATE, "unsupported record kinds for the ghost rows");
  }
  SG_CHECK_HIP(hipGetLastError());
}
void applyFields(Sim& s, bool geometry, int rec) {
  if (s.dim == 1) applyFieldsD<1>(s, geometry, rec);
  else if (s.dim == 2) applyFieldsD<2>(s, geometry, rec);
  else applyFieldsD<3>(s, geometry, rec);
}

// Every plane's ghosts, with the running row count kept on the device: the
// launches cover a capacity of `est` ghosts, and the neighbour build reads the
// counts back with its bounds (finishGeneration), one wait for both.  Generation
// reads only internal rows, so a short capacity costs a second one.
template <int D> void generateD(Sim& s, double ext, int64_t est) {
  hipStream_t st = s.stream;
  const int64_t nInt = s.nInt, cap = nInt + est;
  SG_REQUIRE(cap < (int64_t(1) << 31) - 1, SPHGPU_ERR_CAPACITY, "too many ghost nodes");
  const int nSubs = int(s.subs.size()), groups = std::max(1, groupCount(s));
  ensureRows(s, cap);
  s.hmaxOf.ensure(sizeof(double) * size_t(cap));
  for (DBuf* b : {&s.ghostControl, &s.ghostSub, &s.ghostIsControl}) b->ensure(sizeof(int32_t) * size_t(est));
  s.genDev.ensure(sizeof(int64_t) * size_t(nSubs + 2));
  unsigned long long* next = nullptr;
  const HmaxBits hb{s.hmaxBits.take(size_t(nSubs) * size_t(groups), st, next), groups};
  double* seg = groupCount(s) > 0 ? s.seg.as<double>() : nullptr;
  // one group of 64 rows a wavefront until every SIMD has one
  const int rows64 = int(std::min<int64_t>(16, std::max<int64_t>(1, nInt / (64 * 1024))));
  hipLaunchKernelGGL(k_gen_start<D>, dim3(nblocks((nInt + rows64 - 1) / rows64)), dim3(kBlock), 0, st,
                     s.pos.as<double>(), s.H.as<double>(), seg, nInt, s.subDev.as<DSub>(), nSubs, ext, hb,
                     s.hmaxOf.as<double>(), s.genDev.as<int64_t>(), next, rows64);
  SG_CHECK_HIP(hipGetLastError());
  for (int b = 0; b < nSubs; ++b) {
    // rows before plane b: all of the capacity but for the first plane
    const GhostPlane<D> op{s.pos.as<double>(), s.H.as<double>(), seg, cap, nInt, s.subDev.as<DSub>(), b, nSubs, ext, hb,
                           s.hmaxOf.as<double>(), s.ghostControl.as<int32_t>(), s.ghostSub.as<int32_t>(),
                           s.ghostIsControl.as<int32_t>(), s.genDev.as<int64_t>()};
    scanItems(op, b == 0 ? nInt : cap, s.scanTmp, st);
  }
  s.genCap = cap;
  s.genPending = true;
  applyFieldsD<D>(s, false, -1);
}

// Ghosts expected of a first generation: four layers of nodes at every plane.
int64_t ghostGuess(const Sim& s) {
  if (s.ghostsGenerated > 0) return s.ghostsGenerated + s.ghostsGenerated / 4 + 1024;
  const double groups = double(std::max(1, groupCount(s))), per = double(s.nInt) / groups;
  const double face = std::pow(std::max(per, 1.0), double(s.dim - 1) / s.dim);
  return int64_t(6.0 * face * groups * double(s.subs.size())) + 4096;
}

}  // namespace

void finishGeneration(Sim& s, const int64_t* gen) {
  const size_t nSubs = s.subs.size();
  if (gen[0]) throw GhostCapacity{};
  s.nTot = gen[1 + nSubs];
  s.subStart.resize(nSubs + 1);
  for (size_t b = 0; b <= nSubs; ++b) s.subStart[b] = gen[1 + b] - s.nInt;
  s.ghostsGenerated = s.nTot - s.nInt;
}

// Integrator::cullGhostNodes, first half: which ghosts stay and their new
// places; the new first ghost of every plane and the ghost count (nsub + 1
// values) and the search flags copied to pinned memory, read after the
// caller's next wait.  The neighbour build issues it before its row readback so
// that one wait serves both.
void cullLaunch(Sim& s, SearchFlags* flagsOut, int32_t* starts) {
  const int64_t ng = s.nTot - s.nInt;
  s.keep.ensure(sizeof(int32_t) * size_t(ng));
  s.keepScan.ensure(sizeof(int32_t) * size_t(ng));
  scanItems(KeepScan{s.slotKeep.as<int32_t>(), s.iperm.as<int32_t>(), s.ghostIsControl.as<int32_t>(),
                     s.keep.as<int32_t>(), s.keepScan.as<int32_t>(), s.nInt, ng, s.genDev.as<int64_t>(),
                     int(s.subs.size()), s.flags.as<int32_t>(), flagsOut, starts},
            ng, s.scanTmp, s.stream);
}

namespace {

void cull(Sim& s) {
  hipStream_t st = s.stream;
  const int64_t n = s.nTot, nInt = s.nInt;
  if (n == nInt) return;
  SG_REQUIRE(s.cullStartsReady && s.cullStarts.size() == s.subStart.size(), SPHGPU_ERR_STATE, "stale cull starts");
  s.cullStartsReady = false;
  const std::vector<int32_t>& starts = s.cullStarts;   // launched and read with the neighbour build's rows
  int32_t* keep = s.keep.as<int32_t>();
  const int64_t nNew = nInt + starts.back();
  if (nNew == n) return;
  const int32_t* scan = s.keepScan.as<int32_t>();

  s.ghostControlSpare.ensure(s.ghostControl.bytes);
  s.ghostSubSpare.ensure(s.ghostSub.bytes);
  s.ipermSpare.ensure(s.iperm.bytes);
  const bool recs = s.recValid;
  // The density records keep the pre-cull caller index of their ghosts: the
  // density sum compares a neighbour's index only with an internal node's
  // (to place the self term), and culling keeps every internal index and
  // every ghost's index above them, so no comparison changes.
  hipLaunchKernelGGL(k_cull, dim3(nblocks(std::max(n, s.nSlots))), dim3(kBlock), 0, st, s.ghostControl.as<int32_t>(),
                     s.ghostSub.as<int32_t>(), s.ghostControlSpare.as<int32_t>(), s.ghostSubSpare.as<int32_t>(),
                     s.iperm.as<int32_t>(), s.ipermSpare.as<int32_t>(), s.perm.as<int32_t>(), keep, scan, nInt, n,
                     s.nSlots, recs ? s.rec.as<double>() : nullptr, s.isotropic ? RL<true>::STRIDE : RL<false>::STRIDE,
                     s.isotropic ? RL<true>::ORIG : RL<false>::ORIG);
  SG_CHECK_HIP(hipGetLastError());
  s.ghostControl.swap(s.ghostControlSpare);
  s.ghostSub.swap(s.ghostSubSpare);
  s.iperm.swap(s.ipermSpare);
  for (size_t b = 0; b < s.subStart.size(); ++b) s.subStart[b] = starts[b];
  s.nTot = nNew;
  // the kept ghost rows at their new places, filled again from the internal
  // nodes (the same maps of the same values)
  applyFields(s, true, -1);
  s.recValid = recs;
  // with several NodeLists the density sum also looks up a neighbour's
  // NodeList by that index: the density records are packed again
  if (s.nLists > 1) s.recSValid = false;
  s.derivsValid = false;
}

}  // namespace

void setBoundaries(Sim& s, int n, const sphgpu_boundary* b) {
  SG_REQUIRE(n >= 0 && (n == 0 || b), SPHGPU_ERR_ARG, "bad boundary list");
  const int D = s.dim;
  std::vector<SubBoundary> subs;
  auto unit = [&](const double* nin, double* nout) {
    // GeomPlane: normal.unitVector() (1-D divides, else multiplies by 1/|n|)
    double m2 = nin[0] * nin[0];
    for (int k = 1; k < D; ++k) m2 = m2 + nin[k] * nin[k];
    const double m = D == 1 ? std::fabs(nin[0]) : std::sqrt(m2);
    SG_REQUIRE(m > 1.0e-50, SPHGPU_ERR_ARG, "boundary plane normal is zero");
    for (int k = 0; k < 3; ++k) nout[k] = 0.0;
    if (D == 1) nout[0] = nin[0] / m;
    else { const double inv = 1.0 / m; for (int k = 0; k < D; ++k) nout[k] = nin[k] * inv; }
  };
  for (int q = 0; q < n; ++q) {
    SG_REQUIRE(b[q].kind == SPHGPU_BOUNDARY_REFLECTING || b[q].kind == SPHGPU_BOUNDARY_PERIODIC, SPHGPU_ERR_ARG,
               "unknown boundary kind");
    double n1[3], n2[3], p1[3] = {0, 0, 0}, p2[3] = {0, 0, 0};
    unit(b[q].plane1.normal, n1);
    for (int k = 0; k < D; ++k) p1[k] = b[q].plane1.point[k];
    SubBoundary a{};
    if (b[q].kind == SPHGPU_BOUNDARY_REFLECTING) {
      for (int k = 0; k < 3; ++k) { a.enterP[k] = a.exitP[k] = p1[k]; a.enterN[k] = a.exitN[k] = n1[k]; }
      a.reflect = 1;
      a.periodicSecond = 0;
      // Tensor::one - 2.0*normal.selfdyad()
      for (int i = 0; i < D; ++i)
        for (int j = 0; j < D; ++j) a.R[i * D + j] = (i == j ? 1.0 : 0.0) - 2.0 * (n1[std::min(i, j)] * n1[std::max(i, j)]);
      subs.push_back(a);
    } else {
      unit(b[q].plane2.normal, n2);
      for (int k = 0; k < D; ++k) p2[k] = b[q].plane2.point[k];
      SubBoundary c{}, d{};
      for (int k = 0; k < 3; ++k) {
        c.enterP[k] = p1[k]; c.enterN[k] = n1[k]; c.exitP[k] = p2[k]; c.exitN[k] = n2[k];
        d.enterP[k] = p2[k]; d.enterN[k] = n2[k]; d.exitP[k] = p1[k]; d.exitN[k] = n1[k];
      }
      c.reflect = d.reflect = 0;
      c.periodicSecond = 0;
      d.periodicSecond = 1;
      subs.push_back(c);
      subs.push_back(d);
    }
  }
  std::vector<DSub> dev;
  for (const SubBoundary& b2 : subs) dev.push_back(toDevice(b2));
  if (s.subDev.p) SG_CHECK_HIP(hipStreamSynchronize(s.stream));   // earlier launches may still read the old planes
  s.subDev.ensure(sizeof(DSub) * std::max<size_t>(dev.size(), 1));
  if (!dev.empty())
    SG_CHECK_HIP(hipMemcpyAsync(s.subDev.p, dev.data(), sizeof(DSub) * dev.size(), hipMemcpyHostToDevice, s.stream));
  SG_CHECK_HIP(hipStreamSynchronize(s.stream));   // `dev` dies on return
  s.subs = subs;
  s.subStart.clear();
}

void setGhostNodes(Sim& s, double ext, bool doCull) {
  SG_REQUIRE(ext > 0.0, SPHGPU_ERR_ARG, "kernel extent must be positive");
  SG_REQUIRE(s.nTot == s.nInt || s.deviceGhosts, SPHGPU_ERR_STATE,
             "sphgpu_set_ghost_nodes needs n_total = n_internal (ghosts are made on the device)");
  hipStream_t st = s.stream;
  SG_CHECK_HIP(hipEventRecord(s.ev[8], st));
  s.neighborsValid = false;
  s.recValid = false;
  s.derivsValid = false;
  struct Pending {                       // neither outlives this call, however it ends
    Sim& s;
    ~Pending() { s.markGhostUse = s.genPending = false; }
  };
  for (int64_t est = ghostGuess(s);; est *= 4) {
    Pending pending{s};
    s.nTot = s.nInt;                     // drop the previous ghosts
    s.subStart.assign(s.subs.size() + 1, 0);
    if (!s.subs.empty()) {
      if (s.dim == 1) generateD<1>(s, ext, est);
      else if (s.dim == 2) generateD<2>(s, ext, est);
      else generateD<3>(s, ext, est);
    }
    s.deviceGhosts = true;
    SG_CHECK_HIP(hipEventRecord(s.ev[9], st));
    s.markGhostUse = doCull;
    try {
      buildNeighbors(s, ext);
      break;
    } catch (const GhostCapacity&) {     // again with room for four times as many
    }
  }
  SG_CHECK_HIP(hipEventRecord(s.ev[10], st));
  if (doCull) cull(s);
  SG_CHECK_HIP(hipEventRecord(s.ev[11], st));
  s.timingPending |= 8u;
}

void applyGhostBoundaries(Sim& s) {
  if (!s.deviceGhosts || s.nTot == s.nInt) return;
  applyFields(s, true, -1);
  s.recValid = false;
  s.derivsValid = false;
}

void applyGhostBoundariesAndRecords(Sim& s, int rec) {
  SG_REQUIRE(s.deviceGhosts || s.nTot == s.nInt, SPHGPU_ERR_STATE, "the ghost rows were not made by the boundaries");
  applyFields(s, true, rec);
  s.recValid = true;
  s.derivsValid = false;
}

void enforceBoundaries(Sim& s) {
  if (s.subs.empty() || s.nInt == 0) return;
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(nblocks(s.nInt)), dim3(kBlock), 0, s.stream, s.pos.as<double>(), s.vel.as<double>(),
                       s.H.as<double>(), s.nInt, s.subDev.as<DSub>(), int(s.subs.size()));
  };
  if (s.dim == 1) go(k_enforce<1>);
  else if (s.dim == 2) go(k_enforce<2>);
  else go(k_enforce<3>);
  SG_CHECK_HIP(hipGetLastError());
  s.recValid = false;
  s.derivsValid = false;
}

void applyGhostScalar(Sim& s, DBuf& field) {
  if (!s.deviceGhosts || s.nTot == s.nInt) return;
  hipLaunchKernelGGL(k_ghost_scalar, dim3(nblocks(s.nTot - s.nInt)), dim3(kBlock), 0, s.stream, field.as<double>(),
                     ghostMap(s), s.nTot);
  SG_CHECK_HIP(hipGetLastError());
}

void ensureStateRows(Sim& s, int64_t rows) { ensureRows(s, rows); }
bool stateFieldUsed(const Sim& s, int which) { return stateUsed(s, which); }

namespace {
__global__ void k_fill_value(double* __restrict__ a, int64_t first, int64_t rows, double v) {
  const int64_t r = blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
  if (r < rows) a[first + r] = v;
}
}  // namespace

// Several NodeLists in one node set: NodeList L owns `counts[L]` consecutive
// internal rows, in NodeList order; their ghosts are made by the device
// boundaries, each NodeList with its own (PlanarBoundary::setGhostNodes per
// NodeList).  gamma (may be null) gives each NodeList its gamma-law EOS.
void setNodeLists(Sim& s, int n, const int64_t* counts, const double* gamma, int sumAll) {
  SG_REQUIRE(!s.ensemble, SPHGPU_ERR_STATE, "an ensemble holds independent simulations, not NodeLists");
  SG_REQUIRE(n >= 1 && counts, SPHGPU_ERR_ARG, "need at least one NodeList");
  SG_REQUIRE(s.nTot == s.nInt, SPHGPU_ERR_STATE,
             "set the NodeLists on internal rows only (n_total = n_internal); the device makes their ghosts");
  std::vector<int64_t> start(size_t(n) + 1, 0);
  for (int L = 0; L < n; ++L) {
    SG_REQUIRE(counts[L] >= 0, SPHGPU_ERR_ARG, "negative NodeList size");
    start[size_t(L) + 1] = start[size_t(L)] + counts[L];
  }
  SG_REQUIRE(start.back() == s.nInt, SPHGPU_ERR_ARG, "the NodeList sizes must add up to n_internal");
  if (gamma)
    for (int L = 0; L < n; ++L) SG_REQUIRE(gamma[L] > 1.0, SPHGPU_ERR_ARG, "a NodeList gamma must exceed 1");
  s.nLists = n > 1 ? n : 0;
  s.listStart = start;
  s.sumAllLists = sumAll != 0;
  s.listGammaHost.assign(gamma ? gamma : nullptr, gamma ? gamma + n : nullptr);
  if (gamma) {
    s.listGamma.ensure(sizeof(double) * size_t(n));
    SG_CHECK_HIP(hipMemcpyAsync(s.listGamma.p, gamma, sizeof(double) * size_t(n), hipMemcpyHostToDevice, s.stream));
  }
  if (s.nLists > 1) {
    ensureRows(s, std::max<int64_t>(s.nTot, 1));
    for (int L = 0; L < n; ++L)
      if (counts[L] > 0)
        hipLaunchKernelGGL(k_fill_value, dim3(nblocks(counts[L])), dim3(kBlock), 0, s.stream, s.seg.as<double>(),
                           start[size_t(L)], counts[L], double(L));
    SG_CHECK_HIP(hipGetLastError());
  }
  SG_CHECK_HIP(hipStreamSynchronize(s.stream));   // `gamma` may be released on return
  s.neighborsValid = false;
  s.recValid = false;
  s.derivsValid = false;
}
DBuf& stateField(Sim& s, int which) { return *stateBufs(s)[size_t(which)]; }
int stateFieldComps(const Sim& s, int which) { return stateComps(s, which); }

void applyGhostVector(Sim& s, DBuf& field) {
  if (!s.deviceGhosts || s.nTot == s.nInt) return;
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(nblocks(s.nTot - s.nInt)), dim3(kBlock), 0, s.stream, field.as<double>(), ghostMap(s),
                       s.nTot);
  };
  if (s.dim == 1) go(k_ghost_vector<1>);
  else if (s.dim == 2) go(k_ghost_vector<2>);
  else go(k_ghost_vector<3>);
  SG_CHECK_HIP(hipGetLastError());
}

void applyGhostDensity(Sim& s) {
  if (!s.deviceGhosts || s.nTot == s.nInt) return;
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(nblocks(s.nTot - s.nInt)), dim3(kBlock), 0, s.stream, s.rec.as<double>(),
                       s.iperm.as<int32_t>(), s.rho.as<double>(), ghostMap(s), s.nTot);
  };
  if (s.isotropic) go(k_ghost_records<true>);
  else go(k_ghost_records<false>);
  SG_CHECK_HIP(hipGetLastError());
}

}  // namespace sphgpu
