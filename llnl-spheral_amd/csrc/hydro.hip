// Device sum density and evaluateDerivatives.
//
// Both passes run in gather form: one lane per internal node (nodes in the
// neighbour build's sorted order), walking its full row.  The reference
// (src/SPH/SPHHydroBase.cc:575-928, src/SPH/computeSPHSumMassDensity.cc:60-103)
// evaluates each unordered pair once in the frame of its owner (the lower index,
// ConnectivityMapInline.hh:182-184) and adds to both ends, visiting owners in
// ascending order; so every node receives its pair terms in ascending neighbour
// order.  With rows in that order (SPHGPU_ROW_ORDER_REFERENCE), walking a row in
// the node's own frame reproduces the reference's FP64 sums exactly:
//   * quantities odd in r_ij (eta, unit vectors, grad W, v_ij, Q accelerations,
//     the acceleration increment) only flip sign with the frame, exactly;
//   * products of two odd quantities (mu, v.gradW, dyads, r r) are unchanged;
//   * the two terms that depend on who owns the pair are kept: the Q
//     accelerations enter the acceleration sum owner first, and the tensile
//     factor uses the owner's W.
// Sum density adds the self term where the reference does: after the
// contributions of lower-index neighbours, before those of higher ones.
// With H = h I (every off-diagonal exactly zero) the SymTensor products reduce
// to h*r componentwise with the same bits, which the isotropic kernels use.
//
// Memory: neighbour indices arrive four at a time (one int4 of the blocked ELL),
// the next neighbour's record is loaded while the current pair is evaluated,
// and the kernel table sits in LDS.
#include <type_traits>
#include "internal.hh"
#include "dgeom.hh"
#include "records.hh"
#include "pack.hh"
#include "ell.hh"
#include "eigen.hh"
#include "lanes.hh"
#include <cstring>
#include <cmath>

namespace sphgpu {

namespace {

constexpr int kBlock = 256;
inline int nblocks(int64_t n, int bs = kBlock) { return int(std::max<int64_t>(1, (n + bs - 1) / bs)); }

// ---------------------------------------------------------------------------
// Record pack: every slot, or the `count` slots listed in `slots`.
// ---------------------------------------------------------------------------
template <int D, bool ISO, int SEC = 0>
__global__ void k_pack(PackIn in, PackOut o, const int32_t* __restrict__ slots, int64_t count) {
  const int64_t t = blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
  if (t >= count) return;
  packSlot<D, ISO, SEC>(slots ? int64_t(slots[t]) : t, in, o);
}

// Table: per point [Ak Bk Ck Ag Bg Cg].
struct TabArgs {
  const double* g;     // global copy
  const float* g32;    // FP32 copy, 8 floats per point
  int n;
  double step, extent;
  const double* nperh;
  const double* wsum;
};

__device__ __forceinline__ void lookupWG(const double* __restrict__ tab, const TabArgs& t, double eta, double Hdet,
                                         double& W, double& gW) {
  if (eta < t.extent) {
    const double q = eta / t.step;
    int lb = int(q);
    lb = lb < t.n - 1 ? lb : t.n - 1;
    const int i0 = lb < t.n - 3 ? lb : t.n - 3;
    const double x = q - i0;
    const double* c = tab + 6 * (i0 + 1);
    W = Hdet * (c[0] + c[1] * x + c[2] * x * x);
    gW = Hdet * (c[3] + c[4] * x + c[5] * x * x);
  } else {
    W = 0.0; gW = 0.0;
  }
}
__device__ __forceinline__ double lookupW(const double* __restrict__ tab, const TabArgs& t, double eta, double Hdet) {
  if (!(eta < t.extent)) return 0.0;
  const double q = eta / t.step;
  int lb = int(q);
  lb = lb < t.n - 1 ? lb : t.n - 1;
  const int i0 = lb < t.n - 3 ? lb : t.n - 3;
  const double x = q - i0;
  const double* c = tab + 6 * (i0 + 1);
  return Hdet * (c[0] + c[1] * x + c[2] * x * x);
}

// Largest table that is staged in LDS (the 1000-point default takes 48 KB).
constexpr int kLdsTablePoints = 1365;
// Staging the table costs a full table read and a barrier per workgroup; it
// pays when each node makes many lookups (2-D rows hold ~28 entries, 3-D rows
// ~120), not for 1-D rows of ~6, which read the table through L1.
constexpr double kLdsMinRow = 16.0;
bool ldsTable(const Sim& s) {
  if (s.table.n > kLdsTablePoints) return false;
  const double perNode = s.nInt > 0 ? double(s.nEntries) / double(s.nInt) : 0.0;
  return perNode >= kLdsMinRow;
}

template <bool LDS> __device__ __forceinline__ const double* stageTable(double* lds, const TabArgs& t) {
  if constexpr (LDS) {
    for (int q = threadIdx.x; q < 6 * t.n; q += blockDim.x) lds[q] = t.g[q];
    __syncthreads();
    return lds;
  } else {
    return t.g;
  }
}

// TableKernel::equivalentNodesPerSmoothingScale (TableKernel.cc:399-429).
__device__ double equivalentNperh(const TabArgs& t, double Wsum) {
  const int n = t.n;
  const double* ws = t.wsum;
  const double* np = t.nperh;
  const bool ascnd = ws[n - 1] >= ws[0];
  int jl = -1, ju = n;
  while (ju - jl > 1) {
    const int jm = (ju + jl) / 2;
    if ((Wsum >= ws[jm]) == ascnd) jl = jm; else ju = jm;
  }
  const int lb = jl, ub = jl + 1;
  if (lb == -1) return np[0];
  if (ub == n) return np[n - 1];
  return dmin(np[ub], dmax(np[lb], np[lb] + (Wsum - ws[lb]) / (ws[ub] - ws[lb]) * (np[ub] - np[lb])));
}

// SPHSmoothingScale::idealSmoothingScale (src/NodeList/SPHSmoothingScale.cc:120-197):
// 1/h1 of the ideal H = h1^-1 I from the root-nu zeroth moment and H.xx.
__device__ __forceinline__ double idealHinv(const TabArgs& t, double zeroth, double Hxx, double nPerh, double hmin,
                                            double hmax) {
  double nperhNow;
  if (fuzzyEqual(zeroth, 0.0)) nperhNow = 0.5 * nPerh;
  else nperhNow = equivalentNperh(t, zeroth);
  const double s = dmin(4.0, dmax(0.25, nPerh / (nperhNow + 1.0e-30)));
  const double aa = (s < 1.0) ? 0.4 * (1.0 + s * s) : 0.4 * (1.0 + 1.0 / (s * s * s));
  const double hi0 = 1.0 / Hxx;
  const double hi1 = dmin(hmax, dmax(hmin, hi0 * (1.0 - aa + aa * s)));
  return 1.0 / hi1;
}

// H.v: with isotropic H the product is h*v componentwise (same bits as the
// SymTensor product with zero off-diagonals).
template <int D, bool ISO> __device__ __forceinline__ V<D> hdot(const S<D>& H, const V<D>& v) {
  if constexpr (ISO) {
    V<D> o;
    for (int c = 0; c < D; ++c) o.c[c] = H.c[0] * v.c[c];
    return o;
  } else {
    return sdot(H, v);
  }
}

// Neighbour indices of one row arrive four at a time (one int4 of the blocked
// ELL); the next int4 is fetched one chunk ahead.
__device__ __forceinline__ int32_t pick4(const int4 v, int q) {
  return q == 0 ? v.x : (q == 1 ? v.y : (q == 2 ? v.z : v.w));
}
// Advance to entry w (w >= 1, called for w = 1, 2, ... in order).
__device__ __forceinline__ int32_t nextIndex(const int4* __restrict__ nb4, int64_t n, int64_t k, int len, int w,
                                             int4& cur, int4& nxt) {
  if ((w & 3) == 0) {
    cur = nxt;
    if (w + 4 < len) nxt = nb4[ellChunk((w >> 2) + 1, n, k)];
  }
  return pick4(cur, w & 3);
}

// What one side of a pair reads from a neighbour's record.
template <int D, bool ISO> struct Nbr {
  V<D> x, v;
  S<D> H;
  double hdet, m, orig, rho, cs, prho, mor, p, som, fcl, fcq, fsh;
};
template <int D, bool ISO, bool WANT_P>
__device__ __forceinline__ Nbr<D, ISO> loadNbr(const double* __restrict__ rec, int32_t j) {
  using R = RL<ISO>;
  const double* r = rec + int64_t(j) * R::STRIDE;
  Nbr<D, ISO> o;
  for (int c = 0; c < D; ++c) { o.x.c[c] = r[R::X + c]; o.v.c[c] = r[R::V + c]; }
  if constexpr (ISO) {
    o.H.c[0] = r[RL<true>::HINV];
    for (int c = 1; c < NSym<D>::value; ++c) o.H.c[c] = 0.0;
    for (int c = 1; c < D; ++c) o.H.c[sdiag<D>(c)] = o.H.c[0];
    o.fcl = o.fcq = o.fsh = 1.0;
  } else {
    for (int c = 0; c < NSym<D>::value; ++c) o.H.c[c] = r[RL<false>::H + c];
    o.fcl = r[RL<false>::FCL]; o.fcq = r[RL<false>::FCQ]; o.fsh = r[RL<false>::FSH];
  }
  o.hdet = r[R::HDET]; o.m = r[R::M]; o.orig = r[R::ORIG]; o.rho = r[R::RHO]; o.cs = r[R::CS];
  o.prho = r[R::PRHO]; o.mor = r[R::MOR];
  if constexpr (WANT_P) { o.p = r[R::P]; o.som = r[R::SOM]; } else { o.p = 0.0; o.som = 0.0; }
  return o;
}

// ---------------------------------------------------------------------------
// computeSPHSumMassDensity
// ---------------------------------------------------------------------------
template <int D, bool ISO> struct DNbr {
  V<D> x;
  S<D> H;
  double hdet, m, orig;
};
template <int D, bool ISO>
__device__ __forceinline__ DNbr<D, ISO> loadDNbr(const double* __restrict__ rec, int32_t j) {
  using R = RL<ISO>;
  const double* r = rec + int64_t(j) * R::STRIDE;
  DNbr<D, ISO> o;
  for (int c = 0; c < D; ++c) o.x.c[c] = r[R::X + c];
  if constexpr (ISO) {
    o.H.c[0] = r[RL<true>::HINV];
    for (int c = 1; c < NSym<D>::value; ++c) o.H.c[c] = 0.0;
    for (int c = 1; c < D; ++c) o.H.c[sdiag<D>(c)] = o.H.c[0];
  } else {
    for (int c = 0; c < NSym<D>::value; ++c) o.H.c[c] = r[RL<false>::H + c];
  }
  o.hdet = r[R::HDET]; o.m = r[R::M]; o.orig = r[R::ORIG];
  return o;
}
// A density record (DensRec).  det H of an exactly isotropic H is (1/h)^D as
// sdet evaluates it (the off-diagonal products are exact zeros): bitwise the
// packed value.
template <int D>
__device__ __forceinline__ DNbr<D, true> loadDensRec(const double* __restrict__ recS, int32_t j) {
  const double2* p = reinterpret_cast<const double2*>(recS) + int64_t(j) * 3;
  const double2 a = p[0], b = p[1], c = p[2];
  DNbr<D, true> o;
  o.x.c[0] = a.x;
  if constexpr (D > 1) o.x.c[1] = a.y;
  if constexpr (D > 2) o.x.c[2] = b.x;
  const double hinv = b.y;
  o.H.c[0] = hinv;
  for (int c2 = 1; c2 < NSym<D>::value; ++c2) o.H.c[c2] = 0.0;
  for (int c2 = 1; c2 < D; ++c2) o.H.c[sdiag<D>(c2)] = hinv;
  o.hdet = D == 1 ? hinv : (D == 2 ? hinv * hinv : (hinv * hinv) * hinv);
  o.m = c.x; o.orig = c.y;
  return o;
}

// Neighbours come from nrec: the density records (DensRec) for isotropic H, else
// the full records.
// L > 1: L lanes to a node, the table through L1.
template <int D, bool ISO, bool LDS, int L = 1>
__global__ void __launch_bounds__(kBlock) k_sum_density(double* __restrict__ rec, const int32_t* __restrict__ rowCount,
                                                        const int32_t* __restrict__ nbr, int64_t n, int64_t nInt,
                                                        const int32_t* __restrict__ work, TabArgs t,
                                                        double* __restrict__ rhoOut, const double* __restrict__ nrec,
                                                        const double* __restrict__ listOf, int sumAll) {
  using R = RL<ISO>;
  extern __shared__ double lds[];
  const double* tab = stageTable<LDS>(lds, t);
  const int64_t tw = (xcdBlock((nInt * L + kBlock - 1) / kBlock) * kBlock + threadIdx.x) / L;
  if (tw >= nInt) return;
  const int64_t k = work[tw];
  double* ri_ = rec + k * R::STRIDE;
  const double oi = ri_[R::ORIG];
  const DNbr<D, ISO> me = loadDNbr<D, ISO>(rec, int32_t(k));
  const double mi = me.m;
  const double self = mi * lookupW(tab, t, 0.0, me.hdet);
  double acc = 0.0;
  bool selfDone = false;
  const int len = rowCount[k];
  auto load = [&](int32_t j) {
    if constexpr (ISO) return loadDensRec<D>(nrec, j);
    else return loadDNbr<D, false>(nrec, j);
  };
  auto term = [&](const DNbr<D, ISO>& nb) {
    // several NodeLists: a pair across them counts with sumAll only, the node
    // taking its own mass (computeSPHSumMassDensity.cc:77-100)
    const bool same = !listOf || listOf[int64_t(nb.orig)] == listOf[int64_t(oi)];
    if (!same && !sumAll) return -0.0;
    const V<D> rij = vsub(me.x, nb.x);
    const double etaj = vmag(hdot<D, ISO>(nb.H, rij));
    return (same ? nb.m : mi) * lookupW(tab, t, etaj, nb.hdet);
  };
  if constexpr (L > 1) {
    alignas(16) __shared__ double buf[kBlock];
    double* wbuf = buf + (threadIdx.x & ~63);
    const int sub = threadIdx.x % L;
    for (int w0 = 0; w0 < len; w0 += L) {
      const bool live = w0 + sub < len;
      const DNbr<D, ISO> nb = load(live ? nbr[ellIndex(w0 + sub, n, k)] : int32_t(k));
      const int first = firstLane<L>(live && nb.orig > oi);
      const double tm = term(nb);
      acc = addInOrder<L>(acc, live ? tm : -0.0, wbuf, selfDone ? 64 : first, self);
      selfDone = selfDone || first < L;
    }
    if (!selfDone) acc += self;
    if (sub != 0) return;
  } else {
    const int4* nb4 = reinterpret_cast<const int4*>(nbr);
    int4 cur = len > 0 ? nb4[ellChunk(0, n, k)] : make_int4(0, 0, 0, 0);
    int4 nxt = len > 4 ? nb4[ellChunk(1, n, k)] : make_int4(0, 0, 0, 0);
    DNbr<D, ISO> nx;
    if (len > 0) nx = load(cur.x);
    for (int w = 0; w < len; ++w) {
      const DNbr<D, ISO> nb = nx;
      if (w + 1 < len) nx = load(nextIndex(nb4, n, k, len, w + 1, cur, nxt));
      if (!selfDone && nb.orig > oi) { acc += self; selfDone = true; }
      acc += term(nb);
    }
    if (!selfDone) acc += self;
  }
  rhoOut[int64_t(oi)] = acc;
  // keep the record consistent with the new density (the pass reads only
  // positions, H and masses of the neighbours)
  const double som = ri_[R::SOM], p = ri_[R::P];
  ri_[R::RHO] = acc;
  ri_[R::PRHO] = som * p / (acc * acc);
  ri_[R::MOR] = mi / acc;
}

// ---------------------------------------------------------------------------
// computeSPHOmegaGradhCorrection (src/SPH/computeSPHOmegaGradhCorrection.cc:26-133)
// Gather form of the owner loop: node i receives W(|H_i r_ij|) det H_i and
// |H_i r_ij| W' from every neighbour in row order, its self term W(0) det H_i
// after the lower-index neighbours, and omega_i = -sum(eta W')/(nu sum W); a
// node without neighbours gets 1.  With index-ordered rows this is the
// reference's sum order; with several NodeLists the reference-order rows come
// in the order the owner loop delivers node i's terms (the internal owners of
// lower index first, then i's own pairs), and the owner of a pair is still its
// end of lower caller index, so the self term goes to the same place.
// ---------------------------------------------------------------------------
template <int D, bool ISO, bool LDS, int L = 1>
__global__ void __launch_bounds__(kBlock) k_omega(const double* __restrict__ rec, const int32_t* __restrict__ rowCount,
                                                  const int32_t* __restrict__ nbr, int64_t n, int64_t nInt,
                                                  const int32_t* __restrict__ work, TabArgs t,
                                                  double* __restrict__ omegaOut) {
  extern __shared__ double lds[];
  const double* tab = stageTable<LDS>(lds, t);
  const int64_t tw = (xcdBlock((nInt * L + kBlock - 1) / kBlock) * kBlock + threadIdx.x) / L;
  if (tw >= nInt) return;
  const int64_t k = work[tw];
  const DNbr<D, ISO> me = loadDNbr<D, ISO>(rec, int32_t(k));
  const int len = rowCount[k];
  const double self = lookupW(tab, t, 0.0, me.hdet);
  double om = 0.0, gs = 0.0;
  bool selfDone = false;
  auto terms = [&](const DNbr<D, ISO>& nb, double& Wv, double& eg) {
    const V<D> rij = vsub(me.x, nb.x);
    const double eta = vmag(hdot<D, ISO>(me.H, rij));
    double gW;
    lookupWG(tab, t, eta, me.hdet, Wv, gW);
    eg = eta * gW;
  };
  if constexpr (L > 1) {
    alignas(16) __shared__ double buf[kBlock];
    double* wbuf = buf + (threadIdx.x & ~63);
    const int sub = threadIdx.x % L;
    for (int w0 = 0; w0 < len; w0 += L) {
      const bool live = w0 + sub < len;
      const DNbr<D, ISO> nb = loadDNbr<D, ISO>(rec, live ? nbr[ellIndex(w0 + sub, n, k)] : int32_t(k));
      const int first = firstLane<L>(live && nb.orig > me.orig);
      double Wv, eg;
      terms(nb, Wv, eg);
      om = addInOrder<L>(om, live ? Wv : -0.0, wbuf, selfDone ? 64 : first, self);
      gs = addInOrder<L>(gs, live ? eg : -0.0, wbuf);
      selfDone = selfDone || first < L;
    }
    if (sub != 0) return;
  } else if (len > 0) {
    const int4* nb4 = reinterpret_cast<const int4*>(nbr);
    int4 cur = nb4[ellChunk(0, n, k)];
    int4 nxt = len > 4 ? nb4[ellChunk(1, n, k)] : make_int4(0, 0, 0, 0);
    DNbr<D, ISO> nx = loadDNbr<D, ISO>(rec, cur.x);
    for (int w = 0; w < len; ++w) {
      const DNbr<D, ISO> nb = nx;
      if (w + 1 < len) nx = loadDNbr<D, ISO>(rec, nextIndex(nb4, n, k, len, w + 1, cur, nxt));
      if (!selfDone && nb.orig > me.orig) { om += self; selfDone = true; }
      double Wv, eg;
      terms(nb, Wv, eg);
      om += Wv;
      gs += eg;
    }
  }
  if (len == 0) {
    omegaOut[int64_t(me.orig)] = 1.0;
    return;
  }
  if (!selfDone) om += self;
  omegaOut[int64_t(me.orig)] = -gs / (double(D) * om);
}

// ---------------------------------------------------------------------------
// evaluateDerivatives, FP64
// ---------------------------------------------------------------------------
struct PassArgs {
  double Cl, Cq, eps2, epsTensile, nPerh, hmin, hmax;
  double W0, WnPerh;
  int XSPH, correctVelocityGradient, evolveTotalEnergy, linearInExpansion, quadraticInExpansion;
  double qInv;   // 1/u and u of the 3-D mixed record's positions
  float qUnit;
  const double* listOf;   // NodeList of every caller row (several NodeLists), or null
  const int32_t* slotList;   // NodeList of every slot (several NodeLists, collapsed kernel), or null
};

__device__ __forceinline__ double muQ(double mu, double Cl, double Cq, double cs, const PassArgs& p) {
  const double m0 = dmin(0.0, mu);
  const double lin = p.linearInExpansion ? mu : m0;
  const double quad = p.quadraticInExpansion ? -(mu < 0.0 ? -1.0 : 1.0) * mu * mu : m0 * m0;
  return -Cl * cs * lin + Cq * quad;
}

struct OutArgs {
  double* base;      // field-major blocks, each n rows
  int64_t n;         // rows per block (sorted slots)
  int off[SPHGPU_NUM_DERIV_FIELDS];
  int updateOnly;    // store only the fields an integrator update reads
  double* pairDv;    // compatible energy: the pair term of every row entry in the node's own
                     // frame, component c at pairDv[c*plane + ellIndex(w, n, k)]; null otherwise
  int64_t plane;
  double* relV;      // dt vote: the largest |v_ij|^2 of the row per slot (FP64 in 1-D: |v_ij|; mixed:
                     // FP32, 3-D with one lane to a node only), -1 for an empty row; null otherwise
};

// The pair limit of GenericHydro::dt (src/Physics/GenericHydro.cc:218-283) is
// the smallest nodeScale/|v_ij|, and rounding is monotonic, so the largest
// |v_ij| of a row gives it to the bit.  The pass at the step start has every
// v_ij at hand; a vote that gathered the velocities again took 1.45 ms at 128^3,
// these terms under 0.1 ms.  A NaN is passed over, as the vote's minimum does.
template <int D> __device__ __forceinline__ double relSpeed(const double* d) {
  if constexpr (D == 1) return dabs(d[0]);
  double s = d[0] * d[0];
  for (int c = 1; c < D; ++c) s = s + d[c] * d[c];
  return s;
}

__device__ __forceinline__ double* outRow(const OutArgs& o, int field, int64_t k, int comps) {
  return o.base + int64_t(o.off[field]) * o.n + k * comps;
}

// Per-node accumulators of the pair loop (FP64 in both precisions).
template <int D> struct Acc {
  double rhoSum, norm, DepsDt, maxVP, effVP, viscW, xsphW, wNS;
  V<D> DvDt, xsphDV;
  T<D> DvDx, M;
  S<D> m2nd;
  __device__ __forceinline__ void zero() {
    rhoSum = norm = DepsDt = maxVP = effVP = viscW = xsphW = wNS = 0.0;
    DvDt = vzero<D>(); xsphDV = vzero<D>(); DvDx = tzero<D>(); M = tzero<D>(); m2nd = szero<D>();
  }
};

// Own-node values the epilogue reads.
template <int D> struct Self {
  V<D> v;
  S<D> H;
  double Hdet, m, rho, mor;
};

// Per-node epilogue (SPHHydroBase.cc:834-902) and the output stores.
template <int D>
__device__ __forceinline__ void epilogue(int64_t k, int len, const Self<D>& me, Acc<D>& a, const TabArgs& t,
                                         const PassArgs& p, const OutArgs& o) {
  constexpr int NS = NSym<D>::value;
  const double tiny = 1.0e-30;
  const V<D> vi = me.v;
  const S<D> Hi = me.H;
  const double Hdeti = me.Hdet, mi = me.m, rhoi = me.rho, mori = me.mor;
  double rhoSum = a.rhoSum, norm = a.norm, DepsDt = a.DepsDt, xsphW = a.xsphW;
  V<D> DvDt = a.DvDt, xsphDV = a.xsphDV;
  T<D> DvDx = a.DvDx, M = a.M;
  S<D> m2nd = a.m2nd;
  rhoSum += mi * p.W0 * Hdeti;
  norm += mori * p.W0 * Hdeti;
  T<D> Mout = M;
  if (p.correctVelocityGradient && fabs(tdet(M)) > 1.0e-10 && double(len) > pownu2<D>()) {
    Mout = tinv(M);
    DvDx = tdot(DvDx, Mout);
  } else {
    tdivEq(DvDx, rhoi);
  }
  const double trace = ttrace(DvDx);
  const double DrhoDt = -rhoi * trace;
  if (p.evolveTotalEnergy) DepsDt = mi * (vdot(vi, DvDt) + DepsDt);
  const double wNSo = rootnu<D>(dmax(0.0, a.wNS / Hdeti));
  m2nd = sdivs(m2nd, Hdeti * Hdeti);
  V<D> DxDt = vi;
  if (p.XSPH) {
    xsphW += Hdeti * mi / rhoi * p.W0;
    const V<D> corr = vdivs(xsphDV, dmax(tiny, xsphW));
    for (int c = 0; c < D; ++c) DxDt.c[c] = vi.c[c] + corr.c[c];
  }
  // SPHSmoothingScale::smoothingScaleDerivative: -H/nu * tr(DvDx)
  S<D> negH;
  for (int c = 0; c < NS; ++c) negH.c[c] = -Hi.c[c];
  S<D> DHDt = sdivs(negH, double(D));
  for (int c = 0; c < NS; ++c) DHDt.c[c] = DHDt.c[c] * trace;
  // SPHSmoothingScale::idealSmoothingScale
  const double hinv = idealHinv(t, wNSo, Hi.c[0], p.nPerh, p.hmin, p.hmax);

  // outputs
  // the fields an integrator update reads
  *outRow(o, SPHGPU_D_DRHODT, k, 1) = DrhoDt;
  *outRow(o, SPHGPU_D_DEPSDT, k, 1) = DepsDt;
  {
    double* dx = outRow(o, SPHGPU_D_DXDT, k, D);
    double* dv = outRow(o, SPHGPU_D_DVDT, k, D);
    for (int c = 0; c < D; ++c) { dx[c] = DxDt.c[c]; dv[c] = DvDt.c[c]; }
    double* hid = outRow(o, SPHGPU_D_HIDEAL, k, NS);
    for (int a2 = 0, s2 = 0; a2 < D; ++a2)
      for (int b2 = a2; b2 < D; ++b2, ++s2) hid[s2] = (a2 == b2 ? 1.0 : 0.0) * hinv;
  }
  if (o.updateOnly) return;
  *outRow(o, SPHGPU_D_RHO_SUM, k, 1) = rhoSum;
  *outRow(o, SPHGPU_D_NORMALIZATION, k, 1) = norm;
  *outRow(o, SPHGPU_D_MAX_VISCOUS_PRESSURE, k, 1) = a.maxVP;
  *outRow(o, SPHGPU_D_EFF_VISCOUS_PRESSURE, k, 1) = a.effVP;
  *outRow(o, SPHGPU_D_VISCOUS_WORK, k, 1) = a.viscW;
  *outRow(o, SPHGPU_D_XSPH_WEIGHT_SUM, k, 1) = xsphW;
  *outRow(o, SPHGPU_D_WEIGHTED_NEIGHBOR_SUM, k, 1) = wNSo;
  {
    double* xv = outRow(o, SPHGPU_D_XSPH_DELTA_V, k, D);
    for (int c = 0; c < D; ++c) xv[c] = xsphDV.c[c];
  }
  {
    double* g = outRow(o, SPHGPU_D_DVDX, k, D * D);
    double* gl = outRow(o, SPHGPU_D_LOCAL_DVDX, k, D * D);
    double* m = outRow(o, SPHGPU_D_M, k, D * D);
    double* ml = outRow(o, SPHGPU_D_LOCAL_M, k, D * D);
    for (int c = 0; c < D * D; ++c) { g[c] = DvDx.c[c]; gl[c] = DvDx.c[c]; m[c] = Mout.c[c]; ml[c] = Mout.c[c]; }
  }
  {
    double* dh = outRow(o, SPHGPU_D_DHDT, k, NS);
    double* m2 = outRow(o, SPHGPU_D_MASS_SECOND_MOMENT, k, NS);
    for (int c = 0; c < NS; ++c) { dh[c] = DHDt.c[c]; m2[c] = m2nd.c[c]; }
  }
}

// The pairs a wavefront evaluated, one entry per wavefront of the work list:
// nothing to clear before the pass, no atomics, and no read-back unless the
// caller asks for the count.  The entry's index is formed again here from
// scalars: a lane's work index kept through the pair loop cost two VGPRs, which
// took the mixed 3-D kernel from 167 to 169 and from three waves per SIMD to two.
template <int BS>
__device__ __forceinline__ void storePairCount(unsigned pairs, int64_t nInt, uint32_t* __restrict__ counts) {
  for (int sh = 32; sh > 0; sh >>= 1) pairs += __shfl_xor(pairs, sh);
  const int64_t wave = xcdBlock((nInt + BS - 1) / BS) * (BS / 64) + (__builtin_amdgcn_readfirstlane(threadIdx.x) >> 6);
  if (__lane_id() == 0 && wave * 64 < nInt) counts[wave] = pairs;
}

// The sums of the pair loop by number, in the order pairTerms adds to them.
template <int D> struct Sum {
  static constexpr int NS = NSym<D>::value;
  static constexpr int WNS = 0, M2 = 1, RHO = M2 + NS, NORM = RHO + 1, EFFVP = NORM + 1, VISCW = EFFVP + 1,
                       DV = VISCW + 1, DEPS = DV + D, DVDX = DEPS + 1, M = DVDX + D * D, XW = M + D * D, XDV = XW + 1,
                       COUNT = XDV + D;
};
template <int D> __device__ __forceinline__ Acc<D> accOf(const double* a) {
  using S_ = Sum<D>;
  Acc<D> o;
  o.wNS = a[S_::WNS]; o.rhoSum = a[S_::RHO]; o.norm = a[S_::NORM]; o.effVP = a[S_::EFFVP]; o.viscW = a[S_::VISCW];
  o.DepsDt = a[S_::DEPS]; o.xsphW = a[S_::XW];
  for (int c = 0; c < D; ++c) { o.DvDt.c[c] = a[S_::DV + c]; o.xsphDV.c[c] = a[S_::XDV + c]; }
  for (int c = 0; c < D * D; ++c) { o.DvDx.c[c] = a[S_::DVDX + c]; o.M.c[c] = a[S_::M + c]; }
  for (int c = 0; c < NSym<D>::value; ++c) o.m2nd.c[c] = a[S_::M2 + c];
  return o;
}

// One pair in node i's frame, with the reference's operations: every term goes
// to add(sum, term), sums in ascending number.  Returns 1 for a pair i owns.
// RELV: the row maximum of the vote, where the pass leaves one.  ALL: add() is an
// exchange that every lane enters, with -0, which changes no sum, where a pair has no
// term; else such a term is branched over (100^3 nodes, one lane to a node: 2.21 ms
// with the selects, 2.13 without).
template <int D, bool ISO, bool TENSILE, bool RELV, bool ALL, class Add>
__device__ __forceinline__ unsigned pairTerms(const Nbr<D, ISO>& me, const Nbr<D, ISO>& nb, int w, int64_t n, int64_t k,
                                              const double* __restrict__ tab, const TabArgs& t, const PassArgs& p,
                                              const OutArgs& o, double& maxVP, double& relV, Add&& add) {
  using S_ = Sum<D>;
  const double Hdeti = me.hdet, rhoi = me.rho, ci = me.cs, mori = me.mor;
  const bool ownerI = nb.orig > me.orig;
  const V<D> rij = vsub(me.x, nb.x);
  const V<D> vij = vsub(me.v, nb.v);
  if constexpr (RELV) {
    if (o.relV) relV = dmax(relV, relSpeed<D>(vij.c));
  }
  const S<D>& Hi = me.H;
  const S<D>& Hj = nb.H;
  const double Hdetj = nb.hdet, mj = nb.m, rhoj = nb.rho, cj = nb.cs, morj = nb.mor;

  const V<D> etai = hdot<D, ISO>(Hi, rij), etaj = hdot<D, ISO>(Hj, rij);
  const double eta2i = vmag2(etai), eta2j = vmag2(etaj);
  const double etaMagi = (D == 1) ? fabs(etai.c[0]) : __builtin_sqrt(eta2i);
  const double etaMagj = (D == 1) ? fabs(etaj.c[0]) : __builtin_sqrt(eta2j);
  const V<D> Hetai = hdot<D, ISO>(Hi, vunit(etai, etaMagi));
  const V<D> Hetaj = hdot<D, ISO>(Hj, vunit(etaj, etaMagj));
  double Wi, gWi, Wj, gWj;
  lookupWG(tab, t, etaMagi, Hdeti, Wi, gWi);
  lookupWG(tab, t, etaMagj, Hdetj, Wj, gWj);
  const V<D> gradWi = vscale(Hetai, gWi);
  const V<D> gradWj = vscale(Hetaj, gWj);

  // moments for the ideal H (SPHHydroBase.cc:737-743)
  const double rij2 = vmag2(rij);
  const double sinv = safeInvVar(rij2 * rij2 * rij2);
  const double g2 = vmag2(gradWi);
  add(S_::WNS, fabs(gWi));
  {
    int s = 0;
    for (int a = 0; a < D; ++a)
      for (int b = a; b < D; ++b, ++s) add(S_::M2 + s, (rij.c[a] * rij.c[b]) * sinv * g2);
  }
  // same-NodeList pairs only (SPHHydroBase.cc:746-751)
  const bool same = !p.listOf || p.listOf[int64_t(nb.orig)] == p.listOf[int64_t(me.orig)];
  if (ALL || same) {
    add(S_::RHO, same ? mj * Wi : -0.0);
    add(S_::NORM, same ? mori * Wi : -0.0);
  }

  // Monaghan-Gingold Q (MonaghanGingoldViscosity.cc:83-132)
  double Cl = p.Cl, Cq = p.Cq;
  if constexpr (!ISO) {
    const double fsh = dmax(me.fsh, nb.fsh);
    Cl *= 0.5 * (me.fcl + nb.fcl) * fsh;
    Cq *= 0.5 * (me.fcq + nb.fcq) * fsh;
  }
  const double mui = vdot(vij, etai) / (eta2i + p.eps2);
  const double muj = vdot(vij, etaj) / (eta2j + p.eps2);
  const double QPi = muQ(mui, Cl, Cq, ci, p) / rhoi;
  const double QPj = muQ(muj, Cl, Cq, cj, p) / rhoj;
  V<D> Qacci, Qaccj;
  for (int c = 0; c < D; ++c) { Qacci.c[c] = 0.5 * (QPi * gradWi.c[c]); Qaccj.c[c] = 0.5 * (QPj * gradWj.c[c]); }
  const double workQi = vdot(vij, Qacci);
  const double Qi = rhoi * rhoi * fabs(QPi);
  maxVP = dmax(maxVP, Qi);
  add(S_::EFFVP, morj * Qi * Wi);
  add(S_::VISCW, mj * workQi);

  double Prhoi = me.prho, Prhoj = nb.prho;
  if constexpr (TENSILE) {
    const double Wo = ownerI ? Wi : Wj, Hdeto = ownerI ? Hdeti : Hdetj;
    const double x = Wo / (Hdeto * p.WnPerh);
    const double fij = p.epsTensile * (x * x * x * x);
    const double Pi = me.p, Pj = nb.p;
    Prhoi = me.som * (Pi + fij * (Pi < 0.0 ? -Pi : 0.0)) / (rhoi * rhoi);
    Prhoj = nb.som * (Pj + fij * (Pj < 0.0 ? -Pj : 0.0)) / (rhoj * rhoj);
  }
  for (int c = 0; c < D; ++c) {
    const double qf = ownerI ? Qacci.c[c] : Qaccj.c[c];
    const double qs = ownerI ? Qaccj.c[c] : Qacci.c[c];
    const double dv = gradWi.c[c] * Prhoi + gradWj.c[c] * Prhoj + qf + qs;
    add(S_::DV + c, dv * (-mj));
    if (o.pairDv) o.pairDv[int64_t(c) * o.plane + ellIndex(w, n, k)] = dv;
  }
  add(S_::DEPS, mj * (Prhoi * vdot(vij, gradWi) + workQi));
  // a difference is the sum with the term's negative, to the bit
  for (int a = 0; a < D; ++a)
    for (int b = 0; b < D; ++b) add(S_::DVDX + a * D + b, -((vij.c[a] * gradWi.c[b]) * mj));
  for (int a = 0; a < D; ++a)
    for (int b = 0; b < D; ++b) add(S_::M + a * D + b, -((rij.c[a] * gradWi.c[b]) * mj));
  if (ALL || p.XSPH) {
    const double w2 = 0.5 * (mori * Wi + morj * Wj);
    add(S_::XW, p.XSPH ? w2 : -0.0);
    for (int c = 0; c < D; ++c) add(S_::XDV + c, p.XSPH ? -(vij.c[c] * w2) : -0.0);
  }
  return ownerI ? 1u : 0u;
}

template <int D, bool ISO>
__device__ __forceinline__ Self<D> selfOf(const Nbr<D, ISO>& me) {
  Self<D> s;
  s.v = me.v; s.H = me.H; s.Hdet = me.hdet; s.m = me.m; s.rho = me.rho; s.mor = me.mor;
  return s;
}

template <int D, bool ISO, bool TENSILE, bool LDS, bool RELV>
__global__ void __launch_bounds__(kBlock) k_derivs_fp64(const double* __restrict__ rec, const int32_t* __restrict__ rowCount,
                                                        const int32_t* __restrict__ nbr, int64_t n, int64_t nInt,
                                                        const int32_t* __restrict__ work, TabArgs t, PassArgs p,
                                                        OutArgs o, uint32_t* __restrict__ pairCounts) {
  extern __shared__ double lds[];
  const double* tab = stageTable<LDS>(lds, t);
  const int64_t tw = xcdBlock((nInt + kBlock - 1) / kBlock) * kBlock + threadIdx.x;
  unsigned pairs = 0;
  if (tw < nInt) {
    const int64_t k = work[tw];
    const Nbr<D, ISO> me = loadNbr<D, ISO, true>(rec, int32_t(k));
    double sum[Sum<D>::COUNT];
#pragma unroll
    for (int q = 0; q < Sum<D>::COUNT; ++q) sum[q] = 0.0;
    double maxVP = 0.0, relV = 0.0;
    const int len = rowCount[k];
    const int4* nb4 = reinterpret_cast<const int4*>(nbr);
    int4 cur = len > 0 ? nb4[ellChunk(0, n, k)] : make_int4(0, 0, 0, 0);
    int4 nxt = len > 4 ? nb4[ellChunk(1, n, k)] : make_int4(0, 0, 0, 0);
    Nbr<D, ISO> nx;
    if (len > 0) nx = loadNbr<D, ISO, TENSILE>(rec, cur.x);
    for (int w = 0; w < len; ++w) {
      const Nbr<D, ISO> nb = nx;
      if (w + 1 < len) nx = loadNbr<D, ISO, TENSILE>(rec, nextIndex(nb4, n, k, len, w + 1, cur, nxt));
      pairs += pairTerms<D, ISO, TENSILE, RELV, false>(me, nb, w, n, k, tab, t, p, o, maxVP, relV,
                                                       [&](int q, double v) { sum[q] += v; });
    }
    if constexpr (RELV) o.relV[k] = len > 0 ? relV : -1.0;
    Acc<D> a = accOf<D>(sum);
    a.maxVP = maxVP;
    epilogue<D>(k, len, selfOf(me), a, t, p, o);
  }
  storePairCount<kBlock>(pairs, nInt, pairCounts);
}

// The same pass with L lanes to a node: the terms of L sums at a time go through
// LDS, and each lane adds up one of them, entry by entry (one read and one add
// per sum and L entries, where sums kept by every lane would take L adds each).
// A lane holds COUNT / L sums instead of COUNT.  LDS rows are padded to 65
// doubles: lane q reads row q, so rows a multiple of 64 apart would all hit the
// same banks.
template <int D, bool ISO, bool TENSILE, int L>
__global__ void __launch_bounds__(kBlock) k_derivs_rows(const double* __restrict__ rec,
                                                        const int32_t* __restrict__ rowCount,
                                                        const int32_t* __restrict__ nbr, int64_t n, int64_t nInt,
                                                        const int32_t* __restrict__ work, TabArgs t, PassArgs p,
                                                        OutArgs o, uint32_t* __restrict__ pairCounts) {
  constexpr int COUNT = Sum<D>::COUNT, BATCH = (COUNT + L - 1) / L, NODES = kBlock / L, PAD = 65;
  __shared__ double terms[kBlock / 64][L][PAD];
  __shared__ double sums[NODES][BATCH * L + 2];
  const int64_t block = xcdBlock((nInt * L + kBlock - 1) / kBlock);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, sub = threadIdx.x % L;
  const int64_t tw = block * NODES + threadIdx.x / L;
  unsigned pairs = 0;
  double maxVP = 0.0, relV = 0.0, acc[BATCH];
#pragma unroll
  for (int q = 0; q < BATCH; ++q) acc[q] = 0.0;
  const int64_t k = tw < nInt ? work[tw] : 0;
  const int len = tw < nInt ? rowCount[k] : 0;
  const Nbr<D, ISO> me = loadNbr<D, ISO, true>(rec, int32_t(k));
  for (int w0 = 0; w0 < len; w0 += L) {
    const int w = w0 + sub;
    const bool live = w < len;
    // a lane past its row evaluates the node's pair with itself, unused
    const int32_t j = live ? nbr[ellIndex(w, n, k)] : int32_t(k);
    const Nbr<D, ISO> nb = loadNbr<D, ISO, TENSILE>(rec, j);
    OutArgs oo = o;
    if (!live) oo.pairDv = nullptr;
    double vp = maxVP, rv = relV;
    const unsigned own = pairTerms<D, ISO, TENSILE, true, true>(
        me, nb, w, n, k, t.g, t, p, oo, vp, rv, [&](int q, double v) {
          terms[wave][q % L][lane] = live ? v : -0.0;
          if (q % L == L - 1 || q == COUNT - 1) {
            waveLdsOrder();
            double a = acc[q / L];
#pragma unroll
            for (int e = 0; e < L; ++e) a += terms[wave][sub][lane - sub + e];
            acc[q / L] = a;
            waveLdsOrder();
          }
        });
    if (live) {
      maxVP = vp;
      relV = rv;
      pairs += own;
    }
  }
  for (int s = L / 2; s > 0; s >>= 1) {
    maxVP = dmax(maxVP, __shfl_xor(maxVP, s));
    relV = dmax(relV, __shfl_xor(relV, s));
  }
  double* mine = sums[threadIdx.x / L];
#pragma unroll
  for (int q = 0; q < BATCH; ++q) mine[q * L + sub] = acc[q];
  if (sub == 0) {
    mine[BATCH * L] = maxVP;
    mine[BATCH * L + 1] = relV;
  }
  __syncthreads();
  // the epilogue, one lane to a node again
  const int64_t te = block * NODES + threadIdx.x;
  if (threadIdx.x < NODES && te < nInt) {
    const int64_t ke = work[te];
    const int le = rowCount[ke];
    const double* a = sums[threadIdx.x];
    double sum[COUNT];
#pragma unroll
    for (int q = 0; q < COUNT; ++q) sum[q] = a[q];
    Acc<D> ac = accOf<D>(sum);
    ac.maxVP = a[BATCH * L];
    if (o.relV) o.relV[ke] = le > 0 ? a[BATCH * L + 1] : -1.0;
    epilogue<D>(ke, le, selfOf(loadNbr<D, ISO, true>(rec, int32_t(ke))), ac, t, p, o);
  }
  storePairCount<kBlock>(pairs, nInt * L, pairCounts);
}

// ---------------------------------------------------------------------------
// Isotropic pair loop in collapsed form, FP32 (mixed precision) or FP64 (the
// search-order FP64 path).  Positions and per-node accumulators are FP64.
//
// With H = h I both unit vectors of a pair are r_hat = r_ij/|r_ij| and
// grad W = r_hat * h * dW/deta * det H, so the pair body reduces to scalars
// along r_hat: the acceleration increment is r_hat * m_j * (g_i (P_i/rho_i^2 +
// Q_i/2) + g_j (P_j/rho_j^2 + Q_j/2)) with g = h W' det H.  The two ends of a
// pair compute the same scalar from the same inputs (r_ij is the negated FP64
// difference, r_hat flips sign exactly), so the pair forces are antisymmetric
// up to the final product with the partner mass.  This reorders the
// reference's arithmetic: in FP64 the results agree with the reference-order
// kernel to round-off (the bar for search row order is 1e-12), in FP32 to the
// mixed-precision bar (1e-5).
//
// Neighbour records (written in pack.hh): the mixed record (MixedRec, 32 / 48 /
// 48 B in 1-D / 2-D / 3-D) and the FP64 record (96 B); both mark
// ghosts by a negative 1/h, and the reader forms det H = (1/h)^D.
// ---------------------------------------------------------------------------
template <typename Real> struct INbr {
  double x[3];
  uint32_t q[3];    // 3-D mixed: quantised position words
  Real hinv, hdet, m, invRho, v[3], cs, prho, mor;
  bool ghost;
};
template <int D>
__device__ __forceinline__ void loadIso(const float4* __restrict__ recM, int32_t j, INbr<float>& o) {
  const float4* p = recM + int64_t(j) * MixedRec<D>::F4;
  auto dbl = [](float lo, float hi) { return __hiloint2double(__float_as_int(hi), __float_as_int(lo)); };
  float h;
  if constexpr (D == 1) {
    const float4 f0 = p[0], f1 = p[1];
    o.x[0] = dbl(f0.x, f0.y); o.x[1] = 0.0; o.x[2] = 0.0;
    h = f0.z; o.m = f0.w;
    o.invRho = f1.x; o.v[0] = f1.y; o.v[1] = 0.0f; o.v[2] = 0.0f; o.cs = f1.z; o.prho = f1.w;
    o.mor = o.m * o.invRho;
  } else if constexpr (D == 2) {
    const float4 f0 = p[0], f1 = p[1], f2 = p[2];
    o.x[0] = dbl(f0.x, f0.y); o.x[1] = dbl(f0.z, f0.w); o.x[2] = 0.0;
    h = f1.x; o.m = f1.y; o.invRho = f1.z; o.v[0] = f1.w;
    o.v[1] = f2.x; o.v[2] = 0.0f; o.cs = f2.y; o.prho = f2.z; o.mor = f2.w;
  } else {
    const float4 f0 = p[0], f1 = p[1], f2 = p[2];
    o.q[0] = __float_as_uint(f0.x); o.q[1] = __float_as_uint(f0.y); o.q[2] = __float_as_uint(f0.z);
    h = f0.w;
    o.m = f1.x; o.invRho = f1.y; o.v[0] = f1.z; o.v[1] = f1.w;
    o.v[2] = f2.x; o.cs = f2.y; o.prho = f2.z; o.mor = f2.w;
  }
  o.ghost = h < 0.0f;
  o.hinv = fabsf(h);
  o.hdet = D == 1 ? o.hinv : (D == 2 ? o.hinv * o.hinv : o.hinv * o.hinv * o.hinv);
}
// det H of an exactly isotropic H is (1/h)^D evaluated as sdet evaluates it
// (the off-diagonal products are exact zeros), so the value is bitwise the
// packed one; m/rho is m * (1/rho), within an ulp.
template <int D>
__device__ __forceinline__ void loadIso(const double2* __restrict__ recD, int32_t j, INbr<double>& o) {
  const double2* p = recD + int64_t(j) * 6;
  const double2 d0 = p[0], d1 = p[1], d2 = p[2], d3 = p[3], e0 = p[4], e1 = p[5];
  o.x[0] = d0.x; o.x[1] = d0.y; o.x[2] = d1.x;
  o.ghost = d1.y < 0.0;
  const double hinv = fabs(d1.y);
  o.hinv = hinv;
  o.hdet = D == 1 ? hinv : (D == 2 ? hinv * hinv : (hinv * hinv) * hinv);
  o.m = d2.x; o.invRho = d2.y; o.cs = d3.x; o.prho = d3.y;
  o.mor = d2.x * d2.y;
  o.v[0] = e0.x; o.v[1] = e0.y; o.v[2] = e1.x;
}

template <int D>
__global__ void k_pack_mixed(const double* __restrict__ rec, int64_t n, int64_t nInt, double qInv,
                             float4* __restrict__ recM) {
  const int64_t k = blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
  if (k < n) writeMixedRec<D>(rec + k * RL<true>::STRIDE, nInt, qInv, recM + k * MixedRec<D>::F4);
}

template <int D>
__global__ void k_pack_fast64(const double* __restrict__ rec, int64_t n, int64_t nInt, double2* __restrict__ recD) {
  const int64_t k = blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
  if (k < n) writeFast64Rec<D>(rec + k * RL<true>::STRIDE, nInt, recD + k * 6);
}

template <int D>
__global__ void k_pack_dens_mixed(const double* __restrict__ rec, int64_t n, float4* __restrict__ recSM) {
  const int64_t k = blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
  if (k < n) writeDensRecMixed<D>(rec + k * RL<true>::STRIDE, recSM + k * DensMixedRec<D>::F4);
}

template <int D>
__global__ void k_pack_dens(const double* __restrict__ rec, int64_t n, double2* __restrict__ recS) {
  const int64_t k = blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
  if (k < n) writeDensRec<D>(rec + k * RL<true>::STRIDE, recS + k * 3);
}

// FP32 table in LDS: 8 floats per point.
template <bool LDS> __device__ __forceinline__ const float* stageTable32(float* lds, const TabArgs& t) {
  if constexpr (LDS) {
    for (int q = threadIdx.x; q < 8 * t.n; q += blockDim.x) lds[q] = t.g32[q];
    __syncthreads();
    return lds;
  } else {
    return t.g32;
  }
}
struct Tab32 {
  float invStep, extent;
  int n;
};
struct Tab64 {
  double invStep, extent;
  int n;
};

__device__ __forceinline__ float fmaR(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fmaR(double a, double b, double c) { return __builtin_fma(a, b, c); }
// reciprocal and reciprocal square root: the hardware approximations in FP32,
// refined by two Newton steps (error squared each step) in FP64
__device__ __forceinline__ float rcpR(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ double rcpR(double x) {
  double y = __builtin_amdgcn_rcp(x);
  y = __builtin_fma(y, __builtin_fma(-x, y, 1.0), y);
  return __builtin_fma(y, __builtin_fma(-x, y, 1.0), y);
}
__device__ __forceinline__ float rsqR(float x) { return __builtin_amdgcn_rsqf(x); }
__device__ __forceinline__ double rsqR(double x) {
  double y = __builtin_amdgcn_rsq(x);
  y = __builtin_fma(0.5 * y, __builtin_fma(-(x * y), y, 1.0), y);
  return __builtin_fma(0.5 * y, __builtin_fma(-(x * y), y, 1.0), y);
}
__device__ __forceinline__ float absR(float x) { return fabsf(x); }
__device__ __forceinline__ double absR(double x) { return fabs(x); }
__device__ __forceinline__ float maxR(float a, float b) { return fmaxf(a, b); }
__device__ __forceinline__ double maxR(double a, double b) { return fmax(a, b); }

__device__ __forceinline__ void lookupWGR(const float* __restrict__ tab, const Tab32& t, float eta, float hdet,
                                          float& W, float& gW) {
  if (eta < t.extent) {
    const float q = eta * t.invStep;
    int lb = int(q);
    lb = lb < t.n - 1 ? lb : t.n - 1;
    const int i0 = lb < t.n - 3 ? lb : t.n - 3;
    const float x = q - float(i0);
    const float4 a = *reinterpret_cast<const float4*>(tab + 8 * (i0 + 1));
    const float4 g = *reinterpret_cast<const float4*>(tab + 8 * (i0 + 1) + 4);
    W = hdet * __builtin_fmaf(__builtin_fmaf(a.z, x, a.y), x, a.x);
    gW = hdet * __builtin_fmaf(__builtin_fmaf(g.z, x, g.y), x, g.x);
  } else {
    W = 0.0f; gW = 0.0f;
  }
}
__device__ __forceinline__ void lookupWGR(const double* __restrict__ tab, const Tab64& t, double eta, double hdet,
                                          double& W, double& gW) {
  if (eta < t.extent) {
    const double q = eta * t.invStep;
    int lb = int(q);
    lb = lb < t.n - 1 ? lb : t.n - 1;
    const int i0 = lb < t.n - 3 ? lb : t.n - 3;
    const double x = q - double(i0);
    const double* c = tab + 6 * (i0 + 1);
    W = hdet * __builtin_fma(__builtin_fma(c[2], x, c[1]), x, c[0]);
    gW = hdet * __builtin_fma(__builtin_fma(c[5], x, c[4]), x, c[3]);
  } else {
    W = 0.0; gW = 0.0;
  }
}
__device__ __forceinline__ float lookupW32(const float* __restrict__ tab, const Tab32& t, float eta, float hdet) {
  if (!(eta < t.extent)) return 0.0f;
  const float q = eta * t.invStep;
  int lb = int(q);
  lb = lb < t.n - 1 ? lb : t.n - 1;
  const int i0 = lb < t.n - 3 ? lb : t.n - 3;
  const float x = q - float(i0);
  const float4 a = *reinterpret_cast<const float4*>(tab + 8 * (i0 + 1));
  return hdet * __builtin_fmaf(__builtin_fmaf(a.z, x, a.y), x, a.x);
}
template <typename Real>
__device__ __forceinline__ Real muQR(Real mu, Real Cl, Real Cq, Real cs, int linear, int quadratic) {
  const Real m0 = mu < Real(0) ? mu : Real(0);
  const Real lin = linear ? mu : m0;
  const Real quad = quadratic ? -(mu < Real(0) ? Real(-1) : Real(1)) * mu * mu : m0 * m0;
  return -Cl * cs * lin + Cq * quad;
}

template <int D, bool LDS, int L = 1>
__global__ void __launch_bounds__(kBlock) k_sum_density_mixed(double* __restrict__ rec, const float4* __restrict__ recSM,
                                                              const int32_t* __restrict__ rowCount,
                                                              const int32_t* __restrict__ nbr, int64_t n, int64_t nInt,
                                                              const int32_t* __restrict__ work, TabArgs t, Tab32 t32,
                                                              double W0, double* __restrict__ rhoOut,
                                                              const int32_t* __restrict__ slotList, int sumAll) {
  using R = RL<true>;
  extern __shared__ float lds32[];
  const float* tab = stageTable32<LDS>(lds32, t);
  const int64_t tw = (xcdBlock((nInt * L + kBlock - 1) / kBlock) * kBlock + threadIdx.x) / L;
  if (tw >= nInt) return;
  const int64_t k = work[tw];
  double* ri_ = rec + k * R::STRIDE;
  double xi[3] = {ri_[R::X], D > 1 ? ri_[R::X + 1] : 0.0, D > 2 ? ri_[R::X + 2] : 0.0};
  const double mi = ri_[R::M], hdeti = ri_[R::HDET];
  double acc = mi * (W0 * hdeti);
  const int len = rowCount[k];
  // the mixed density record: x (FP64 bits), 1/h, m
  auto load = [&](int32_t j, float4& a, float4& b) {
    const float4* p = recSM + int64_t(j) * DensMixedRec<D>::F4;
    a = p[0];
    if constexpr (D > 1) b = p[1];
    else b = make_float4(0.0f, 0.0f, a.z, a.w);
  };
  // several NodeLists: a pair across NodeLists counts with sumAll only, the
  // node taking its own mass (computeSPHSumMassDensity.cc:77-100)
  const int32_t lk = slotList ? slotList[k] : 0;
  const float mif = float(mi);
  auto term = [&](const float4 a, const float4 b, int32_t j) {
    float mj = b.w;
    if (slotList && slotList[j] != lk) {
      if (!sumAll) return -0.0;
      mj = mif;
    }
    const double xj[3] = {__hiloint2double(__float_as_int(a.y), __float_as_int(a.x)),
                          __hiloint2double(__float_as_int(a.w), __float_as_int(a.z)),
                          __hiloint2double(__float_as_int(b.y), __float_as_int(b.x))};
    float r2 = 0.0f;
    for (int c = 0; c < D; ++c) {
      const float rc = float(xi[c] - xj[c]);
      r2 = __builtin_fmaf(rc, rc, r2);
    }
    const float hj = b.z;
    const float hdetj = D == 1 ? hj : (D == 2 ? hj * hj : hj * hj * hj);
    const float eta = hj * __builtin_sqrtf(r2);
    return double(mj * lookupW32(tab, t32, eta, hdetj));
  };
  if constexpr (L > 1) {
    alignas(16) __shared__ double buf[kBlock];
    double* wbuf = buf + (threadIdx.x & ~63);
    const int sub = threadIdx.x % L;
    for (int w0 = 0; w0 < len; w0 += L) {
      const bool live = w0 + sub < len;
      const int32_t j = live ? nbr[ellIndex(w0 + sub, n, k)] : int32_t(k);
      float4 a, b;
      load(j, a, b);
      const double tm = term(a, b, j);
      acc = addInOrder<L>(acc, live ? tm : -0.0, wbuf);
    }
    if (sub != 0) return;
  } else {
    const int4* nb4 = reinterpret_cast<const int4*>(nbr);
    int4 cur = len > 0 ? nb4[ellChunk(0, n, k)] : make_int4(0, 0, 0, 0);
    int4 nxt = len > 4 ? nb4[ellChunk(1, n, k)] : make_int4(0, 0, 0, 0);
    float4 na, nb2;
    int32_t jn = cur.x;
    if (len > 0) load(jn, na, nb2);
    for (int w = 0; w < len; ++w) {
      const float4 a = na, b = nb2;
      const int32_t j = jn;
      if (w + 1 < len) {
        jn = nextIndex(nb4, n, k, len, w + 1, cur, nxt);
        load(jn, na, nb2);
      }
      acc += term(a, b, j);
    }
  }
  rhoOut[int64_t(ri_[R::ORIG])] = acc;
  const double som = ri_[R::SOM], p = ri_[R::P];
  ri_[R::RHO] = acc;
  ri_[R::PRHO] = som * p / (acc * acc);
  ri_[R::MOR] = mi / acc;
}

// The table of the collapsed pair loop: FP32 (8 floats per point) or FP64 (6
// doubles per point), staged in LDS.
template <typename Real> struct IsoTab;
template <> struct IsoTab<float> {
  using T = Tab32;
  using Rec = float4;
  using Elem = float;
  static constexpr int PER = 8;
};
template <> struct IsoTab<double> {
  using T = Tab64;
  using Rec = double2;
  using Elem = double;
  static constexpr int PER = 6;
};

// Mixed precision: the pair terms of up to kSumBlock consecutive neighbours
// are summed in FP32 (fused into the term's last product where it has one),
// and each block's partial sums are added once to the FP64 per-node
// accumulators: one conversion and one FP64 add per block instead of per
// entry.  A block's FP32 sum of 16 terms is within 16 u32 (1e-6) of its
// absolute sum; the per-node sums stay FP64.
constexpr int kSumBlock = 16;
template <int D> struct SumsF {
  float DvDt[D], xsphDV[D], DvDx[D * D], M[D * (D + 1) / 2], m2nd[D * (D + 1) / 2];
  float DepsDt, viscW, effVP, rhoSum, norm, wNS, xsphW;
  __device__ __forceinline__ void zero() {
    for (int c = 0; c < D; ++c) DvDt[c] = xsphDV[c] = 0.0f;
    for (int c = 0; c < D * D; ++c) DvDx[c] = 0.0f;
    for (int c = 0; c < D * (D + 1) / 2; ++c) M[c] = m2nd[c] = 0.0f;
    DepsDt = viscW = effVP = rhoSum = norm = wNS = xsphW = 0.0f;
  }
  // add into the FP64 accumulators (M and m2nd as upper triangles) and restart
  template <class Add> __device__ __forceinline__ void flushInto(Acc<D>& a, Add&& add) {
    auto to = [&](double& s, float v) { s = add(s, double(v)); };
    for (int c = 0; c < D; ++c) {
      to(a.DvDt.c[c], DvDt[c]);
      to(a.xsphDV.c[c], xsphDV[c]);
    }
    for (int c = 0; c < D * D; ++c) to(a.DvDx.c[c], DvDx[c]);
    int s2 = 0;
    for (int c = 0; c < D; ++c)
      for (int b = c; b < D; ++b, ++s2) {
        to(a.M.c[c * D + b], M[s2]);
        to(a.m2nd.c[s2], m2nd[s2]);
      }
    to(a.DepsDt, DepsDt);
    to(a.viscW, viscW);
    to(a.effVP, effVP);
    to(a.rhoSum, rhoSum);
    to(a.norm, norm);
    to(a.wNS, wNS);
    to(a.xsphW, xsphW);
    zero();
  }
};

// The node's own state for the epilogue, read again after the loop so that it
// holds no registers during it.
template <int D>
__device__ __forceinline__ void isoEpilogue(int64_t k, int len, const double* __restrict__ ri_, Acc<D>& a,
                                            const TabArgs& t, const PassArgs& p, const OutArgs& o) {
  using R = RL<true>;
  Self<D> me;
  for (int c = 0; c < D; ++c) me.v.c[c] = ri_[R::V + c];
  const double hinvD = ri_[RL<true>::HINV];
  for (int c = 0; c < NSym<D>::value; ++c) me.H.c[c] = 0.0;
  for (int c = 0; c < D; ++c) me.H.c[sdiag<D>(c)] = hinvD;
  me.Hdet = ri_[R::HDET]; me.m = ri_[R::M]; me.rho = ri_[R::RHO]; me.mor = ri_[R::MOR];
  epilogue<D>(k, len, me, a, t, p, o);
}

// The node's side of a pair.
template <typename Real, int D> struct IsoNode {
  double xi[3];
  uint32_t qi[3];
  Real vi[3];
  Real hi, ci, hdeti, invRhoi, rhoi2, Prhoi, mori, Cl, Cq, eps2;
};
// the 3-D mixed record holds quantised positions
template <typename Real, int D> constexpr bool kQPos = std::is_same<Real, float>::value && D == 3;
template <typename Real, int D>
__device__ __forceinline__ IsoNode<Real, D> loadIsoNode(const double* __restrict__ ri_, const PassArgs& p) {
  using R = RL<true>;
  IsoNode<Real, D> m;
  for (int c = 0; c < 3; ++c) {
    m.xi[c] = c < D ? ri_[R::X + c] : 0.0;
    if constexpr (kQPos<Real, D>) m.qi[c] = quantPos(m.xi[c], p.qInv);
    m.vi[c] = c < D ? Real(ri_[R::V + c]) : Real(0);
  }
  const double rho0 = ri_[R::RHO];
  m.hi = Real(ri_[RL<true>::HINV]);
  m.ci = Real(ri_[R::CS]);
  // det H as a neighbour's record gives it (from the same 1/h), so that the
  // two ends of a pair evaluate the same kernel gradient and their pair
  // terms are exact negatives of each other (FP64: the packed det H is
  // already that value)
  m.hdeti = std::is_same<Real, float>::value ? (D == 1 ? m.hi : (D == 2 ? m.hi * m.hi : m.hi * m.hi * m.hi))
                                             : Real(ri_[R::HDET]);
  m.invRhoi = Real(1.0 / rho0);
  m.rhoi2 = Real(rho0 * rho0);
  m.Prhoi = Real(ri_[R::PRHO]);
  m.mori = Real(ri_[R::MOR]);
  m.Cl = Real(p.Cl);
  m.Cq = Real(p.Cq);
  m.eps2 = Real(p.eps2);
  return m;
}

// One neighbour's factors of the sums.
template <typename Real, int D> struct IsoPair {
  Real rij[3], vij[3];
  Real Wi, absG, wg, fsr, f2, mv, pi, halfQi, Qi, morQi, w2, dsc;
};
template <typename Real, int D>
__device__ __forceinline__ IsoPair<Real, D> isoPair(const IsoNode<Real, D>& m, const INbr<Real>& nb,
                                                    const typename IsoTab<Real>::Elem* __restrict__ tab,
                                                    const typename IsoTab<Real>::T& tt, const PassArgs& p) {
  IsoPair<Real, D> o;
  Real r2 = Real(0), vdotr = Real(0);
  for (int c = 0; c < D; ++c) {
    if constexpr (kQPos<Real, D>) o.rij[c] = Real(int32_t(m.qi[c] - nb.q[c])) * p.qUnit;
    else o.rij[c] = Real(m.xi[c] - nb.x[c]);
    o.vij[c] = m.vi[c] - nb.v[c];
    r2 = fmaR(o.rij[c], o.rij[c], r2);
    vdotr = fmaR(o.vij[c], o.rij[c], vdotr);
  }
  const Real hi = m.hi, hj = nb.hinv;
  const Real rinv = r2 > Real(1.0e-30) ? rsqR(r2) : Real(0);
  const Real rmag = r2 * rinv;
  Real Wi, gWi, Wj, gWj;
  lookupWGR(tab, tt, hi * rmag, m.hdeti, Wi, gWi);
  lookupWGR(tab, tt, hj * rmag, nb.hdet, Wj, gWj);
  const Real gi = hi * gWi, gj = hj * gWj;     // grad W = r_hat * g
  // Monaghan-Gingold Q: mu = v_ij . eta / (eta^2 + eps2), eta = h r_ij
  // (FP64: one refined reciprocal of the product serves both ends)
  const Real da = fmaR(hi * hi, r2, m.eps2), db = fmaR(hj * hj, r2, m.eps2);
  Real ia, ib;
  if constexpr (std::is_same<Real, double>::value) {
    const Real inv = rcpR(da * db);
    ia = db * inv;
    ib = da * inv;
  } else {
    ia = rcpR(da);
    ib = rcpR(db);
  }
  const Real mui = hi * vdotr * ia;
  const Real muj = hj * vdotr * ib;
  const Real QPi = muQR(mui, m.Cl, m.Cq, m.ci, p.linearInExpansion, p.quadraticInExpansion) * m.invRhoi;
  const Real QPj = muQR(muj, m.Cl, m.Cq, nb.cs, p.linearInExpansion, p.quadraticInExpansion) * nb.invRho;
  o.Qi = m.rhoi2 * absR(QPi);
  const Real vdr = vdotr * rinv;                 // v_ij . r_hat
  o.halfQi = Real(0.5) * QPi * gi;
  o.pi = fmaR(gi, m.Prhoi, o.halfQi);
  const Real pj = fmaR(gj, nb.prho, Real(0.5) * QPj * gj);
  const Real mj = nb.m;
  o.fsr = mj * (o.pi + pj) * rinv;              // acceleration along r_ij
  o.wg = mj * gi * rinv;                       // grad W_i * m_j = r_ij * wg
  // gi^2 / max(1e-30, r^6); FP64 takes 1/r^6 from 1/r
  if constexpr (std::is_same<Real, double>::value) {
    const Real ri2 = rinv * rinv;
    o.f2 = r2 * r2 * r2 > Real(1.0e-30) ? gi * gi * (ri2 * ri2 * ri2) : gi * gi * Real(1.0e30);
  } else {
    o.f2 = gi * gi * rcpR(maxR(Real(1.0e-30), r2 * r2 * r2));
  }
  o.dsc = (o.pi + pj) * rinv;                   // compatible energy: the own-frame pair term along r_ij
  o.mv = mj * vdr;
  o.morQi = nb.mor * o.Qi;
  o.Wi = Wi;
  o.absG = absR(gWi);
  o.w2 = Real(0.5) * fmaR(m.mori, Wi, nb.mor * Wj);
  return o;
}

// L > 1 (mixed, small node sets): L lanes to a node, each taking whole blocks of
// kSumBlock entries, and the blocks' FP32 sums enter the FP64 sums in row order:
// the bits are those of one lane.
// RELV: the pass leaves the row maxima of the dt vote.  An instance of its own, so that
// the passes that leave none hold no register for them.  The 3-D mixed one is held to
// 168 VGPRs, three wavefronts per SIMD: it needs one register more and would run at two.
template <typename Real, int D, int L> constexpr bool kCanRelV = !std::is_same<Real, float>::value || (D == 3 && L == 1);
template <typename Real, int D, bool RELV>
constexpr int kIsoBlocks = RELV && std::is_same<Real, float>::value && D == 3 ? 3 : 1;
template <typename Real, int D, bool LDS, bool PREFETCH, int BS = kBlock, int L = 1, bool RELV = false>
__global__ void __launch_bounds__(BS, (kIsoBlocks<Real, D, RELV>)) k_derivs_iso(const double* __restrict__ rec,
                                                       const typename IsoTab<Real>::Rec* __restrict__ recN,
                                                       const int32_t* __restrict__ rowCount,
                                                       const int32_t* __restrict__ nbr, int64_t n, int64_t nInt,
                                                       const int32_t* __restrict__ work, TabArgs t,
                                                       typename IsoTab<Real>::T tt, PassArgs p, OutArgs o,
                                                       uint32_t* __restrict__ pairCounts) {
  using R = RL<true>;
  using E = typename IsoTab<Real>::Elem;
  constexpr bool F32 = std::is_same<Real, float>::value;
  static_assert(L == 1 || (F32 && !LDS), "several lanes to a node: mixed, the table through L1");
  static_assert(!RELV || kCanRelV<Real, D, L>, "no row maxima here");
  extern __shared__ double ldsIso[];
  const E* tab;
  if constexpr (LDS) {
    E* l = reinterpret_cast<E*>(ldsIso);
    const E* g = F32 ? reinterpret_cast<const E*>(t.g32) : reinterpret_cast<const E*>(t.g);
    for (int q = threadIdx.x; q < IsoTab<Real>::PER * t.n; q += blockDim.x) l[q] = g[q];
    __syncthreads();
    tab = l;
  } else {
    tab = F32 ? reinterpret_cast<const E*>(t.g32) : reinterpret_cast<const E*>(t.g);
  }
  const int64_t tw = (xcdBlock((nInt * L + BS - 1) / BS) * BS + threadIdx.x) / L;
  unsigned pairs = 0;
  if (tw < nInt) {
    const int64_t k = work[tw];
    const int32_t lk = p.slotList ? p.slotList[k] : 0;
    const double* ri_ = rec + k * R::STRIDE;
    const IsoNode<Real, D> me = loadIsoNode<Real, D>(ri_, p);

    Acc<D> a;
    a.zero();
    SumsF<F32 ? D : 1> af;
    if constexpr (F32) af.zero();
    Real maxVP = Real(0), relV = Real(0);
    const int len = rowCount[k];
    // One neighbour's contribution, in row order (w: its place in the row).
    auto pair = [&](const INbr<Real>& nb, int32_t j, int w) {
      pairs += (nb.ghost || j > int32_t(k)) ? 1u : 0u;
      const IsoPair<Real, D> q = isoPair<Real, D>(me, nb, tab, tt, p);
      if constexpr (RELV && !F32) {
        relV = dmax(relV, relSpeed<D>(q.vij));
      } else if constexpr (RELV) {
        float v2 = q.vij[0] * q.vij[0];
        for (int c = 1; c < D; ++c) v2 = fmaR(q.vij[c], q.vij[c], v2);
        relV = maxR(relV, v2);
      }
      maxVP = maxR(maxVP, q.Qi);
      if (o.pairDv)
        for (int c = 0; c < D; ++c) o.pairDv[int64_t(c) * o.plane + ellIndex(w, n, k)] = double(q.rij[c] * q.dsc);
      // several NodeLists: rhoSum and the normalization take same-NodeList
      // pairs only (SPHHydroBase.cc:746-751)
      const bool sameList = !p.slotList || p.slotList[j] == lk;
      auto addTo = [&](auto& b, auto* DvDt, auto* xsphDV, auto* DvDx, auto&& M, auto* m2nd) {
        for (int c = 0; c < D; ++c) DvDt[c] = fmaR(-q.rij[c], q.fsr, DvDt[c]);
        b.DepsDt = fmaR(q.mv, q.pi, b.DepsDt);
        b.viscW = fmaR(q.mv, q.halfQi, b.viscW);
        b.effVP = fmaR(q.morQi, q.Wi, b.effVP);
        if (sameList) {
          b.rhoSum = fmaR(nb.m, q.Wi, b.rhoSum);
          b.norm = fmaR(me.mori, q.Wi, b.norm);
        }
        b.wNS += q.absG;
        for (int c = 0; c < D; ++c) {
          const Real u = q.vij[c] * q.wg;
          for (int e = 0; e < D; ++e) DvDx[c * D + e] = fmaR(-u, q.rij[e], DvDx[c * D + e]);
        }
        int s2 = 0;
        for (int c = 0; c < D; ++c) {
          const Real rw = q.rij[c] * q.wg, rf = q.rij[c] * q.f2;
          for (int e = c; e < D; ++e, ++s2) {
            M(c, e, s2) = fmaR(-rw, q.rij[e], M(c, e, s2));
            m2nd[s2] = fmaR(rf, q.rij[e], m2nd[s2]);
          }
        }
        if (p.XSPH) {
          b.xsphW += q.w2;
          for (int c = 0; c < D; ++c) xsphDV[c] = fmaR(-q.vij[c], q.w2, xsphDV[c]);
        }
      };
      if constexpr (F32) {
        addTo(af, af.DvDt, af.xsphDV, af.DvDx, [&](int, int, int s2) -> float& { return af.M[s2]; }, af.m2nd);
      } else {
        // FP64, search row order: every accumulation fused
        addTo(a, a.DvDt.c, a.xsphDV.c, a.DvDx.c, [&](int c, int e, int) -> double& { return a.M.c[c * D + e]; },
              a.m2nd.c);
      }
    };
    if constexpr (L > 1) {
      alignas(16) __shared__ double buf[BS];
      double* wbuf = buf + (threadIdx.x & ~63);
      const int sub = threadIdx.x % L;
      for (int w0 = 0; w0 < len; w0 += L * kSumBlock) {
        const int wb = w0 + sub * kSumBlock;
        const int we = wb + kSumBlock < len ? wb + kSumBlock : len;
        for (int w = wb; w < we; ++w) {
          const int32_t j = nbr[ellIndex(w, n, k)];
          INbr<Real> nb;
          loadIso<D>(recN, j, nb);
          pair(nb, j, w);
        }
        af.flushInto(a, [&](double s, double v) { return addInOrder<L>(s, v, wbuf); });
      }
      a.maxVP = double(maxVP);
      for (int s = L / 2; s > 0; s >>= 1) a.maxVP = dmax(a.maxVP, __shfl_xor(a.maxVP, s));
    } else {
      const int4* nb4 = reinterpret_cast<const int4*>(nbr);
      int4 cur = len > 0 ? nb4[ellChunk(0, n, k)] : make_int4(0, 0, 0, 0);
      int4 nxt = len > 4 ? nb4[ellChunk(1, n, k)] : make_int4(0, 0, 0, 0);
      INbr<Real> nx;
      int32_t jn = cur.x;
      if (PREFETCH && len > 0) loadIso<D>(recN, jn, nx);
      for (int w = 0; w < len; ++w) {
        INbr<Real> nb;
        int32_t j;
        if constexpr (PREFETCH) {
          // the next record is loaded while this pair is evaluated
          nb = nx;
          j = jn;
          if (w + 1 < len) {
            jn = nextIndex(nb4, n, k, len, w + 1, cur, nxt);
            loadIso<D>(recN, jn, nx);
          }
        } else {
          // one record in flight per lane (fewer registers, more waves)
          j = w == 0 ? cur.x : nextIndex(nb4, n, k, len, w, cur, nxt);
          loadIso<D>(recN, j, nb);
        }
        pair(nb, j, w);
        if constexpr (F32) {
          if ((w & (kSumBlock - 1)) == kSumBlock - 1) af.flushInto(a, [](double s, double v) { return s + v; });
        }
      }
      if constexpr (F32) af.flushInto(a, [](double s, double v) { return s + v; });
      a.maxVP = double(maxVP);
    }
    if (L == 1 || threadIdx.x % L == 0) {
      for (int c = 0; c < D; ++c)
        for (int b = 0; b < c; ++b) a.M.c[c * D + b] = a.M.c[b * D + c];
      if constexpr (RELV) o.relV[k] = len > 0 ? double(relV) : -1.0;
      isoEpilogue<D>(k, len, ri_, a, t, p, o);
    }
  }
  storePairCount<BS>(pairs, nInt * L, pairCounts);
}

// The factors of the FP64 sums, one LDS row each, and each sum as the product of
// two of them (a fused multiply-add per entry): every sum of k_derivs_iso<double>
// is fma(A, B, sum) for the rows named here, to the bit (a sign moves between the
// factors exactly, and a plain addition is a factor of one).
template <int D> struct IsoRow {
  static constexpr int NR = 0, FSR = D, U = FSR + 1, RW = U + D, NRF = RW + D, MV = NRF + D, PI = MV + 1, HQ = PI + 1,
                       MQ = HQ + 1, WI = MQ + 1, MJ = WI + 1, MORI = MJ + 1, AG = MORI + 1, NW2 = AG + 1, V0 = NW2 + 1,
                       ONE = V0 + D, MONE = ONE + 1, COUNT = MONE + 1;
  static constexpr int SUMS = Sum<D>::COUNT - D * (D - 1) / 2;   // M by its upper triangle
  // rows of sum q, in the order of Acc's members below
  static constexpr int pack(int a, int b) { return a | (b << 8); }
  static __device__ __forceinline__ int rows(int q) {
    int at = 0;
    if (q < D) return pack(FSR, NR + q);                                   // DvDt
    at = D;
    if (q < at + D * D) return pack(U + (q - at) / D, NR + (q - at) % D);  // DvDx
    at += D * D;
    for (int c = 0; c < D; ++c)
      for (int e = c; e < D; ++e, ++at)
        if (q == at) return pack(RW + c, NR + e);                          // M
    for (int c = 0; c < D; ++c)
      for (int e = c; e < D; ++e, ++at)
        if (q == at) return pack(NRF + c, NR + e);                         // m2nd
    if (q < at + D) return pack(V0 + (q - at), NW2);                       // xsphDV
    at += D;
    switch (q - at) {
      case 0: return pack(MV, PI);        // DepsDt
      case 1: return pack(MV, HQ);        // viscW
      case 2: return pack(MQ, WI);        // effVP
      case 3: return pack(MJ, WI);        // rhoSum
      case 4: return pack(MORI, WI);      // norm
      case 5: return pack(AG, ONE);       // wNS
      case 6: return pack(NW2, MONE);     // xsphW
    }
    return pack(0, 0);
  }
  static __device__ __forceinline__ Acc<D> acc(const double* s) {
    Acc<D> a;
    int q = 0;
    for (int c = 0; c < D; ++c) a.DvDt.c[c] = s[q++];
    for (int c = 0; c < D * D; ++c) a.DvDx.c[c] = s[q++];
    for (int c = 0; c < D; ++c)
      for (int e = c; e < D; ++e) { a.M.c[c * D + e] = a.M.c[e * D + c] = s[q++]; }
    for (int c = 0; c < NSym<D>::value; ++c) a.m2nd.c[c] = s[q++];
    for (int c = 0; c < D; ++c) a.xsphDV.c[c] = s[q++];
    a.DepsDt = s[q++]; a.viscW = s[q++]; a.effVP = s[q++]; a.rhoSum = s[q++]; a.norm = s[q++]; a.wNS = s[q++];
    a.xsphW = s[q++];
    return a;
  }
};

// The FP64 collapsed pass with L lanes to a node (small node sets), bitwise
// k_derivs_iso<double>: a lane evaluates one entry of L and leaves its factors in
// LDS, then runs SUMS / L of the sums over the L entries, in row order.  Lanes
// past the row leave zeros (a sum that starts at +0 is never -0, so adding a
// zero product leaves it).
template <int D, int L>
__global__ void __launch_bounds__(kBlock) k_derivs_iso_rows(const double* __restrict__ rec,
                                                            const double2* __restrict__ recN,
                                                            const int32_t* __restrict__ rowCount,
                                                            const int32_t* __restrict__ nbr, int64_t n, int64_t nInt,
                                                            const int32_t* __restrict__ work, TabArgs t, Tab64 tt,
                                                            PassArgs p, OutArgs o, uint32_t* __restrict__ pairCounts) {
  using R = RL<true>;
  using W = IsoRow<D>;
  constexpr int BATCH = (W::SUMS + L - 1) / L, NODES = kBlock / L, PAD = 65;
  __shared__ double rows[kBlock / 64][W::COUNT][PAD];
  const int64_t block = xcdBlock((nInt * L + kBlock - 1) / kBlock);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, sub = threadIdx.x % L;
  const int64_t tw = block * NODES + threadIdx.x / L;
  unsigned pairs = 0;
  double maxVP = 0.0, relV = 0.0, sum[BATCH];
  int which[BATCH];
#pragma unroll
  for (int q = 0; q < BATCH; ++q) {
    sum[q] = 0.0;
    which[q] = W::rows(q * L + sub);
  }
  const int64_t k = tw < nInt ? work[tw] : 0;
  const int len = tw < nInt ? rowCount[k] : 0;
  const IsoNode<double, D> me = loadIsoNode<double, D>(rec + k * R::STRIDE, p);
  double(*row)[PAD] = rows[wave];
  row[W::ONE][lane] = 1.0;
  row[W::MONE][lane] = -1.0;
  for (int w0 = 0; w0 < len; w0 += L) {
    const int w = w0 + sub;
    const bool live = w < len;
    const int32_t j = live ? nbr[ellIndex(w, n, k)] : int32_t(k);
    INbr<double> nb;
    loadIso<D>(recN, j, nb);
    const IsoPair<double, D> q = isoPair<double, D>(me, nb, t.g, tt, p);
    if (live) {
      pairs += (nb.ghost || j > int32_t(k)) ? 1u : 0u;
      if (o.relV) relV = dmax(relV, relSpeed<D>(q.vij));
      maxVP = maxR(maxVP, q.Qi);
    }
    auto put = [&](int r, double v) { row[r][lane] = live ? v : 0.0; };
    for (int c = 0; c < D; ++c) {
      put(W::NR + c, -q.rij[c]);
      put(W::U + c, q.vij[c] * q.wg);
      put(W::RW + c, q.rij[c] * q.wg);
      put(W::NRF + c, -(q.rij[c] * q.f2));
      put(W::V0 + c, p.XSPH ? q.vij[c] : 0.0);
    }
    put(W::FSR, q.fsr); put(W::MV, q.mv); put(W::PI, q.pi); put(W::HQ, q.halfQi); put(W::MQ, q.morQi);
    put(W::WI, q.Wi); put(W::MJ, nb.m); put(W::MORI, me.mori); put(W::AG, q.absG);
    put(W::NW2, p.XSPH ? -q.w2 : 0.0);
    waveLdsOrder();
#pragma unroll
    for (int b = 0; b < BATCH; ++b) {
      const double* ra = row[which[b] & 0xff] + (lane - sub);
      const double* rb = row[which[b] >> 8] + (lane - sub);
      double s = sum[b];
#pragma unroll
      for (int e = 0; e < L; ++e) s = __builtin_fma(ra[e], rb[e], s);
      sum[b] = s;
    }
    waveLdsOrder();
  }
  for (int s = L / 2; s > 0; s >>= 1) {
    maxVP = dmax(maxVP, __shfl_xor(maxVP, s));
    relV = dmax(relV, __shfl_xor(relV, s));
  }
  // the epilogue, one lane to a node again: the sums through the same LDS
  __syncthreads();
  static_assert(sizeof(double) * NODES * (BATCH * L + 2) <= sizeof(rows), "the sums fit the rows' LDS");
  double(*sums)[BATCH * L + 2] = reinterpret_cast<double(*)[BATCH * L + 2]>(&rows[0][0][0]);
  double* mine = sums[threadIdx.x / L];
#pragma unroll
  for (int b = 0; b < BATCH; ++b) mine[b * L + sub] = sum[b];
  if (sub == 0) {
    mine[BATCH * L] = maxVP;
    mine[BATCH * L + 1] = relV;
  }
  __syncthreads();
  const int64_t te = block * NODES + threadIdx.x;
  if (threadIdx.x < NODES && te < nInt) {
    const int64_t ke = work[te];
    const int le = rowCount[ke];
    const double* sm = sums[threadIdx.x];
    Acc<D> a = W::acc(sm);
    a.maxVP = sm[BATCH * L];
    if (o.relV) o.relV[ke] = le > 0 ? sm[BATCH * L + 1] : -1.0;
    isoEpilogue<D>(ke, le, rec + ke * R::STRIDE, a, t, p, o);
  }
  storePairCount<kBlock>(pairs, nInt * L, pairCounts);
}

TabArgs tabArgs(const Sim& s) {
  return TabArgs{s.dTable.as<double>(), s.dTable32.as<float>(), s.table.n, s.table.step, s.table.extent,
                 s.dNperh.as<double>(), s.dWsum.as<double>()};
}

}  // namespace

PackIn packInputs(Sim& s) {
  return PackIn{s.perm.as<int32_t>(), s.pos.as<double>(), s.vel.as<double>(), s.mass.as<double>(),
                s.rho.as<double>(), s.P.as<double>(), s.cs.as<double>(), s.H.as<double>(), s.omega.as<double>(),
                s.hasMultipliers ? s.fCl.as<double>() : nullptr, s.hasMultipliers ? s.fCq.as<double>() : nullptr,
                s.hasMultipliers ? s.fshear.as<double>() : nullptr};
}

PackOut packOutputs(Sim& s, int sec) {
  const int64_t n = s.nSlots;
  const bool iso = s.isotropic;
  SG_REQUIRE(sec == 0 || iso, SPHGPU_ERR_STATE, "the pair kernels' records need H = h I");
  SG_REQUIRE((sec & 3) != 3, SPHGPU_ERR_STATE, "one pair-kernel record per pack");
  const int stride = iso ? RL<true>::STRIDE : RL<false>::STRIDE;
  s.rec.ensure(sizeof(double) * size_t(n) * stride);
  PackOut o{s.rec.as<double>(), nullptr, nullptr, n, s.nInt, nullptr, (sec & 1) ? quantInv(s) : 1.0};
  if (sec & 1) {
    s.recM.ensure(sizeof(float) * 16 * size_t(std::max<int64_t>(n, 1)));
    o.sec = s.recM.p;
  } else if (sec & 2) {
    s.recD.ensure(sizeof(double) * 12 * size_t(std::max<int64_t>(n, 1)));
    o.sec = s.recD.p;
  }
  if (sec & 4) {
    s.recS.ensure(sizeof(double) * DensRec::STRIDE * size_t(std::max<int64_t>(n, 1)));
    o.sec2 = s.recS.p;
  }
  if (sec & 8) {
    s.recSM.ensure(sizeof(float) * 8 * size_t(std::max<int64_t>(n, 1)));
    o.sec3 = s.recSM.p;
  }
  o.vel = nullptr;
  s.recSValid = (sec & 4) != 0;
  s.recSMValid = (sec & 8) != 0;
  s.pairRec = sec & 3;
  return o;
}

template <int D>
void launchPack(Sim& s, int sec, const int32_t* slots, int64_t count) {
  if (count <= 0) return;
  const PackOut o = packOutputs(s, sec);
  const PackIn in = packInputs(s);
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(nblocks(count)), dim3(kBlock), 0, s.stream, in, o, slots, count);
  };
  if (!s.isotropic) {
    go(k_pack<D, false, 0>);
  } else {
    switch (sec) {
      case 1: go(k_pack<D, true, 1>); break;
      case 2: go(k_pack<D, true, 2>); break;
      case 4: go(k_pack<D, true, 4>); break;
      case 5: go(k_pack<D, true, 5>); break;
      case 6: go(k_pack<D, true, 6>); break;
      case 8: go(k_pack<D, true, 8>); break;
      case 9: go(k_pack<D, true, 9>); break;
      default: go(k_pack<D, true, 0>); break;
    }
  }
  SG_CHECK_HIP(hipGetLastError());
}

// Records from the caller-order fields; sec bits 1 / 2 / 4 also write the
// mixed or FP64 isotropic pair kernel's record and the density sum's record
// in the same pass.
template <int D>
void packD(Sim& s, int sec = 0) {
  // With every slot live (no culled ghost), walk the caller rows so that the
  // field reads are contiguous and each slot's record is written whole; else
  // walk the slots, which also writes the dead ones.
  if (s.nSlots == s.nTot) launchPack<D>(s, sec, s.iperm.as<int32_t>(), s.nTot);
  else launchPack<D>(s, sec, nullptr, s.nSlots);
}

int pairRecordSec(const Sim& s, const sphgpu_hydro_params& hp) {
  const bool tensile = hp.epsTensile != 0.0;
  const bool compat = hp.compatibleEnergyEvolution != 0;
  if (hp.precision == SPHGPU_PRECISION_MIXED) return 1;
  // search row order is held to round-off of the reference sums, not to
  // their bits: the collapsed isotropic algebra in FP64 (one NodeList)
  return (s.rowOrder == SPHGPU_ROW_ORDER_SEARCH && s.isotropic && !tensile && !compat && s.nLists <= 1) ? 2 : 0;
}

int densityRecordSec(const Sim& s) {
  if (!s.isotropic) return 0;
  return s.precision == SPHGPU_PRECISION_MIXED ? 8 : 4;
}

namespace {

Tab32 tab32(const Sim& s) { return Tab32{float(1.0 / s.table.step), float(s.table.extent), s.table.n}; }

template <int D>
void packMixed(Sim& s) {
  s.recM.ensure(sizeof(float) * 16 * size_t(std::max<int64_t>(s.nSlots, 1)));
  hipLaunchKernelGGL(k_pack_mixed<D>, dim3(nblocks(s.nSlots)), dim3(kBlock), 0, s.stream, s.rec.as<double>(), s.nSlots,
                     s.nInt, quantInv(s), s.recM.as<float4>());
  s.pairRec = 1;
  SG_CHECK_HIP(hipGetLastError());
}

template <int D>
void packFast64(Sim& s) {
  s.recD.ensure(sizeof(double) * 12 * size_t(std::max<int64_t>(s.nSlots, 1)));
  hipLaunchKernelGGL(k_pack_fast64<D>, dim3(nblocks(s.nSlots)), dim3(kBlock), 0, s.stream, s.rec.as<double>(),
                     s.nSlots, s.nInt, s.recD.as<double2>());
  s.pairRec = 2;
  SG_CHECK_HIP(hipGetLastError());
}

Tab64 tab64(const Sim& s) { return Tab64{1.0 / s.table.step, s.table.extent, s.table.n}; }

__global__ void k_slot_lists(const int32_t* __restrict__ perm, const double* __restrict__ seg, int64_t nSlots,
                             int32_t* __restrict__ out) {
  const int64_t k = blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
  if (k < nSlots) {
    const int32_t i = perm[k];
    out[k] = i >= 0 ? int32_t(seg[i]) : -1;
  }
}

// Several NodeLists: the NodeList of every slot of the current build (for the
// collapsed kernels, whose records hold no caller index); null with one.
const int32_t* slotLists(Sim& s) {
  if (s.nLists <= 1) return nullptr;
  s.slotList.ensure(sizeof(int32_t) * size_t(std::max<int64_t>(s.nSlots, 1)));
  hipLaunchKernelGGL(k_slot_lists, dim3(nblocks(s.nSlots)), dim3(kBlock), 0, s.stream, s.perm.as<int32_t>(),
                     s.seg.as<double>(), s.nSlots, s.slotList.as<int32_t>());
  SG_CHECK_HIP(hipGetLastError());
  return s.slotList.as<int32_t>();
}

template <int D>
void sumDensityD(Sim& s) {
  const int64_t n = s.nSlots;
  TabArgs t = tabArgs(s);
  const bool lds = ldsTable(s);
  const size_t ldsBytes = lds ? sizeof(double) * 6 * size_t(s.table.n) : 0;
  if (!s.capturing) SG_CHECK_HIP(hipEventRecord(s.ev[2], s.stream));
  if (s.precision == SPHGPU_PRECISION_MIXED) {
    SG_REQUIRE(s.isotropic, SPHGPU_ERR_UNSUPPORTED, "mixed precision needs H = h I and no Q multipliers");
    if (!s.recSMValid) {
      s.recSM.ensure(sizeof(float) * 8 * size_t(std::max<int64_t>(n, 1)));
      hipLaunchKernelGGL(k_pack_dens_mixed<D>, dim3(nblocks(n)), dim3(kBlock), 0, s.stream, s.rec.as<double>(), n,
                         s.recSM.as<float4>());
      SG_CHECK_HIP(hipGetLastError());
      s.recSMValid = true;
    }
    const size_t lds32 = lds ? sizeof(float) * 8 * size_t(s.table.n) : 0;
    const double W0 = s.table.kernelValue(0.0, 1.0);
    const int32_t* lists = slotLists(s);
    auto go = [&](auto kern, int L, size_t ldsB) {
      hipLaunchKernelGGL(kern, dim3(xcdGrid(nblocks(s.nInt * L))), dim3(kBlock), ldsB, s.stream, s.rec.as<double>(),
                         s.recSM.as<float4>(), s.rowCount.as<int32_t>(), s.nbr.as<int32_t>(), n, s.nInt,
                         s.work.as<int32_t>(), t, tab32(s), W0, s.rho.as<double>(), lists, s.sumAllLists ? 1 : 0);
    };
    withLanes<D>(rowLanes(RowPass::kDensity, D, s.nInt), [&](auto lanes) {
      constexpr int L = decltype(lanes)::value;
      if (L > 1) go(k_sum_density_mixed<D, false, L>, L, 0);
      else if (lds) go(k_sum_density_mixed<D, true>, 1, lds32);
      else go(k_sum_density_mixed<D, false>, 1, 0);
    });
    SG_CHECK_HIP(hipGetLastError());
    applyGhostDensity(s);
    if (!s.capturing) SG_CHECK_HIP(hipEventRecord(s.ev[3], s.stream));
    return;
  }
  // isotropic H: neighbours from the 48-B density records
  if (s.isotropic && !s.recSValid) {
    s.recS.ensure(sizeof(double) * DensRec::STRIDE * size_t(std::max<int64_t>(n, 1)));
    hipLaunchKernelGGL(k_pack_dens<D>, dim3(nblocks(n)), dim3(kBlock), 0, s.stream, s.rec.as<double>(), n,
                       s.recS.as<double2>());
    SG_CHECK_HIP(hipGetLastError());
    s.recSValid = true;
  }
  const double* nrec = s.isotropic ? s.recS.as<double>() : s.rec.as<double>();
  const double* listOf = s.nLists > 1 ? s.seg.as<double>() : nullptr;
  auto go = [&](auto kern, int L, size_t ldsB) {
    hipLaunchKernelGGL(kern, dim3(xcdGrid(nblocks(s.nInt * L))), dim3(kBlock), ldsB, s.stream, s.rec.as<double>(),
                       s.rowCount.as<int32_t>(), s.nbr.as<int32_t>(), n, s.nInt, s.work.as<int32_t>(), t,
                       s.rho.as<double>(), nrec, listOf, s.sumAllLists ? 1 : 0);
  };
  withLanes<D>(rowLanes(s.isotropic ? RowPass::kDensity : RowPass::kDensityAnyH, D, s.nInt), [&](auto lanes) {
    constexpr int L = decltype(lanes)::value;
    auto any = [&](auto iso) {
      constexpr bool ISO = decltype(iso)::value;
      if (L > 1) go(k_sum_density<D, ISO, false, L>, L, 0);
      else if (lds) go(k_sum_density<D, ISO, true>, 1, ldsBytes);
      else go(k_sum_density<D, ISO, false>, 1, 0);
    };
    if (s.isotropic) any(std::true_type{}); else any(std::false_type{});
  });
  SG_CHECK_HIP(hipGetLastError());
  // SPHHydroBase::finalize then applies the boundaries to the mass density
  applyGhostDensity(s);
  if (!s.capturing) SG_CHECK_HIP(hipEventRecord(s.ev[3], s.stream));
}

// The collapsed isotropic pair kernel with BS-thread workgroups, its table in
// LDS or read through L1.  Tuning variant v: with a table that fits in LDS,
// BS = 64 << (v / 2) and the table in LDS when v is odd; otherwise BS = 64 << v.
template <typename Real> typename IsoTab<Real>::T isoTable(const Sim& s);
template <> Tab32 isoTable<float>(const Sim& s) { return tab32(s); }
template <> Tab64 isoTable<double>(const Sim& s) { return tab64(s); }
template <typename Real, int D, bool PF, int BS, int L = 1>
void isoLaunch(Sim& s, bool inLds, hipStream_t st, int64_t n, const TabArgs& t, const PassArgs& p, const OutArgs& o,
               uint32_t* counts) {
  using Rec = typename IsoTab<Real>::Rec;
  const Rec* recN = reinterpret_cast<const Rec*>(std::is_same<Real, float>::value ? s.recM.p : s.recD.p);
  const size_t lb = inLds ? sizeof(typename IsoTab<Real>::Elem) * IsoTab<Real>::PER * size_t(s.table.n) : 0;
  const dim3 g(unsigned(xcdGrid(nblocks(s.nInt * L, BS)))), b(BS);
  auto go = [&](auto kern, size_t ldsB) {
    hipLaunchKernelGGL(kern, g, b, ldsB, st, s.rec.as<double>(), recN, s.rowCount.as<int32_t>(), s.nbr.as<int32_t>(), n,
                       s.nInt, s.work.as<int32_t>(), t, isoTable<Real>(s), p, o, counts);
  };
  auto tables = [&](auto relV) {
    constexpr bool RELV = decltype(relV)::value;
    if (L == 1 && inLds) go(k_derivs_iso<Real, D, L == 1, PF, BS, L, RELV>, lb);
    else go(k_derivs_iso<Real, D, false, PF, BS, L, RELV>, 0);
  };
  if constexpr (kCanRelV<Real, D, L>) {
    if (o.relV) return tables(std::true_type{});
  }
  tables(std::false_type{});
}
template <typename Real, int D, bool PF>
void isoVariant(Sim& s, int v, bool fits, hipStream_t st, int64_t n, const TabArgs& t, const PassArgs& p,
                const OutArgs& o, uint32_t* counts) {
  const int bsLog = fits ? v >> 1 : v;
  const bool inLds = fits && (v & 1);
  if constexpr (D == 3) {
    isoLaunch<Real, D, PF, 256>(s, inLds, st, n, t, p, o, counts);
  } else {
    switch (bsLog) {
      case 0: isoLaunch<Real, D, PF, 64>(s, inLds, st, n, t, p, o, counts); break;
      case 1: isoLaunch<Real, D, PF, 128>(s, inLds, st, n, t, p, o, counts); break;
      case 2: isoLaunch<Real, D, PF, 256>(s, inLds, st, n, t, p, o, counts); break;
      default: isoLaunch<Real, D, PF, 512>(s, inLds, st, n, t, p, o, counts); break;
    }
  }
  SG_CHECK_HIP(hipGetLastError());
}

template <int D>
void evalDerivsD(Sim& s, const sphgpu_hydro_params& hp, bool updateOnly, bool relV) {
  const int64_t n = s.nSlots;
  hipStream_t st = s.stream;
  const int total = derivTotalDoubles(s.dim);
  s.out.ensure(sizeof(double) * size_t(n) * total);
  s.outStride = n;
  // the pair kernel decides the record it reads
  const bool tensile = hp.epsTensile != 0.0;
  const bool compat = hp.compatibleEnergyEvolution != 0;
  const bool mixed = hp.precision == SPHGPU_PRECISION_MIXED;
  if (mixed)
    SG_REQUIRE(s.isotropic && !tensile, SPHGPU_ERR_UNSUPPORTED,
               "mixed precision needs H = h I, no Q multipliers and epsTensile = 0");
  const int sec = pairRecordSec(s, hp);
  const bool fast64 = sec == 2;
  // lanes to a node: mixed blocks need rows of several blocks, so 1-D keeps one
  const int lanes = mixed ? mixedLanes(D, s.nInt)
                          : rowLanes(fast64 ? RowPass::kIsoPairs
                                            : !s.isotropic ? RowPass::kPairsAnyH
                                                           : compat ? RowPass::kPairsStored : RowPass::kPairs,
                                     D, s.nInt);
  s.pairWaves = (s.nInt * lanes + 63) / 64;
  s.pairCounts.ensure(sizeof(uint32_t) * size_t(std::max<int64_t>(s.pairWaves, 1)));
  uint32_t* counts = s.pairCounts.as<uint32_t>();

  if (!s.capturing) SG_CHECK_HIP(hipEventRecord(s.ev[4], st));
  if (!s.recValid) {
    packD<D>(s, sec);
    s.recValid = true;
  } else if (sec == 1 && s.pairRec != 1) {
    packMixed<D>(s);
  } else if (sec == 2 && s.pairRec != 2) {
    packFast64<D>(s);
  }
  if (!s.capturing) SG_CHECK_HIP(hipEventRecord(s.ev[5], st));

  TabArgs t = tabArgs(s);
  const bool lds = ldsTable(s);
  const size_t ldsBytes = lds ? sizeof(double) * 6 * size_t(s.table.n) : 0;
  PassArgs p{};
  p.Cl = hp.Cl; p.Cq = hp.Cq; p.eps2 = hp.eps2; p.epsTensile = hp.epsTensile; p.nPerh = hp.nPerh;
  p.hmin = hp.hmin; p.hmax = hp.hmax;
  p.W0 = s.table.kernelValue(0.0, 1.0);
  p.WnPerh = s.table.kernelValue(1.0 / hp.nPerh, 1.0);
  p.XSPH = hp.XSPH; p.correctVelocityGradient = hp.correctVelocityGradient; p.evolveTotalEnergy = hp.evolveTotalEnergy;
  p.linearInExpansion = hp.linearInExpansion; p.quadraticInExpansion = hp.quadraticInExpansion;
  p.qInv = mixed ? quantInv(s) : 1.0;
  p.qUnit = float(1.0 / p.qInv);
  p.listOf = s.nLists > 1 ? s.seg.as<double>() : nullptr;
  p.slotList = mixed ? slotLists(s) : nullptr;
  OutArgs o{};
  o.base = s.out.as<double>();
  o.n = n;
  o.updateOnly = updateOnly ? 1 : 0;
  if (relV) {
    SG_REQUIRE(!mixed || (D == 3 && lanes == 1), SPHGPU_ERR_STATE, "mixed row maxima: 3-D, one lane to a node");
    s.relV.ensure(sizeof(double) * size_t(std::max<int64_t>(n, 1)));
    o.relV = s.relV.as<double>();
  }
  for (int f = 0; f < SPHGPU_NUM_DERIV_FIELDS; ++f) o.off[f] = derivOffsetDoubles(s.dim, f);
  if (compat) {
    // pairAccelerations: the own-frame pair term of every row entry
    o.plane = n * int64_t(s.ellCap);
    s.pairDv.ensure(sizeof(double) * size_t(D) * size_t(std::max<int64_t>(o.plane, 1)));
    o.pairDv = s.pairDv.as<double>();
  }
  // Mixed: one record in flight per lane keeps the kernel at 167 VGPRs, three
  // wavefronts per SIMD (2.11 ms at 128^3 against 2.53 ms with the next
  // record prefetched at 179 VGPRs, two wavefronts).  The pass that leaves the
  // vote's row maxima spills two registers to stay at three: 2.05 ms where a pass
  // without them takes 2.00.  FP64: the prefetch wins (3.44 ms at 194 VGPRs
  // against 3.51 ms at 168).
  if (mixed && lanes > 1) {
    if constexpr (D > 1) isoLaunch<float, D, false, kBlock, D == 3 ? 8 : 2>(s, false, st, n, t, p, o, counts);
    SG_CHECK_HIP(hipGetLastError());
  } else if (fast64 && lanes > 1) {
    withLanes<D>(lanes, [&](auto ln) {
      constexpr int L = decltype(ln)::value;
      if constexpr (L > 1)
        hipLaunchKernelGGL((k_derivs_iso_rows<D, L>), dim3(xcdGrid(nblocks(s.nInt * L))), dim3(kBlock), 0, st,
                           s.rec.as<double>(), s.recD.as<double2>(), s.rowCount.as<int32_t>(), s.nbr.as<int32_t>(), n,
                           s.nInt, s.work.as<int32_t>(), t, tab64(s), p, o, counts);
    });
  } else if (mixed || fast64) {
    // 1-D and 2-D (ensembles, serving): the workgroup size and the table's
    // place (LDS or read through L1) are autotuned per workload class.  3-D
    // runs 256-thread workgroups with the table in LDS when it fits.
    const bool fits = s.table.n <= kLdsTablePoints;
    const int nv = fits ? 8 : 4;
    auto run = [&](int v) {
      if (mixed) isoVariant<float, D, false>(s, v, fits, st, n, t, p, o, counts);
      else isoVariant<double, D, true>(s, v, fits, st, n, t, p, o, counts);
    };
    const int def = fits ? (4 + (lds ? 1 : 0)) : 2;      // 256 threads, the row-length rule for the table
    int v = def;
    if (D < 3) {
      const double perNode = s.nInt > 0 ? double(s.nEntries) / double(s.nInt) : 0.0;
      v = tunedVariant(s, tuneKey(kTunePairIso, D, mixed ? 1 : 0, perNode, s.nInt), nv, def, run);
    }
    run(v);
  } else {
    auto launch = [&](auto kern) {
      hipLaunchKernelGGL(kern, dim3(xcdGrid(nblocks(s.nInt))), dim3(kBlock), ldsBytes, st, s.rec.as<double>(),
                         s.rowCount.as<int32_t>(), s.nbr.as<int32_t>(), n, s.nInt, s.work.as<int32_t>(), t, p, o,
                         counts);
    };
    if (lanes > 1) {
      withLanes<D>(lanes, [&](auto ln) {
        constexpr int L = decltype(ln)::value;
        if constexpr (L > 1) {
          auto any = [&](auto iso, auto tens) {
            hipLaunchKernelGGL((k_derivs_rows<D, decltype(iso)::value, decltype(tens)::value, L>),
                               dim3(xcdGrid(nblocks(s.nInt * L))), dim3(kBlock), 0, st, s.rec.as<double>(),
                               s.rowCount.as<int32_t>(), s.nbr.as<int32_t>(), n, s.nInt, s.work.as<int32_t>(), t, p, o,
                               counts);
          };
          const std::true_type yes{};
          const std::false_type no{};
          if (s.isotropic) { if (tensile) any(yes, yes); else any(yes, no); }
          else { if (tensile) any(no, yes); else any(no, no); }
        }
      });
    } else {
      auto any = [&](auto iso, auto tens, auto relv) {
        constexpr bool ISO = decltype(iso)::value, TENSILE = decltype(tens)::value, RELV = decltype(relv)::value;
        if (lds) launch(k_derivs_fp64<D, ISO, TENSILE, true, RELV>);
        else launch(k_derivs_fp64<D, ISO, TENSILE, false, RELV>);
      };
      auto votes = [&](auto iso, auto tens) {
        if (relV) any(iso, tens, std::true_type{});
        else any(iso, tens, std::false_type{});
      };
      const std::true_type yes{};
      const std::false_type no{};
      if (s.isotropic) { if (tensile) votes(yes, yes); else votes(yes, no); }
      else { if (tensile) votes(no, yes); else votes(no, no); }
    }
  }
  SG_CHECK_HIP(hipGetLastError());
  if (!s.capturing) SG_CHECK_HIP(hipEventRecord(s.ev[6], st));
}

}  // namespace

template <int D>
void omegaGradhD(Sim& s) {
  const int64_t n = s.nSlots;
  TabArgs t = tabArgs(s);
  const bool lds = ldsTable(s);
  const size_t ldsBytes = lds ? sizeof(double) * 6 * size_t(s.table.n) : 0;
  auto go = [&](auto kern, int L, size_t ldsB) {
    hipLaunchKernelGGL(kern, dim3(xcdGrid(nblocks(s.nInt * L))), dim3(kBlock), ldsB, s.stream, s.rec.as<double>(),
                       s.rowCount.as<int32_t>(), s.nbr.as<int32_t>(), n, s.nInt, s.work.as<int32_t>(), t,
                       s.omega.as<double>());
  };
  withLanes<D>(rowLanes(s.isotropic ? RowPass::kOmega : RowPass::kOmegaAnyH, D, s.nInt), [&](auto lanes) {
    constexpr int L = decltype(lanes)::value;
    auto any = [&](auto iso) {
      constexpr bool ISO = decltype(iso)::value;
      if (L > 1) go(k_omega<D, ISO, false, L>, L, 0);
      else if (lds) go(k_omega<D, ISO, true>, 1, ldsBytes);
      else go(k_omega<D, ISO, false>, 1, 0);
    };
    if (s.isotropic) any(std::true_type{}); else any(std::false_type{});
  });
  SG_CHECK_HIP(hipGetLastError());
}

void omegaGradh(Sim& s) {
  SG_REQUIRE(s.neighborsValid, SPHGPU_ERR_STATE, "the grad-h correction needs a neighbour build");
  SG_REQUIRE(s.table.n > 0, SPHGPU_ERR_STATE, "no kernel table installed");
  if (!s.recValid) packRecords(s);
  if (s.dim == 1) omegaGradhD<1>(s);
  else if (s.dim == 2) omegaGradhD<2>(s);
  else omegaGradhD<3>(s);
  // SPHHydroBase::initialize applies the boundaries to omega
  applyGhostScalar(s, s.omega);
  s.recValid = false;         // records hold safeInv(omega)
  s.derivsValid = false;
}

// One iterateIdealH pass (src/Utilities/iterateIdealH.cc:139-230) with the
// SPH smoothing scale: one lane per internal node; a node whose last change is
// within tol keeps its H, the others take zeroth = rootnu(sum over the row of
// |W.gradValue(|H_i x_ij|, 1)|) in row order, H1 = idealSmoothingScale, and the
// change max|phi - 1| over the eigenvalues c/lambda(H_i) of H1^1/2 H_i^-1 H1^1/2
// (H1 = c I).  Node i reads only its own H (neighbour positions come from
// the records), so H is replaced in place.
// L > 1: L lanes to a node (its rows are of one length in a wavefront, nearly).
template <int D, bool ISO, bool LDS, int L = 1>
__global__ void __launch_bounds__(kBlock) k_ideal_h(const double* __restrict__ rec, const int32_t* __restrict__ rowCount,
                                                    const int32_t* __restrict__ nbr, int64_t n, int64_t nInt,
                                                    const int32_t* __restrict__ work, const int32_t* __restrict__ perm,
                                                    TabArgs t, double nPerh, double hmin, double hmax, double tol,
                                                    double* __restrict__ H, double* __restrict__ deltaH,
                                                    unsigned long long* __restrict__ maxBits,
                                                    const double* __restrict__ listOf) {
  using R = RL<ISO>;
  constexpr int NS = NSym<D>::value;
  extern __shared__ double lds[];
  const double* tab = stageTable<LDS>(lds, t);
  const int64_t block = xcdBlock((nInt * L + kBlock - 1) / kBlock);
  const int64_t tw = (block * kBlock + threadIdx.x) / L;
  double zeroth = 0.0, d = 0.0;
  bool open = false;      // the node still iterates
  if (tw < nInt) {
    const int64_t k = work[tw];
    const int64_t i = perm[k];
    open = deltaH[i] > tol;
    if (open) {
      S<D> Hi;
      for (int c = 0; c < NS; ++c) Hi.c[c] = H[i * NS + c];
      const double* ri_ = rec + k * R::STRIDE;
      V<D> xi;
      for (int c = 0; c < D; ++c) xi.c[c] = ri_[R::X + c];
      // several NodeLists: a neighbour of another NodeList counts with
      // m_j rho_i / (m_i rho_j) (iterateIdealH.cc:183-194)
      const double li = listOf ? listOf[i] : 0.0, mi = ri_[R::M], rhoi = ri_[R::RHO];
      const int len = rowCount[k];
      auto term = [&](int32_t j) {
        const double* rj = rec + int64_t(j) * R::STRIDE;
        V<D> xij;
        for (int c = 0; c < D; ++c) xij.c[c] = xi.c[c] - rj[R::X + c];
        const double etai = vmag(sdot(Hi, xij));
        double Wv, gW;
        lookupWG(tab, t, etai, 1.0, Wv, gW);
        double fw = 1.0;
        if (listOf && listOf[int64_t(rj[R::ORIG])] != li) fw = rj[R::M] * rhoi / (mi * rj[R::RHO]);
        return fw * dabs(gW);
      };
      if constexpr (L > 1) {
        // (a node done earlier leaves its lanes out of the exchange as a group)
        alignas(16) __shared__ double buf[kBlock];
        double* wbuf = buf + (threadIdx.x & ~63);
        const int sub = threadIdx.x % L;
        for (int w0 = 0; w0 < len; w0 += L) {
          const bool live = w0 + sub < len;
          const double tm = term(live ? nbr[ellIndex(w0 + sub, n, k)] : int32_t(k));
          zeroth = addInOrder<L>(zeroth, live ? tm : -0.0, wbuf);
        }
      } else {
        // four entries at a time: their four records are in flight together
        // (40^3 nodes: 104 us one by one, 88 us)
        const int4* nb4 = reinterpret_cast<const int4*>(nbr);
        for (int w = 0; w < len; w += 4) {
          const int4 j = nb4[ellChunk(w / 4, n, k)];
          const int32_t self = int32_t(k);
          const double t0 = term(j.x), t1 = term(w + 1 < len ? j.y : self);
          const double t2 = term(w + 2 < len ? j.z : self), t3 = term(w + 3 < len ? j.w : self);
          zeroth += t0;
          zeroth += w + 1 < len ? t1 : -0.0;
          zeroth += w + 2 < len ? t2 : -0.0;
          zeroth += w + 3 < len ? t3 : -0.0;
        }
      }
    }
  }
  // The root, the table's inverse and the eigenvalues take as long as a row: one
  // lane to a node again, in as few wavefronts as hold them.
  int64_t te = tw;
  if constexpr (L > 1) {
    __shared__ double sums[kBlock / L];
    __shared__ int still[kBlock / L];
    if (threadIdx.x % L == 0) {
      sums[threadIdx.x / L] = zeroth;
      still[threadIdx.x / L] = open;
    }
    __syncthreads();
    open = threadIdx.x < kBlock / L && still[threadIdx.x % (kBlock / L)];
    zeroth = sums[threadIdx.x % (kBlock / L)];
    te = block * (kBlock / L) + threadIdx.x;
  }
  if (open) {
    const int64_t i = perm[work[te]];
    S<D> Hi;
    for (int c = 0; c < NS; ++c) Hi.c[c] = H[i * NS + c];
    zeroth = rootnu<D>(zeroth);
    const double c1 = idealHinv(t, zeroth, Hi.c[0], nPerh, hmin, hmax);
    const double phimin = c1 / maxEigen<D>(Hi.c), phimax = c1 / minEigen<D>(Hi.c);
    d = dmax(dabs(phimin - 1.0), dabs(phimax - 1.0));
    deltaH[i] = d;
    int q = 0;
    for (int a = 0; a < D; ++a)
      for (int b = a; b < D; ++b, ++q) H[i * NS + q] = (a == b) ? c1 : 0.0;
  }
  for (int sh = 32; sh > 0; sh >>= 1) d = dmax(d, __shfl_xor(d, sh));
  if ((threadIdx.x & 63) == 0 && d > 0.0) atomicMax(maxBits, (unsigned long long)__double_as_longlong(d));
}

template <int D>
double idealHPassD(Sim& s, const sphgpu_hydro_params& hp, double tol, double* deltaH, unsigned long long* bits) {
  const int64_t n = s.nSlots;
  TabArgs t = tabArgs(s);
  const bool lds = ldsTable(s);
  const size_t ldsBytes = lds ? sizeof(double) * 6 * size_t(s.table.n) : 0;
  auto go = [&](auto kern, int L, size_t ldsB) {
    hipLaunchKernelGGL(kern, dim3(xcdGrid(nblocks(s.nInt * L))), dim3(kBlock), ldsB, s.stream, s.rec.as<double>(),
                       s.rowCount.as<int32_t>(), s.nbr.as<int32_t>(), n, s.nInt, s.work.as<int32_t>(),
                       s.perm.as<int32_t>(), t, hp.nPerh, hp.hmin, hp.hmax, tol, s.H.as<double>(), deltaH, bits,
                       s.nLists > 1 ? s.seg.as<double>() : nullptr);
  };
  withLanes<D>(rowLanes(RowPass::kIdealH, D, s.nInt), [&](auto lanes) {
    constexpr int L = decltype(lanes)::value;
    auto any = [&](auto iso) {
      constexpr bool ISO = decltype(iso)::value;
      if (L > 1) go(k_ideal_h<D, ISO, false, L>, L, 0);
      else if (lds) go(k_ideal_h<D, ISO, true>, 1, ldsBytes);
      else go(k_ideal_h<D, ISO, false>, 1, 0);
    };
    if (s.isotropic) any(std::true_type{}); else any(std::false_type{});
  });
  SG_CHECK_HIP(hipGetLastError());
  unsigned long long hb = 0;
  SG_CHECK_HIP(hipMemcpyAsync(&hb, bits, sizeof(hb), hipMemcpyDeviceToHost, s.stream));
  SG_CHECK_HIP(hipStreamSynchronize(s.stream));
  double m;
  std::memcpy(&m, &hb, sizeof(m));
  return m;
}

double idealHPass(Sim& s, const sphgpu_hydro_params& hp, double tol, double* deltaH, unsigned long long* bits) {
  SG_REQUIRE(s.neighborsValid, SPHGPU_ERR_STATE, "the ideal H pass needs a neighbour build");
  SG_REQUIRE(s.table.n > 0, SPHGPU_ERR_STATE, "no kernel table installed");
  if (!s.recValid) packRecords(s);
  double m;
  if (s.dim == 1) m = idealHPassD<1>(s, hp, tol, deltaH, bits);
  else if (s.dim == 2) m = idealHPassD<2>(s, hp, tol, deltaH, bits);
  else m = idealHPassD<3>(s, hp, tol, deltaH, bits);
  s.recValid = false;
  s.derivsValid = false;
  return m;
}

void packRecords(Sim& s, int sec) {
  if (s.dim == 1) packD<1>(s, sec);
  else if (s.dim == 2) packD<2>(s, sec);
  else packD<3>(s, sec);
  s.recValid = true;
}

void sumDensity(Sim& s) {
  SG_REQUIRE(s.neighborsValid, SPHGPU_ERR_STATE, "sum density needs a neighbour build");
  SG_REQUIRE(s.table.n > 0, SPHGPU_ERR_STATE, "no kernel table installed");
  if (!s.recValid) {
    if (s.isotropic) {
      // the records and the density kernel's own record in one pass
      const int sec = densityRecordSec(s);
      if (s.dim == 1) packD<1>(s, sec);
      else if (s.dim == 2) packD<2>(s, sec);
      else packD<3>(s, sec);
      s.recValid = true;
    } else {
      packRecords(s);
    }
  }
  if (s.dim == 1) sumDensityD<1>(s);
  else if (s.dim == 2) sumDensityD<2>(s);
  else sumDensityD<3>(s);
  s.pairRec = 0;      // the density changed rho in the records
  if (!s.capturing) s.timingPending |= 2u;
  s.derivsValid = false;
}

void evalDerivs(Sim& s, const sphgpu_hydro_params& p, bool updateOnly, bool relV) {
  SG_REQUIRE(s.neighborsValid, SPHGPU_ERR_STATE, "evaluateDerivatives needs a neighbour build");
  SG_REQUIRE(s.table.n > 0, SPHGPU_ERR_STATE, "no kernel table installed");
  SG_REQUIRE(!(p.compatibleEnergyEvolution && p.evolveTotalEnergy), SPHGPU_ERR_ARG,
             "compatibleEnergyEvolution and evolveTotalEnergy exclude each other");
  SG_REQUIRE(p.precision == SPHGPU_PRECISION_FP64 || p.precision == SPHGPU_PRECISION_MIXED, SPHGPU_ERR_ARG,
             "unknown precision");
  SG_REQUIRE(p.nPerh > 0.0, SPHGPU_ERR_ARG, "nPerh must be positive");
  s.derivsValid = false;
  if (s.dim == 1) evalDerivsD<1>(s, p, updateOnly, relV);
  else if (s.dim == 2) evalDerivsD<2>(s, p, updateOnly, relV);
  else evalDerivsD<3>(s, p, updateOnly, relV);
  if (!s.capturing) s.timingPending |= 4u;
  s.derivsValid = true;
  s.pairsValid = true;
}

int derivComponents(int dim, int f) {
  const int ns = nsymOf(dim);
  switch (f) {
    case SPHGPU_D_DXDT: case SPHGPU_D_DVDT: case SPHGPU_D_XSPH_DELTA_V: return dim;
    case SPHGPU_D_DVDX: case SPHGPU_D_LOCAL_DVDX: case SPHGPU_D_M: case SPHGPU_D_LOCAL_M: return dim * dim;
    case SPHGPU_D_DHDT: case SPHGPU_D_HIDEAL: case SPHGPU_D_MASS_SECOND_MOMENT: return ns;
    default: return 1;
  }
}
int derivOffsetDoubles(int dim, int f) {
  int o = 0;
  for (int q = 0; q < f; ++q) o += derivComponents(dim, q);
  return o;
}
int derivTotalDoubles(int dim) { return derivOffsetDoubles(dim, SPHGPU_NUM_DERIV_FIELDS); }

}  // namespace sphgpu
