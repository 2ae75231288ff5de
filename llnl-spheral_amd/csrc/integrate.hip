// Time integration on the device: GammaLawGas, GenericHydro::dt and
// SynchronousRK2::step with the SPH state policies.
//
// Step (src/Integrator/SynchronousRK2.cc:78-144):
//   ghosts + neighbours (Integrator::preStepInitialize -> setGhostNodes),
//   dt = selectDt(GenericHydro::dt) with dtGrowth and the dtMin/dtMax clamps,
//   derivatives at t, state0 <- state, update by dt/2, ghosts,
//   derivatives at t + dt/2, state <- state0 updated by dt with them, ghosts,
//   SPHHydroBase::finalize (sum density with the step's neighbour rows),
//   Integrator::enforceBoundaries.
// State::update with the policies of SPHHydroBase::registerState
// (src/SPH/SPHHydroBase.cc:238-336) on the internal rows:
//   x += m*DxDt, v += m*DvDt, eps += m*DepsDt          (IncrementFieldList)
//   rho = min(rhoMax, max(rhoMin, rho + m*DrhoDt))      (IncrementBoundedState)
//   H = ideal H with eigenvalues bounded by 1/hmax, 1/hmin (ReplaceBoundedState;
//       the SPH ideal H is h1^-1 I, so the bound is a clamp of the diagonal)
//   P, c from the gamma-law EOS                         (Pressure/SoundSpeedPolicy)
// With compatibleEnergyEvolution, eps follows SpecificThermalEnergyPolicy
// (src/Hydro/SpecificThermalEnergyPolicy.cc:64-189): eps += m*DepsDt with
// DepsDt rebuilt from the pair accelerations of the pass and the step-start
// velocities.
// The state is walked in caller order and the derivative fields gathered from
// each row's slot.
#include "internal.hh"
#include "dgeom.hh"
#include "eigen.hh"
#include "ell.hh"
#include "pack.hh"
#include "lanes.hh"
#include <cfloat>
#include <cstring>
#include <algorithm>
#include <mutex>

namespace sphgpu {

namespace {

constexpr int kBlock = 256;
inline int nblocks(int64_t n, int bs = kBlock) { return int(std::max<int64_t>(1, (n + bs - 1) / bs)); }

struct Eos {
  double gamma, gamma1, Pmin, Pmax;
  int floor;
};
// GammaLawGas::pressure with applyPressureLimits, soundSpeed
__device__ __forceinline__ double eosP(const Eos& e, double rho, double eps) {
  const double P = e.gamma1 * rho * eps;
  return P < e.Pmin ? (e.floor ? e.Pmin : 0.0) : (P > e.Pmax ? e.Pmax : P);
}
__device__ __forceinline__ double eosCs(const Eos& e, double eps) { return sqrt(dmax(0.0, e.gamma * e.gamma1 * eps)); }

__global__ void k_eos(const double* __restrict__ rho, const double* __restrict__ eps, double* __restrict__ P,
                      double* __restrict__ cs, int64_t n, Eos e) {
  const int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
  if (i >= n) return;
  P[i] = eosP(e, rho[i], eps[i]);
  cs[i] = eosCs(e, eps[i]);
}

struct Fields {
  double *pos, *vel, *eps, *rho, *H, *P, *cs;
};
struct Base {
  double *pos, *vel, *eps, *rho;
};
struct DerivIn {
  const double* base;  // field-major blocks of the last evaluation, slot rows
  int64_t n;
  int oDx, oDv, oDeps, oDrho, oHid, oVP, oDvDx;
  const double* compDe;  // compatible energy: DepsDt of the policy per slot, else null
};
struct Bounds {
  double rhoMin, rhoMax, hmaxInv, hminInv;
};
// Ensemble members: the update's multiplier (dt or dt/2) and gamma per member.
struct SelectArgs {
  double cfl, dtMin, dtMax, dtGrowth;
};
// Integrator::selectDt of one member from its vote (src/Integrator/Integrator.cc:167-212):
// a handful of operations on uniform values, so every kernel that needs dt
// forms it again from the vote rather than waiting for a launch that does.
__device__ __forceinline__ double selectDt(const SegState& g, const SelectArgs& a) {
  const double dtMin = dmin(a.dtMin, g.tEnd - g.t), dtMax = dmin(a.dtMax, g.tEnd - g.t);
  const double vote = a.cfl * __longlong_as_double((long long)g.voteBits);
  double dt = dtMax;
  if (vote > 0.0 && vote < dt) dt = vote;
  dt = dmin(dt, a.dtGrowth * g.lastDt);
  return dmin(dtMax, dmax(dtMin, dt));
}
struct SegArgs {
  const double* seg;        // member of each row; null: one simulation
  SegState* st;
  int half;                 // 1: multiply by dt/2
  SelectArgs sel;
  const double* listOf = nullptr;      // several NodeLists with their own gamma-law EOS:
  const double* listGamma = nullptr;   //   each row's NodeList, and the NodeLists' gammas
};
// The update's multiplier and the EOS of row i.
__device__ __forceinline__ void rowMultEos(const SegArgs& sa, int64_t i, double& mult, Eos& e) {
  if (sa.listGamma) {
    const double g = sa.listGamma[int(sa.listOf[i])];
    e.gamma = g;
    e.gamma1 = g - 1.0;
  }
  const SegState& g = sa.st[sa.seg ? int(sa.seg[i]) : 0];
  const double dt = selectDt(g, sa.sel);
  mult = sa.half ? 0.5 * dt : dt;
  if (!sa.seg) return;
  e.gamma = g.gamma;
  e.gamma1 = g.gamma - 1.0;
}

// REC >= 0: also write the slot's records (pack sec bits REC, isotropic
// layout) from the values just stored, as the record pack would.
// TRIAL: the update to t + dt/2 starts from the state itself and saves it as
// state0 (b) on the way, in place of copies of the whole state before it (at
// 128^3 five copies of 235 MB in all, of which H was never read back).  The
// final update starts from b and leaves the dt vote's inputs of the next step
// (maxViscousPressure, tr DvDx, DvDt by caller index) in dtIn.
// One lane per caller row: its eleven state arrays are then read and written
// contiguously, and only the five derivatives are gathered from its slot (an
// internal row's slot is iperm[i]).  By slot it was the other way round.
// In 2-D the lines of the slots that a row touches are touched again a few hundred
// rows on: each XCD takes a run of workgroups, so they meet in one L2 (500^2: 33.5 ->
// 27.1 us and 30.9 -> 24.7 us).  In 3-D they come again planes later, and the runs
// cost 4 % at 128^3.
template <int D, int REC, bool TRIAL>
__global__ void __launch_bounds__(kBlock) k_update(const int32_t* __restrict__ iperm, int64_t nInt, Fields f, Base b,
                                                   DerivIn d, Bounds bd, Eos e, SegArgs sa, PackIn pin, PackOut pout,
                                                   double* __restrict__ dtIn) {
  constexpr int NS = NSym<D>::value;
  const int64_t i = (D == 2 ? xcdBlock((nInt + kBlock - 1) / kBlock) : blockIdx.x) * int64_t(kBlock) + threadIdx.x;
  if (i >= nInt) return;
  const int64_t k = iperm[i];
  double mult;
  rowMultEos(sa, i, mult, e);
  const double* dx = d.base + int64_t(d.oDx) * d.n + k * D;
  const double* dv = d.base + int64_t(d.oDv) * d.n + k * D;
  PackRow<D> w;
  double dvc[D];
  for (int c = 0; c < D; ++c) {
    const double x0 = (TRIAL ? f.pos : b.pos)[i * D + c], v0 = (TRIAL ? f.vel : b.vel)[i * D + c];
    if (TRIAL) { b.pos[i * D + c] = x0; b.vel[i * D + c] = v0; }
    dvc[c] = dv[c];
    w.x.c[c] = x0 + mult * dx[c];
    w.v.c[c] = v0 + mult * dvc[c];
    f.pos[i * D + c] = w.x.c[c];
    f.vel[i * D + c] = w.v.c[c];
  }
  const double eps0 = (TRIAL ? f.eps : b.eps)[i], rho0 = (TRIAL ? f.rho : b.rho)[i];
  if (TRIAL) { b.eps[i] = eps0; b.rho[i] = rho0; }
  const double eps = d.compDe ? eps0 + d.compDe[k] * mult : eps0 + mult * d.base[int64_t(d.oDeps) * d.n + k];
  const double rho = dmin(bd.rhoMax, dmax(bd.rhoMin, rho0 + mult * d.base[int64_t(d.oDrho) * d.n + k]));
  f.eps[i] = eps;
  f.rho[i] = rho;
  const double* hid = d.base + int64_t(d.oHid) * d.n + k * NS;
  int c = 0;
  for (int a = 0; a < D; ++a)
    for (int q = a; q < D; ++q, ++c) {
      w.h.c[c] = (a == q) ? dmin(bd.hminInv, dmax(bd.hmaxInv, hid[c])) : hid[c];
      f.H[i * NS + c] = w.h.c[c];
    }
  const double P = eosP(e, rho, eps), cs = eosCs(e, eps);
  f.P[i] = P;
  f.cs[i] = cs;
  if constexpr (REC >= 0) {
    w.rho = rho;
    w.P = P;
    w.cs = cs;
    w.m = pin.mass[i];
    w.omega = pin.omega[i];
    packRow<D, true, REC>(k, i, w, pout);
  }
  if constexpr (!TRIAL) {
    constexpr int W = 2 + D;
    dtIn[i * W] = d.base[int64_t(d.oVP) * d.n + k];
    const double* g = d.base + int64_t(d.oDvDx) * d.n + k * D * D;
    double tr = g[0];
    for (int a = 1; a < D; ++a) tr = tr + g[a * D + a];
    dtIn[i * W + 1] = tr;
    for (int c2 = 0; c2 < D; ++c2) dtIn[i * W + 2 + c2] = dvc[c2];
  }
  // an ensemble member whose state turns non-finite fails alone (the step's
  // final update; NaN at the midpoint reaches it)
  if (!TRIAL && sa.seg) {
    bool ok = isfinite(eps) && isfinite(rho) && isfinite(P) && isfinite(cs);
    for (int c2 = 0; c2 < D; ++c2) ok = ok && isfinite(w.x.c[c2]) && isfinite(w.v.c[c2]);
    for (int c2 = 0; c2 < NS; ++c2) ok = ok && isfinite(w.h.c[c2]);
    if (!ok) atomicOr(&sa.st[int(sa.seg[i])].fail, unsigned(SPHGPU_MEMBER_NONFINITE));
  }
}

template <int D> __device__ __forceinline__ double vmagArr(const double* a) {
  if constexpr (D == 1) return dabs(a[0]);
  double s = a[0] * a[0];
  for (int c = 1; c < D; ++c) s = s + a[c] * a[c];
  return sqrt(s);
}

// GenericHydro::dt candidates of one internal node; the minimum over all
// nodes is reduced with one 64-bit atomic min per wavefront on the bit
// pattern of the (positive) candidate.
// Where the pair limit's velocities come from:
//   kVoteRows   the caller-order velocities of the row's nodes (sphgpu_hydro_dt)
//   kVoteSlots  velocities packed by slot with the build (a mixed step, whose pair
//               kernel holds FP32 velocities: the vote stays FP64); four
//               neighbours' loads in flight
//   kVoteDone   the row maxima the FP64 pass at the step start left (relV)
//   kVoteBounds the FP32 row maxima a large mixed step's pass left: bounds of the
//               FP64 maximum.  The upper end of each pair limit enters the vote, the
//               lower goes to `low`, and k_dt_exact gathers the FP64 velocities of
//               the rows whose lower end lies under the vote: the row that decides is
//               among them, so the result is the gather's, to the bit.  100^3: 0.42 ms
//               for the gather of all rows, 0.10 for the two and 0.04 more in each pass
// An entry that would not lower the minimum is left out (a plain read may be
// stale, then the atomic decides): 32 k atomics on one word were 0.3 ms of the
// vote at 128^3.
__device__ __forceinline__ void enterMin(unsigned long long* p, double m) {
  const unsigned long long v = (unsigned long long)__double_as_longlong(m);
  if (v < *static_cast<volatile unsigned long long*>(p)) atomicMin(p, v);
}
enum { kVoteRows, kVoteSlots, kVoteDone, kVoteBounds };
struct VoteArgs {
  const int32_t *list, *perm, *rowCount, *nbr;   // list: kVoteDone, kVoteBounds caller row -> slot, else the work list
  int64_t n, nInt;
  const double *H, *cs, *rho, *vel, *dtIn;
  int haveDtIn;
  double nPerh;
  int useVelMag;
  const double* seg;
  const double *velS, *relV;
  double* low;
};
// The largest |v_ij|^2 (1-D: |v_ij|) of slot k's row from the velocities packed by
// slot, four neighbours' loads in flight.
template <int D>
__device__ __forceinline__ double rowRelSpeed(const VoteArgs& a, int64_t k, int len, const double* vi) {
  const int4* nb4 = reinterpret_cast<const int4*>(a.nbr);
  double r = 0.0;
  for (int w = 0; w < len; w += 4) {
    const int4 j4 = nb4[ellChunk(w >> 2, a.n, k)];
    const int32_t j[4] = {j4.x, j4.y, j4.z, j4.w};
    double d[4][3];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const double* p = a.velS + int64_t(w + q < len ? j[q] : j[0]) * velStride(D);
      if constexpr (D == 1) {
        d[q][0] = p[0];
      } else {
        const double2 lo = reinterpret_cast<const double2*>(p)[0];
        d[q][0] = lo.x;
        d[q][1] = lo.y;
        if constexpr (D == 3) d[q][2] = p[2];
      }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      for (int c = 0; c < D; ++c) d[q][c] = vi[c] - d[q][c];
      double s = D == 1 ? dabs(d[q][0]) : d[q][0] * d[q][0];
      for (int c = 1; c < D; ++c) s = s + d[q][c] * d[q][c];
      r = dmax(r, s);
    }
  }
  return r;
}
template <int D> __device__ __forceinline__ double pairLimit(double nodeScale, double speed) {
  return nodeScale * (1.0 / dmax(1.0e-30, speed));
}
template <int D, int FROM>
__global__ void __launch_bounds__(kBlock) k_dt(VoteArgs a, unsigned long long* __restrict__ minBits, int64_t minStride) {
  constexpr int NS = NSym<D>::value;
  // rows in slot order where neighbours are gathered, else in caller order
  const int64_t t = xcdBlock((a.nInt + kBlock - 1) / kBlock) * kBlock + threadIdx.x;
  double m = double(FLT_MAX);
  int sg = 0;
  if (t < a.nInt) {
    int64_t k, i;
    if constexpr (FROM == kVoteDone || FROM == kVoteBounds) {
      i = t;
      k = a.list[i];
    } else {
      k = a.list[t];
      i = a.perm[k];
    }
    if (a.seg) sg = int(a.seg[i]);
    const double nodeScale = 1.0 / maxEigen<D>(a.H + i * NS) / a.nPerh;
    m = dmin(m, nodeScale / (a.cs[i] + FLT_MIN));
    constexpr int W = 2 + D;
    double vp = 0.0, divv = 0.0, acc[3] = {0.0, 0.0, 0.0};
    if (a.haveDtIn) {
      vp = a.dtIn[i * W];
      divv = a.dtIn[i * W + 1];
      for (int c = 0; c < D; ++c) acc[c] = a.dtIn[i * W + 2 + c];
    }
    const double csq = sqrt(vp / a.rho[i]);
    m = dmin(m, nodeScale / (csq + FLT_MIN));
    m = dmin(m, 1.0 / (dabs(divv) + FLT_MIN));
    double vi[3];
    for (int c = 0; c < D; ++c) vi[c] = a.vel[i * D + c];
    if constexpr (FROM == kVoteDone) {
      const double r = a.relV[k];
      if (r >= 0.0) m = dmin(m, pairLimit<D>(nodeScale, D == 1 ? r : sqrt(r)));
    } else if constexpr (FROM == kVoteBounds) {
      const double r = a.relV[k];
      double low = double(FLT_MAX);
      if (r >= 0.0) {
        // FP32 velocities are within u |v| of theirs (u = 2^-24), so the maximum is
        // within u (2 |v_i| + 4 M) of M; three times that, and room for products
        // that underflow.  Speeds near the end of the FP32 range give no bounds.
        const double M = sqrt(r), vm = vmagArr<D>(vi), err = 4.0e-7 * vm + 6.0e-7 * M + 1.0e-18;
        const bool safe = r < 1.0e36 && vm < 1.0e18;
        low = safe ? pairLimit<D>(nodeScale, M + err) : 0.0;
        if (safe) m = dmin(m, pairLimit<D>(nodeScale, M - err));
      }
      a.low[i] = low;
    } else if constexpr (FROM == kVoteSlots) {
      // the pair term is monotonic in |v_ij|^2, to the bit: one square root a row
      const int len = a.rowCount[k];
      const double r = rowRelSpeed<D>(a, k, len, vi);
      if (len > 0) m = dmin(m, pairLimit<D>(nodeScale, D == 1 ? r : sqrt(r)));
    } else {
      const int len = a.rowCount[k];
      for (int w = 0; w < len; ++w) {
        const int64_t j = a.perm[a.nbr[ellIndex(w, a.n, k)]];
        double d[3];
        for (int c = 0; c < D; ++c) d[c] = vi[c] - a.vel[j * D + c];
        m = dmin(m, nodeScale * (1.0 / dmax(1.0e-30, vmagArr<D>(d))));
      }
    }
    m = dmin(m, sqrt(nodeScale / (vmagArr<D>(acc) + FLT_MIN)));
    if (a.useVelMag) m = dmin(m, nodeScale / (vmagArr<D>(vi) + 1.0e-10));
  }
  const int s0 = __shfl(sg, 0);
  if (__all(sg == s0)) {
    for (int sh = 32; sh > 0; sh >>= 1) m = dmin(m, __shfl_xor(m, sh));
    if ((threadIdx.x & 63) == 0) enterMin(minBits + s0 * minStride, m);
  } else if (t < a.nInt) {
    enterMin(minBits + sg * minStride, m);
  }
}

// The rows that k_dt<D, kVoteBounds> left open, one lane to a caller row.
template <int D>
__global__ void __launch_bounds__(kBlock) k_dt_exact(VoteArgs a, unsigned long long* __restrict__ minBits,
                                                     int64_t minStride) {
  const int64_t i = blockIdx.x * int64_t(kBlock) + threadIdx.x;
  if (i >= a.nInt) return;
  unsigned long long* word = minBits + (a.seg ? int64_t(a.seg[i]) * minStride : 0);
  if (!(a.low[i] <= __longlong_as_double((long long)*static_cast<volatile unsigned long long*>(word)))) return;
  const int64_t k = a.list[i];
  const int len = a.rowCount[k];
  if (len == 0) return;
  double vi[3];
  for (int c = 0; c < D; ++c) vi[c] = a.vel[i * D + c];
  const double r = rowRelSpeed<D>(a, k, len, vi);
  const double nodeScale = 1.0 / maxEigen<D>(a.H + i * NSym<D>::value) / a.nPerh;
  enterMin(word, dmin(double(FLT_MAX), pairLimit<D>(nodeScale, D == 1 ? r : sqrt(r))));
}

template <int D, int FROM>
void voteD(Sim& s, double nPerh, int useVelMag, const double* seg, unsigned long long* bits, int64_t stride) {
  if (FROM == kVoteBounds) s.voteLow.ensure(sizeof(double) * size_t(std::max<int64_t>(s.nInt, 1)));
  VoteArgs a{FROM == kVoteDone || FROM == kVoteBounds ? s.iperm.as<int32_t>() : s.work.as<int32_t>(), s.perm.as<int32_t>(),
             s.rowCount.as<int32_t>(), s.nbr.as<int32_t>(), s.nSlots, s.nInt, s.H.as<double>(), s.cs.as<double>(),
             s.rho.as<double>(), s.vel.as<double>(), s.dtIn.as<double>(), s.haveDtIn ? 1 : 0, nPerh, useVelMag, seg,
             s.velS.as<double>(), s.relV.as<double>(), s.voteLow.as<double>()};
  hipLaunchKernelGGL((k_dt<D, FROM>), dim3(xcdGrid(nblocks(s.nInt))), dim3(kBlock), 0, s.stream, a, bits, stride);
  if constexpr (FROM == kVoteBounds)
    hipLaunchKernelGGL(k_dt_exact<D>, dim3(nblocks(s.nInt)), dim3(kBlock), 0, s.stream, a, bits, stride);
  SG_CHECK_HIP(hipGetLastError());
}

__global__ void k_set_u64(unsigned long long* p, unsigned long long v) { *p = v; }
__global__ void k_fill_value(double* __restrict__ a, int64_t n, double v) {
  const int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
  if (i < n) a[i] = v;
}

// ---- SpecificThermalEnergyPolicy ------------------------------------------
// DvDt and DepsDt of the internal slots to caller order; the ghost rows are
// then filled by the boundaries (SPHHydroBase::finalizeDerivatives).
template <int D>
__global__ void k_compat_scatter(const int32_t* __restrict__ work, const int32_t* __restrict__ perm, int64_t nInt,
                                 const double* __restrict__ out, int64_t n, int oDv, int oDeps,
                                 double* __restrict__ acc, double* __restrict__ de0) {
  const int64_t t = blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
  if (t >= nInt) return;
  const int64_t k = work[t];
  const int64_t i = perm[k];
  for (int c = 0; c < D; ++c) acc[i * D + c] = out[int64_t(oDv) * n + k * D + c];
  de0[i] = out[int64_t(oDeps) * n + k];
}

// Per slot: v + a hdt, |DepsDt0| + epsilon, m and the caller index (the pair
// owner is the node of smaller caller index).  Dead slots are in no row.
template <int D>
__global__ void k_compat_rec(const int32_t* __restrict__ perm, int64_t nSlots, const double* __restrict__ vel0,
                             const double* __restrict__ acc, const double* __restrict__ de0,
                             const double* __restrict__ mass, SegArgs sa, double* __restrict__ crec) {
  const int64_t k = blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
  if (k >= nSlots) return;
  const int64_t i = perm[k];
  double r[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  if (i >= 0) {
    Eos unused{};
    double mult;
    rowMultEos(sa, i, mult, unused);
    const double hdt = 0.5 * mult;
    for (int c = 0; c < D; ++c) r[c] = vel0[i * D + c] + acc[i * D + c] * hdt;
    r[3] = dabs(de0[i]) + DBL_EPSILON;
    r[4] = mass[i];
    r[5] = double(i);
  }
  double2* o = reinterpret_cast<double2*>(crec + k * 8);
  o[0] = make_double2(r[0], r[1]);
  o[1] = make_double2(r[2], r[3]);
  o[2] = make_double2(r[4], r[5]);
}

// DepsDt of one internal node, gathered along its row.  The row holds the
// pass's own-frame pair term dv of each neighbour j; the reference's pair
// accelerations are -m_j dv for the node's own pairs (i owns when its caller
// index is the smaller) and m_i dv for the neighbour's end of a pair j owns.
// The owner end receives w_i du, the other end (1 - w_i) du m_i/m_j, written
// here from the receiving node with the owner's operands in the reference's
// order.  With rows in caller-index order the sum runs in the reference's
// order (owners j < i ascending, then the node's own pairs).
// L > 1: L lanes to a node (lanes.hh).  One lane to a node waits for each
// entry's record in turn; eight have theirs in flight together, and a term costs
// far more than the exchange, so two and three dimensions take them at any size.
template <int D, int L>
__global__ void __launch_bounds__(kBlock) k_compat(const int32_t* __restrict__ work, const int32_t* __restrict__ rowCount,
                                                   const int32_t* __restrict__ nbr, int64_t n, int64_t nInt,
                                                   const double* __restrict__ crec, const double* __restrict__ pairDv,
                                                   int64_t plane, double* __restrict__ compDe) {
  const int64_t t = (xcdBlock((nInt * L + kBlock - 1) / kBlock) * kBlock + threadIdx.x) / L;
  if (t >= nInt) return;
  const int64_t k = work[t];
  const double2* mr = reinterpret_cast<const double2*>(crec + k * 8);
  const double2 a0 = mr[0], a1 = mr[1], a2 = mr[2];
  const double vi[3] = {a0.x, a0.y, a1.x};
  const double wti = a1.y, mi = a2.x, oi = a2.y;
  double de = 0.0;
  const int len = rowCount[k];
  auto term = [&](int64_t e) {
    const double2* nr = reinterpret_cast<const double2*>(crec + int64_t(nbr[e]) * 8);
    const double2 b0 = nr[0], b1 = nr[1], b2 = nr[2];
    const double vj[3] = {b0.x, b0.y, b1.x};
    const double wtj = b1.y, mj = b2.x, oj = b2.y;
    double du = 0.0;
    if (oj > oi) {
      for (int c = 0; c < D; ++c) {
        const double pa = pairDv[int64_t(c) * plane + e] * (-mj);
        const double tc = (vj[c] - vi[c]) * pa;
        du = (c == 0) ? tc : du + tc;
      }
      const double wi = wti / (wti + wtj);
      return wi * du;
    }
    for (int c = 0; c < D; ++c) {
      const double pa = pairDv[int64_t(c) * plane + e] * mi;
      const double tc = (vi[c] - vj[c]) * pa;
      du = (c == 0) ? tc : du + tc;
    }
    const double wj = wtj / (wtj + wti);
    return (1.0 - wj) * du * mj / mi;
  };
  if constexpr (L > 1) {
    alignas(16) __shared__ double buf[kBlock];
    double* wbuf = buf + (threadIdx.x & ~63);
    const int sub = threadIdx.x % L;
    for (int w0 = 0; w0 < len; w0 += L) {
      const double v = w0 + sub < len ? term(ellIndex(w0 + sub, n, k)) : -0.0;
      de = addInOrder<L>(de, v, wbuf);
    }
    if (sub == 0) compDe[k] = de;
  } else {
    for (int w = 0; w < len; ++w) de += term(ellIndex(w, n, k));
    compDe[k] = de;
  }
}

Eos makeEos(double gamma, double Pmin, double Pmax, int floor) { return Eos{gamma, gamma - 1.0, Pmin, Pmax, floor}; }

// SpecificThermalEnergyPolicy::update's DepsDt into s.compDe (slot rows) for
// the update of `sa`, with vel0 the step-start velocities (every row).
template <int D> void compatD(Sim& s, const double* vel0, const SegArgs& sa) {
  hipStream_t st = s.stream;
  const size_t nt = size_t(std::max<int64_t>(s.nTot, 1)), ns = size_t(std::max<int64_t>(s.nSlots, 1));
  s.compAcc.ensure(sizeof(double) * D * nt);
  s.compDe0.ensure(sizeof(double) * nt);
  s.compRec.ensure(sizeof(double) * 8 * ns);
  s.compDe.ensure(sizeof(double) * ns);
  hipLaunchKernelGGL(k_compat_scatter<D>, dim3(nblocks(s.nInt)), dim3(kBlock), 0, st, s.work.as<int32_t>(),
                     s.perm.as<int32_t>(), s.nInt, s.out.as<double>(), s.outStride,
                     derivOffsetDoubles(D, SPHGPU_D_DVDT), derivOffsetDoubles(D, SPHGPU_D_DEPSDT),
                     s.compAcc.as<double>(), s.compDe0.as<double>());
  applyGhostVector(s, s.compAcc);
  applyGhostScalar(s, s.compDe0);
  hipLaunchKernelGGL(k_compat_rec<D>, dim3(nblocks(s.nSlots)), dim3(kBlock), 0, st, s.perm.as<int32_t>(), s.nSlots,
                     vel0, s.compAcc.as<double>(), s.compDe0.as<double>(), s.mass.as<double>(), sa,
                     s.compRec.as<double>());
  withLanes<D, D == 1>(rowLanes(RowPass::kCompat, D, s.nInt), [&](auto lanes) {
    constexpr int L = decltype(lanes)::value;
    hipLaunchKernelGGL((k_compat<D, L>), dim3(xcdGrid(nblocks(s.nInt * L))), dim3(kBlock), 0, st, s.work.as<int32_t>(),
                       s.rowCount.as<int32_t>(), s.nbr.as<int32_t>(), s.nSlots, s.nInt, s.compRec.as<double>(),
                       s.pairDv.as<double>(), s.nSlots * int64_t(s.ellCap), s.compDe.as<double>());
  });
  SG_CHECK_HIP(hipGetLastError());
}

// rec >= 0: the update also writes the internal slots' records (pack sec bits;
// isotropic H only) and the caller packs the ghost slots' records after the
// ghost rows are refreshed.
template <int D, bool TRIAL> void updateD(Sim& s, const Base& b, const Bounds& bd, const Eos& e,
                                          const double* compDe, const SegArgs& sa, int rec = -1) {
  Fields f{s.pos.as<double>(), s.vel.as<double>(), s.eps.as<double>(), s.rho.as<double>(), s.H.as<double>(),
           s.P.as<double>(), s.cs.as<double>()};
  DerivIn d{s.out.as<double>(), s.outStride, derivOffsetDoubles(D, SPHGPU_D_DXDT), derivOffsetDoubles(D, SPHGPU_D_DVDT),
            derivOffsetDoubles(D, SPHGPU_D_DEPSDT), derivOffsetDoubles(D, SPHGPU_D_DRHODT),
            derivOffsetDoubles(D, SPHGPU_D_HIDEAL), derivOffsetDoubles(D, SPHGPU_D_MAX_VISCOUS_PRESSURE),
            derivOffsetDoubles(D, SPHGPU_D_DVDX), compDe};
  if (!TRIAL) {
    s.dtIn.ensure(sizeof(double) * size_t(2 + D) * size_t(std::max<int64_t>(s.nInt, 1)));
    s.haveDtIn = true;
  }
  SG_REQUIRE(rec < 0 || s.isotropic, SPHGPU_ERR_STATE, "records from the update need H = h I");
  const PackIn pin = rec >= 0 ? packInputs(s) : PackIn{};
  const PackOut pout = rec >= 0 ? packOutputs(s, rec) : PackOut{};
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(D == 2 ? xcdGrid(nblocks(s.nInt)) : nblocks(s.nInt)), dim3(kBlock), 0, s.stream,
                       s.iperm.as<int32_t>(), s.nInt, f, b, d, bd, e, sa, pin, pout, s.dtIn.as<double>());
  };
  // the trial update writes the pair kernel's records, the final one the density sum's
  if constexpr (TRIAL) {
    switch (rec) {
      case -1: go(k_update<D, -1, true>); break;
      case 0: go(k_update<D, 0, true>); break;
      case 1: go(k_update<D, 1, true>); break;
      case 2: go(k_update<D, 2, true>); break;
      default: SG_REQUIRE(false, SPHGPU_ERR_STATE, "unsupported record kinds for the trial update");
    }
  } else {
    switch (rec) {
      case -1: go(k_update<D, -1, false>); break;
      case 4: go(k_update<D, 4, false>); break;
      case 8: go(k_update<D, 8, false>); break;
      default: SG_REQUIRE(false, SPHGPU_ERR_STATE, "unsupported record kinds for the final update");
    }
  }
  SG_CHECK_HIP(hipGetLastError());
  s.recValid = false;
}

template <int D> double hydroDtD(Sim& s, double nPerh, double cfl, int useVelMag) {
  s.reduceTmp.ensure(sizeof(double) * 16);
  unsigned long long* bits = reinterpret_cast<unsigned long long*>(s.reduceTmp.as<double>() + 9);
  const double init = double(FLT_MAX);
  unsigned long long ib;
  std::memcpy(&ib, &init, sizeof(ib));
  hipLaunchKernelGGL(k_set_u64, dim3(1), dim3(1), 0, s.stream, bits, ib);
  if (!s.haveDtIn) s.dtIn.ensure(sizeof(double) * 8);
  voteD<D, kVoteRows>(s, nPerh, useVelMag, nullptr, bits, 0);
  unsigned long long hb = 0;
  SG_CHECK_HIP(hipMemcpyAsync(&hb, bits, sizeof(hb), hipMemcpyDeviceToHost, s.stream));
  SG_CHECK_HIP(hipStreamSynchronize(s.stream));
  double minDt;
  std::memcpy(&minDt, &hb, sizeof(minDt));
  return cfl * minDt;
}

// Every member's vote and failure flags before a step.
__global__ void k_seg_vote_init(SegState* __restrict__ st, int n, unsigned long long v) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    st[i].voteBits = v;
    st[i].fail = 0u;
  }
}
// The end of a step: the clock, and the states to pinned host memory (one
// launch in place of a selection, an advance and a copy).  dtThreshold > 0: a
// member whose vote falls below it (a collapsing step) is flagged; its step
// has run and it is evicted afterwards.
__global__ void k_seg_advance(SegState* __restrict__ st, int n, SelectArgs sel, double dtThreshold,
                              SegState* __restrict__ host) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  SegState g = st[i];
  const double vote = sel.cfl * __longlong_as_double((long long)g.voteBits);
  if (dtThreshold > 0.0 && !(vote >= dtThreshold)) g.fail |= unsigned(SPHGPU_MEMBER_DT_COLLAPSE);
  g.dt = selectDt(g, sel);
  g.t = g.t + g.dt;
  g.lastDt = g.dt;
  g.cycle = g.cycle + 1.0;
  st[i] = g;
  host[i] = g;
}

// Integrator::preStepInitialize: ghosts and connectivity.  The build's record
// pack also writes the pair kernel's record, which the step reads first (grad-h
// recomputes omega, which the records hold, before that).
void preStep(Sim& s, const sphgpu_hydro_params& hp, const sphgpu_integrator_params& ip) {
  const bool mixed = hp.precision == SPHGPU_PRECISION_MIXED;
  const bool fast64 = s.rowOrder == SPHGPU_ROW_ORDER_SEARCH && hp.epsTensile == 0.0 && !hp.compatibleEnergyEvolution;
  struct Hint {     // the hint holds for this build only, also when it throws
    Sim& s;
    ~Hint() {
      s.buildRecHint = -1;
      s.buildVel = false;
    }
  } hint{s};
  s.buildVel = mixed;
  s.buildRecHint = ip.gradhCorrection ? 0 : (mixed ? 1 : (fast64 ? 2 : 0));
  if (!s.subs.empty()) setGhostNodes(s, ip.kernelExtent, ip.cullGhostNodes != 0);
  else buildNeighbors(s, ip.kernelExtent);
}

// Where the dt votes go: one word, or one per ensemble member.
struct Vote {
  const double* seg;
  unsigned long long* bits;
  int64_t stride;
};

// The dt vote, the two derivative passes and updates of SynchronousRK2::step, then
// SPHHydroBase::finalize and Integrator::enforceBoundaries.  Multipliers are
// dt/2, dt (plain simulation) or per member (half, full).
template <int D> void stepBody(Sim& s, const sphgpu_hydro_params& hp, const sphgpu_integrator_params& ip,
                               const Vote& vote, const SegArgs& half, const SegArgs& full) {
  hipStream_t st = s.stream;
  const bool compat = hp.compatibleEnergyEvolution != 0;
  SG_REQUIRE(!compat || s.deviceGhosts || s.nTot == s.nInt, SPHGPU_ERR_UNSUPPORTED,
             "compatible energy with caller-supplied ghost rows: the ghost derivatives need the device boundaries");
  const Bounds bd{ip.rhoMin, ip.rhoMax, 1.0 / hp.hmax, 1.0 / hp.hmin};
  const Eos e = makeEos(ip.gamma, ip.Pmin, ip.Pmax, ip.pressureFloor);

  // derivatives at t (SPHHydroBase::initialize first: the grad-h correction); the
  // midpoint pass below rewrites every field before anything but the trial
  // update reads one, so this pass stores only the fields the update reads
  // (the vote needs nothing the pass writes but the rows' largest relative speeds,
  // and the pass nothing of the vote)
  const bool mixed = hp.precision == SPHGPU_PRECISION_MIXED;
  auto cast = [&](auto from) {
    voteD<D, decltype(from)::value>(s, hp.nPerh, ip.useVelocityMagnitudeForDt, vote.seg, vote.bits, vote.stride);
  };
  // In 2-D a row has 28 neighbours and the gather is no slower than the two launches
  // (250 k nodes: 20 and 18 + 5 us).  In 3-D the pair pass keeps maxima with one lane to
  // a node, from 49153 nodes; the bounds gain there already, a little (a whole step with
  // the gather and with them: 51 k nodes 660 and 649 us, 104 k 839 and 817, 141 k 1053
  // and 1027, 262 k 1612 and 1584), and are taken from 131073, where they were first measured.
  const bool bounds = mixed && D == 3 && s.nInt > 131072;
  if (mixed && !bounds) cast(std::integral_constant<int, kVoteSlots>{});
  if (ip.gradhCorrection) omegaGradh(s);
  evalDerivs(s, hp, true, !mixed || bounds);
  if (!mixed) cast(std::integral_constant<int, kVoteDone>{});
  else if constexpr (D == 3) {
    if (bounds) cast(std::integral_constant<int, kVoteBounds>{});
  }
  // state0 (the policy reads every row's step-start velocity, ghosts included)
  const size_t n = size_t(s.nInt), nv = compat ? size_t(s.nTot) : n;
  const size_t rows[4] = {n * D, nv * D, n, n};
  for (int q = 0; q < 4; ++q) s.state0[q].ensure(std::max<size_t>(sizeof(double) * rows[q], 8));
  const Base b0{s.state0[0].as<double>(), s.state0[1].as<double>(), s.state0[2].as<double>(), s.state0[3].as<double>()};
  if (nv > n)
    SG_CHECK_HIP(hipMemcpyAsync(b0.vel + n * D, s.vel.as<double>() + n * D, sizeof(double) * (nv - n) * D,
                                hipMemcpyDeviceToDevice, st));
  // omega has no update policy (SPHHydroBase::registerState enrolls it bare):
  // state.assign(state0) gives the final update the step-start value again
  const size_t omegaBytes = sizeof(double) * size_t(s.nTot);
  if (ip.gradhCorrection && omegaBytes) {
    s.omega0.ensure(omegaBytes);
    SG_CHECK_HIP(hipMemcpyAsync(s.omega0.p, s.omega.p, omegaBytes, hipMemcpyDeviceToDevice, st));
  }
  // The updates write the records the next pass reads (isotropic H; grad-h
  // recomputes omega, which the records hold, before the midpoint pass).
  const bool recs = s.isotropic && !ip.gradhCorrection;
  const int recMid = recs ? pairRecordSec(s, hp) : -1;
  const int recEnd = recs ? densityRecordSec(s) : -1;
  auto ghostsAndRecords = [&](int rec) {
    if (rec >= 0) applyGhostBoundariesAndRecords(s, rec);
    else applyGhostBoundaries(s);
  };
  // trial advance to the midpoint
  if (compat) compatD<D>(s, s.vel.as<double>(), half);
  updateD<D, true>(s, b0, bd, e, compat ? s.compDe.as<double>() : nullptr, half, recMid);
  ghostsAndRecords(recMid);
  // derivatives at t + dt/2 with the step's neighbour rows
  if (ip.gradhCorrection) omegaGradh(s);
  evalDerivs(s, hp);
  if (ip.gradhCorrection && omegaBytes)
    SG_CHECK_HIP(hipMemcpyAsync(s.omega.p, s.omega0.p, omegaBytes, hipMemcpyDeviceToDevice, st));
  // advance from state0 with the midpoint derivatives
  if (compat) compatD<D>(s, b0.vel, full);
  updateD<D, false>(s, b0, bd, e, compat ? s.compDe.as<double>() : nullptr, full, recEnd);
  ghostsAndRecords(recEnd);
  // SPHHydroBase::finalize: sum density
  sumDensity(s);
  // Integrator::enforceBoundaries
  enforceBoundaries(s);
}

// The clock of a plain simulation as one SegState, so that the kernels of the step
// select its dt (selectDt) and the step needs no host round trip before its end.
__global__ void k_plain_seg_init(SegState* __restrict__ g, double t, double lastDt, double tEnd, double gamma,
                                 unsigned long long vote) {
  g->t = t;
  g->lastDt = lastDt;
  g->tEnd = tEnd;
  g->gamma = gamma;
  g->dt = 0.0;
  g->voteBits = vote;
  g->cycle = 0.0;
  g->fail = 0u;
  g->failPad = 0u;
}

// ---- the device part of a step as a HIP graph ---------------------------------
// Everything between the neighbour build and the clock read-back (dt vote,
// dt selection, both passes, updates, ghost refreshes, finalize, boundary
// enforcement, clock advance) is launched without a host round trip.  Its
// launches depend on the node and slot counts, the device buffers, the
// parameters and the host-side record flags at its start: that is the key
// (stepkey.cpp).
// The first step with a new key runs eagerly (sizing every buffer), the next
// step with the same key is captured and instantiated, and later steps with
// that key replay the graph; the host flags the step leaves are saved at the
// capture and restored after each replay.  An ensemble whose membership and
// ghost counts hold still (most steps of a tube ensemble) replays one graph
// per step.  Graphs hold no memset node and no stage-timing events.
Sim::StepFlags stepFlagsOf(const Sim& s) {
  return Sim::StepFlags{s.recValid, s.recSValid, s.recSMValid, s.derivsValid, s.pairsValid, s.haveDtIn,
                        s.pairRec, s.outStride, s.timingPending, s.pairWaves};
}
void restoreStepFlags(Sim& s, const Sim::StepFlags& f) {
  s.recValid = f.recValid;
  s.recSValid = f.recSValid;
  s.recSMValid = f.recSMValid;
  s.derivsValid = f.derivsValid;
  s.pairsValid = f.pairsValid;
  s.haveDtIn = f.haveDtIn;
  s.pairRec = f.pairRec;
  s.outStride = f.outStride;
  s.timingPending = f.timingPending;
  s.pairWaves = f.pairWaves;
}

// A few graphs and recent keys are kept: culling swaps the ghosts' controls and planes
// and the caller -> slot map with their spares, so a step's buffers alternate between
// two sets.
constexpr size_t kStepGraphs = 4;

template <class F> void runStep(Sim& s, const sphgpu_hydro_params& hp, const sphgpu_integrator_params& ip, F&& launches) {
  if (!s.useGraphs) {
    launches();
    return;
  }
  std::vector<uint64_t> key = stepKey(s, hp, ip);
  for (Sim::StepGraph& g : s.stepGraphs)
    if (g.key == key) {
      SG_CHECK_HIP(hipGraphLaunch(g.exec, s.stream));
      restoreStepFlags(s, g.flags);
      ++s.graphReplays;
      return;
    }
  if (std::find(s.recentKeys.begin(), s.recentKeys.end(), key) == s.recentKeys.end()) {
    // a new key: run eagerly, which also sizes every buffer the step uses
    launches();
    s.recentKeys.push_back(std::move(key));
    if (s.recentKeys.size() > kStepGraphs) s.recentKeys.erase(s.recentKeys.begin());
    return;
  }
  SG_CHECK_HIP(hipStreamBeginCapture(s.stream, hipStreamCaptureModeThreadLocal));
  s.capturing = true;
  try {
    launches();
  } catch (...) {
    s.capturing = false;
    hipGraph_t g = nullptr;
    (void)hipStreamEndCapture(s.stream, &g);
    if (g) (void)hipGraphDestroy(g);
    throw;
  }
  s.capturing = false;
  hipGraph_t g = nullptr;
  SG_CHECK_HIP(hipStreamEndCapture(s.stream, &g));
  hipGraphExec_t exec = nullptr;
  const hipError_t e = hipGraphInstantiate(&exec, g, nullptr, nullptr, 0);
  (void)hipGraphDestroy(g);
  SG_CHECK_HIP(e);
  if (s.stepGraphs.size() >= kStepGraphs) {
    SG_CHECK_HIP(hipGraphExecDestroy(s.stepGraphs.front().exec));
    s.stepGraphs.erase(s.stepGraphs.begin());
  }
  Sim::StepGraph sg;
  sg.key = std::move(key);
  sg.exec = exec;
  sg.flags = stepFlagsOf(s);
  s.stepGraphs.push_back(std::move(sg));
  SG_CHECK_HIP(hipGraphLaunch(exec, s.stream));
  ++s.graphCaptures;
}

template <int D> double rk2D(Sim& s, const sphgpu_hydro_params& hp, const sphgpu_integrator_params& ip,
                             double maxTime) {
  hipStream_t st = s.stream;
  preStep(s, hp, ip);
  // GenericHydro::dt, then selectDt (dtMin/dtMax clamped to maxTime - t, dtGrowth)
  s.plainSeg.ensure(sizeof(SegState));
  SegState* sd = s.plainSeg.as<SegState>();
  const double init = double(FLT_MAX);
  unsigned long long ib;
  std::memcpy(&ib, &init, sizeof(ib));
  hipLaunchKernelGGL(k_plain_seg_init, dim3(1), dim3(1), 0, st, sd, s.time, s.lastDt, maxTime, ip.gamma, ib);
  if (!s.haveDtIn) s.dtIn.ensure(sizeof(double) * 8);
  const SelectArgs sel{ip.cfl, ip.dtMin, ip.dtMax, ip.dtGrowth};
  SegState* hs = static_cast<SegState*>(hostStaging(s, 0, sizeof(SegState)));
  runStep(s, hp, ip, [&] {
    const Vote vote{nullptr, &sd->voteBits, 0};
    const bool perList = s.nLists > 1 && !s.listGammaHost.empty();
    const double* lo = perList ? s.seg.as<double>() : nullptr;
    const double* lg = perList ? s.listGamma.as<double>() : nullptr;
    const SegArgs half{nullptr, sd, 1, sel, lo, lg}, full{nullptr, sd, 0, sel, lo, lg};
    stepBody<D>(s, hp, ip, vote, half, full);
    hipLaunchKernelGGL(k_seg_advance, dim3(1), dim3(kBlock), 0, st, sd, 1, sel, 0.0, hs);
    SG_CHECK_HIP(hipGetLastError());
  });
  SG_CHECK_HIP(hipStreamSynchronize(st));
  const SegState h = *hs;
  s.time = h.t;
  s.lastDt = h.lastDt;
  s.cycle += 1;
  s.derivsValid = false;
  return h.dt;
}

// One SynchronousRK2 step of every ensemble member, each with its own dt.
template <int D> void ensembleRk2D(Sim& s, const sphgpu_hydro_params& hp, const sphgpu_integrator_params& ip) {
  hipStream_t st = s.stream;
  const int ns = s.nSeg;
  SegState* sd = s.segState.as<SegState>();
  preStep(s, hp, ip);
  // GenericHydro::dt per member, then selectDt per member
  const double init = double(FLT_MAX);
  unsigned long long ib;
  std::memcpy(&ib, &init, sizeof(ib));
  if (!s.haveDtIn) s.dtIn.ensure(sizeof(double) * 8);
  const SelectArgs sel{ip.cfl, ip.dtMin, ip.dtMax, ip.dtGrowth};
  SegState* hs = static_cast<SegState*>(hostStaging(s, 0, sizeof(SegState) * size_t(ns)));
  runStep(s, hp, ip, [&] {
    hipLaunchKernelGGL(k_seg_vote_init, dim3(nblocks(ns)), dim3(kBlock), 0, st, sd, ns, ib);
    const Vote vote{s.seg.as<double>(), &sd->voteBits, int64_t(sizeof(SegState) / sizeof(unsigned long long))};
    SG_CHECK_HIP(hipGetLastError());
    const SegArgs half{s.seg.as<double>(), sd, 1, sel}, full{s.seg.as<double>(), sd, 0, sel};
    stepBody<D>(s, hp, ip, vote, half, full);
    hipLaunchKernelGGL(k_seg_advance, dim3(nblocks(ns)), dim3(kBlock), 0, st, sd, ns, sel, s.dtThreshold, hs);
    SG_CHECK_HIP(hipGetLastError());
  });
  SG_CHECK_HIP(hipStreamSynchronize(st));
  s.segHost.assign(hs, hs + ns);
  s.derivsValid = false;
}

__global__ void k_eos_rows(const double* __restrict__ rho, const double* __restrict__ eps, double* __restrict__ P,
                           double* __restrict__ cs, int64_t first, int64_t rows, Eos e) {
  const int64_t r = blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
  if (r >= rows) return;
  const int64_t i = first + r;
  P[i] = eosP(e, rho[i], eps[i]);
  cs[i] = eosCs(e, eps[i]);
}

}  // namespace

void eosGammaLaw(Sim& s, double gamma, double Pmin, double Pmax, int floorType) {
  if (s.nInt == 0) return;
  if (s.nLists > 1 && !s.listGammaHost.empty()) {
    // each NodeList with its own gamma-law gas
    for (int L = 0; L < s.nLists; ++L) {
      const int64_t first = s.listStart[size_t(L)], rows = s.listStart[size_t(L) + 1] - first;
      if (rows > 0) eosRows(s, first, rows, s.listGammaHost[size_t(L)], Pmin, Pmax, floorType);
    }
    SG_CHECK_HIP(hipStreamSynchronize(s.stream));
    s.recValid = false;
    s.derivsValid = false;
    return;
  }
  hipLaunchKernelGGL(k_eos, dim3(nblocks(s.nInt)), dim3(kBlock), 0, s.stream, s.rho.as<double>(), s.eps.as<double>(),
                     s.P.as<double>(), s.cs.as<double>(), s.nInt, makeEos(gamma, Pmin, Pmax, floorType));
  SG_CHECK_HIP(hipGetLastError());
  SG_CHECK_HIP(hipStreamSynchronize(s.stream));
  s.recValid = false;
  s.derivsValid = false;
}

double hydroDt(Sim& s, double nPerh, double cfl, int useVelMag) {
  SG_REQUIRE(s.neighborsValid, SPHGPU_ERR_STATE, "the dt vote needs a neighbour build");
  SG_REQUIRE(nPerh > 0.0, SPHGPU_ERR_ARG, "nPerh must be positive");
  if (s.dim == 1) return hydroDtD<1>(s, nPerh, cfl, useVelMag);
  if (s.dim == 2) return hydroDtD<2>(s, nPerh, cfl, useVelMag);
  return hydroDtD<3>(s, nPerh, cfl, useVelMag);
}

void ensembleRk2(Sim& s, const sphgpu_hydro_params& hp, const sphgpu_integrator_params& ip) {
  if (s.dim == 1) ensembleRk2D<1>(s, hp, ip);
  else if (s.dim == 2) ensembleRk2D<2>(s, hp, ip);
  else ensembleRk2D<3>(s, hp, ip);
}

// ---- SpheralConservation totals ---------------------------------------------
// Per block, in a fixed order, over rows [r0, r1): mass, linear momentum (3),
// angular momentum about the origin (3), 2 x kinetic energy, thermal energy.
constexpr int kCons = 9;
template <int D>
__global__ void k_conserve_partial(const double* __restrict__ pos, const double* __restrict__ vel,
                                   const double* __restrict__ mass, const double* __restrict__ eps, int64_t r0,
                                   int64_t r1, double* __restrict__ partial) {
  __shared__ double sh[kCons][kBlock];
  double a[kCons] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  for (int64_t i = r0 + blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < r1; i += int64_t(gridDim.x) * blockDim.x) {
    const double m = mass[i];
    double x[3] = {0, 0, 0}, v[3] = {0, 0, 0};
    for (int c = 0; c < D; ++c) { x[c] = pos[i * D + c]; v[c] = vel[i * D + c]; }
    a[0] += m;
    for (int c = 0; c < D; ++c) a[1 + c] += m * v[c];
    if (D == 2) a[6] += m * (x[0] * v[1] - x[1] * v[0]);
    if (D == 3) {
      a[4] += m * (x[1] * v[2] - x[2] * v[1]);
      a[5] += m * (x[2] * v[0] - x[0] * v[2]);
      a[6] += m * (x[0] * v[1] - x[1] * v[0]);
    }
    double v2 = v[0] * v[0];
    for (int c = 1; c < D; ++c) v2 = v2 + v[c] * v[c];
    a[7] += m * v2;
    a[8] += m * eps[i];
  }
  for (int q = 0; q < kCons; ++q) sh[q][threadIdx.x] = a[q];
  __syncthreads();
  for (int st = kBlock / 2; st > 0; st >>= 1) {
    if (threadIdx.x < st)
      for (int q = 0; q < kCons; ++q) sh[q][threadIdx.x] += sh[q][threadIdx.x + st];
    __syncthreads();
  }
  if (threadIdx.x < kCons) partial[blockIdx.x * kCons + threadIdx.x] = sh[threadIdx.x][0];
}
__global__ void k_conserve_final(const double* __restrict__ partial, int nb, double* __restrict__ out) {
  const int q = threadIdx.x;
  if (q >= kCons) return;
  double t = 0.0;
  for (int b = 0; b < nb; ++b) t += partial[b * kCons + q];
  out[q] = t;
}

// The totals as reported: the kinetic energy is half the summed m v^2.
__global__ void k_conserve_report(const double* __restrict__ partial, int nb, double* __restrict__ out) {
  const int q = threadIdx.x;
  if (q >= kCons) return;
  double t = 0.0;
  for (int b = 0; b < nb; ++b) t += partial[b * kCons + q];
  out[q] = q == 7 ? 0.5 * t : t;
}

// Workgroups of the partial sums (the same for every row count, so the
// summation order depends only on the rows).
constexpr int kConserveBlocks = 256;
inline int conserveBlocks(int64_t rows) {
  return int(std::min<int64_t>(kConserveBlocks, std::max<int64_t>(1, (rows + kBlock - 1) / kBlock)));
}
void conservePartials(Sim& s, int64_t r0, int64_t r1, int nb, double* partial) {
  if (s.dim == 1)
    hipLaunchKernelGGL(k_conserve_partial<1>, dim3(nb), dim3(kBlock), 0, s.stream, s.pos.as<double>(),
                       s.vel.as<double>(), s.mass.as<double>(), s.eps.as<double>(), r0, r1, partial);
  else if (s.dim == 2)
    hipLaunchKernelGGL(k_conserve_partial<2>, dim3(nb), dim3(kBlock), 0, s.stream, s.pos.as<double>(),
                       s.vel.as<double>(), s.mass.as<double>(), s.eps.as<double>(), r0, r1, partial);
  else
    hipLaunchKernelGGL(k_conserve_partial<3>, dim3(nb), dim3(kBlock), 0, s.stream, s.pos.as<double>(),
                       s.vel.as<double>(), s.mass.as<double>(), s.eps.as<double>(), r0, r1, partial);
}

// Totals of rows [r0, r1) (internal nodes of the sim, or of one ensemble
// member): [mass, p (3), L (3), kinetic, thermal], as SpheralConservation
// (src/SimulationControl/SpheralConservation.py:66-150) takes them.
void conservationTotals(Sim& s, int64_t r0, int64_t r1, double* out) {
  const int nb = conserveBlocks(r1 - r0);
  DBuf tmp;
  tmp.ensure(sizeof(double) * size_t(nb + 1) * kCons);
  double* partial = tmp.as<double>();
  double* res = partial + size_t(nb) * kCons;
  conservePartials(s, r0, r1, nb, partial);
  hipLaunchKernelGGL(k_conserve_final, dim3(1), dim3(64), 0, s.stream, partial, nb, res);
  SG_CHECK_HIP(hipGetLastError());
  double h[kCons];
  SG_CHECK_HIP(hipMemcpyAsync(h, res, sizeof(h), hipMemcpyDeviceToHost, s.stream));
  SG_CHECK_HIP(hipStreamSynchronize(s.stream));
  for (int q = 0; q < kCons; ++q) out[q] = h[q];
  out[7] = 0.5 * h[7];
}

// ---- the allocation-free totals ---------------------------------------------
// Partial sums of sphgpu_conservation_noalloc live in a file-scope device
// array instead of a per-call allocation: kConserveBlocks x kCons doubles
// (18 KB), held by every GPU the library runs on until the process ends.
// Each device has its own copy at its own address, resolved once per device
// with hipGetSymbolAddress (host code never passes the array's name itself).
// The partial kernel writes every slot it is read back from, so nothing needs
// clearing; calls that overlap on one GPU share the array and race.
constexpr size_t kScratchDoubles = size_t(kConserveBlocks) * kCons;
static __device__ __align__(256) double scratch[kScratchDoubles];
namespace {
constexpr int kMaxDevices = 64;
void* gScratch[kMaxDevices] = {};   // the array's address on each device
std::mutex gScratchMu;
}  // namespace

void resolveScratch(int device) {
  SG_REQUIRE(device >= 0 && device < kMaxDevices, SPHGPU_ERR_ARG, "device index beyond the scratch table");
  std::lock_guard<std::mutex> lock(gScratchMu);
  if (gScratch[device]) return;
  void* p = nullptr;
  SG_CHECK_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));   // the device is current
  gScratch[device] = p;
}

void conservationTotalsNoAlloc(Sim& s, int64_t r0, int64_t r1, double* outDevice) {
  void* p = nullptr;
  {
    std::lock_guard<std::mutex> lock(gScratchMu);
    p = (s.device >= 0 && s.device < kMaxDevices) ? gScratch[s.device] : nullptr;
  }
  SG_REQUIRE(p, SPHGPU_ERR_STATE, "the device's scratch array was not resolved");
  const int nb = conserveBlocks(r1 - r0);
  SG_REQUIRE(size_t(nb) * kCons <= kScratchDoubles, SPHGPU_ERR_CAPACITY,
             "conservation partial sums exceed the scratch array");
  double* partial = static_cast<double*>(p);
  conservePartials(s, r0, r1, nb, partial);
  hipLaunchKernelGGL(k_conserve_report, dim3(1), dim3(64), 0, s.stream, partial, nb, outDevice);
  SG_CHECK_HIP(hipGetLastError());
}

// iterateIdealH (src/Utilities/iterateIdealH.cc:30-310), SPH smoothing scale,
// nPerhForIteration = 0, no spherical start, no fixed determinant.  Each
// iteration makes the ghosts of the sim's boundaries (or only the
// connectivity without boundaries) from the current H and passes over the
// internal nodes; the loop ends after maxIterations or once the largest
// change is within tol.  The ghosts are remade from the final H at the end.
int iterateIdealH(Sim& s, const sphgpu_hydro_params& hp, int maxIterations, double tol, double ext, bool cull,
                  double* maxDelta) {
  SG_REQUIRE(s.nInt > 0, SPHGPU_ERR_STATE, "no nodes");
  SG_REQUIRE(!s.ensemble, SPHGPU_ERR_STATE, "ensembles iterate H per member alone");
  SG_REQUIRE(s.nTot == s.nInt || s.deviceGhosts, SPHGPU_ERR_STATE,
             "iterateIdealH makes its own ghosts: set_nodes(n_internal, n_internal)");
  SG_REQUIRE(maxIterations >= 0 && tol >= 0.0 && ext > 0.0, SPHGPU_ERR_ARG, "bad iteration parameters");
  DBuf deltaH, bits;
  deltaH.ensure(sizeof(double) * size_t(s.nInt));
  bits.ensure(sizeof(unsigned long long));
  const double init = 2.0 * tol;
  hipLaunchKernelGGL(k_fill_value, dim3(nblocks(s.nInt)), dim3(kBlock), 0, s.stream, deltaH.as<double>(), s.nInt, init);
  double m = 2.0 * tol;
  int it = 0;
  // several NodeLists: the pass walks each node's full connectivity, in
  // ConnectivityMap order (reference row order)
  struct MapOrder {
    Sim& s;
    explicit MapOrder(Sim& x) : s(x) { s.rowsMapOrder = s.nLists > 1; }
    ~MapOrder() { s.rowsMapOrder = false; }
  };
  {
    MapOrder mo(s);
    while (it < maxIterations && m > tol) {
      ++it;
      if (!s.subs.empty()) setGhostNodes(s, ext, cull);
      else buildNeighbors(s, ext);
      hipLaunchKernelGGL(k_set_u64, dim3(1), dim3(1), 0, s.stream, bits.as<unsigned long long>(), 0ull);
      m = idealHPass(s, hp, tol, deltaH.as<double>(), bits.as<unsigned long long>());
    }
  }
  // leave the ghosts made from the final H (rows in the pass's order)
  if (!s.subs.empty()) setGhostNodes(s, ext, cull);
  else s.neighborsValid = false;
  SG_CHECK_HIP(hipStreamSynchronize(s.stream));
  if (maxDelta) *maxDelta = m;
  return it;
}

void eosRows(Sim& s, int64_t first, int64_t rows, double gamma, double Pmin, double Pmax, int floorType) {
  if (rows <= 0) return;
  hipLaunchKernelGGL(k_eos_rows, dim3(nblocks(rows)), dim3(kBlock), 0, s.stream, s.rho.as<double>(),
                     s.eps.as<double>(), s.P.as<double>(), s.cs.as<double>(), first, rows,
                     makeEos(gamma, Pmin, Pmax, floorType));
  SG_CHECK_HIP(hipGetLastError());
}

double rk2Step(Sim& s, const sphgpu_hydro_params& hp, const sphgpu_integrator_params& ip, double maxTime) {
  SG_REQUIRE(!s.ensemble, SPHGPU_ERR_STATE, "an ensemble steps with sphgpu_ensemble_step");
  SG_REQUIRE(s.nInt > 0, SPHGPU_ERR_STATE, "no nodes");
  SG_REQUIRE(s.table.n > 0, SPHGPU_ERR_STATE, "no kernel table installed");
  SG_REQUIRE(ip.kernelExtent > 0.0 && ip.cfl > 0.0 && ip.dtGrowth > 0.0, SPHGPU_ERR_ARG, "bad integrator parameters");
  SG_REQUIRE(s.nTot == s.nInt || s.deviceGhosts, SPHGPU_ERR_STATE,
             "the integrator makes its own ghosts: set_nodes(n_internal, n_internal)");
  if (s.dim == 1) return rk2D<1>(s, hp, ip, maxTime);
  if (s.dim == 2) return rk2D<2>(s, hp, ip, maxTime);
  return rk2D<3>(s, hp, ip, maxTime);
}

}  // namespace sphgpu
