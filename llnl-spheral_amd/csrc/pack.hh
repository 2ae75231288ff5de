// Record packing shared by the record pack (hydro.hip) and the integrator
// update (integrate.hip), so that both write bitwise the same records.
#pragma once
#include <cstdint>
#include <hip/hip_runtime.h>
#include "dgeom.hh"
#include "records.hh"

namespace sphgpu {

// ---------------------------------------------------------------------------
// Records
// ---------------------------------------------------------------------------
// The neighbour records of the isotropic pair and density kernels, each made
// from an FP64 record r (isotropic layout).  The kernels' time is set by the
// number of 16-B loads per neighbour gather, so each record holds only what
// its kernel reads.
// The mixed pair kernel's record (FP32), float4s per slot by dimension: 1-D
// (x, +-1/h, m | 1/rho, v, c, P/rho^2/omega), 2-D (x, y | +-1/h, m, 1/rho, vx |
// vy, c, P/rho^2/omega, m/rho) with x, y as FP64 bits, 3-D (qx, qy, qz, +-1/h |
// m, 1/rho, vx, vy | vz, c, P/rho^2/omega, m/rho).  1/h is negative for ghost
// rows; det H = (1/h)^D and in 1-D m/rho = m * (1/rho) are formed by the reader.
// In 3-D the position is the low 32 bits of round(x / u) for a power of two u
// with the largest search radius below 2^30 u: the 32-bit difference of two
// neighbours' words is the exact difference of their rounded positions, so
// r_ij carries an error of at most u (1e-9 of the search radius), far below
// the FP32 rounding of r_ij itself.
__device__ __forceinline__ uint32_t quantPos(double x, double qInv) {
  return uint32_t(uint64_t(static_cast<long long>(rint(x * qInv))));
}
template <int D> struct MixedRec {
  static constexpr int F4 = D == 1 ? 2 : 3;
};
__device__ __forceinline__ float dlo(double x) { return __int_as_float(__double2loint(x)); }
__device__ __forceinline__ float dhi(double x) { return __int_as_float(__double2hiint(x)); }
template <int D>
__device__ __forceinline__ void writeMixedRec(const double* r, int64_t nInt, double qInv, float4* __restrict__ p) {
  using R = RL<true>;
  const bool ghost = r[R::ORIG] >= double(nInt);
  const float hinv = ghost ? -float(r[R::HINV]) : float(r[R::HINV]);
  const double rho = r[R::RHO];
  const float invRho = rho != 0.0 ? float(1.0 / rho) : 0.0f;
  const float m = float(r[R::M]), cs = float(r[R::CS]), prho = float(r[R::PRHO]), mor = float(r[R::MOR]);
  if constexpr (D == 1) {
    p[0] = make_float4(dlo(r[R::X]), dhi(r[R::X]), hinv, m);
    p[1] = make_float4(invRho, float(r[R::V]), cs, prho);
  } else if constexpr (D == 2) {
    p[0] = make_float4(dlo(r[R::X]), dhi(r[R::X]), dlo(r[R::X + 1]), dhi(r[R::X + 1]));
    p[1] = make_float4(hinv, m, invRho, float(r[R::V]));
    p[2] = make_float4(float(r[R::V + 1]), cs, prho, mor);
  } else {
    p[0] = make_float4(__uint_as_float(quantPos(r[R::X], qInv)), __uint_as_float(quantPos(r[R::X + 1], qInv)),
                       __uint_as_float(quantPos(r[R::X + 2], qInv)), hinv);
    p[1] = make_float4(m, invRho, float(r[R::V]), float(r[R::V + 1]));
    p[2] = make_float4(float(r[R::V + 2]), cs, prho, mor);
  }
}
// The FP64 isotropic pair kernel's record, 96 B per slot: x y z, 1/h (negative for
// ghosts), m, 1/rho, c, P/rho^2/omega, v, 0.  det H and m/rho are recomputed by
// the loader.  230 MB at 2.4 M slots fit the 256 MB Infinity Cache,
// and one plane beats two: the gather brings in 1.5 lines a record instead of 2
// (loads of all records of the rows at 128^3, in one run: 2.15 ms, as 64 + 32 B
// 2.38 ms, one to a 128-B line 2.55 ms).
template <int D>
__device__ __forceinline__ void writeFast64Rec(const double* r, int64_t nInt, double2* __restrict__ p) {
  using R = RL<true>;
  const bool ghost = r[R::ORIG] >= double(nInt);
  const double rho = r[R::RHO];
  p[0] = make_double2(r[R::X], D > 1 ? r[R::X + 1] : 0.0);
  p[1] = make_double2(D > 2 ? r[R::X + 2] : 0.0, ghost ? -r[R::HINV] : r[R::HINV]);
  p[2] = make_double2(r[R::M], rho != 0.0 ? 1.0 / rho : 0.0);
  p[3] = make_double2(r[R::CS], r[R::PRHO]);
  p[4] = make_double2(r[R::V], D > 1 ? r[R::V + 1] : 0.0);
  p[5] = make_double2(D > 2 ? r[R::V + 2] : 0.0, 0.0);
}

// The density sum's neighbour record (DensRec).
template <int D>
__device__ __forceinline__ void writeDensRec(const double* r, double2* __restrict__ p) {
  using R = RL<true>;
  p[0] = make_double2(r[R::X], D > 1 ? r[R::X + 1] : 0.0);
  p[1] = make_double2(D > 2 ? r[R::X + 2] : 0.0, r[R::HINV]);
  p[2] = make_double2(r[R::M], r[R::ORIG]);
}

// The mixed density sum's neighbour record: x (FP64 bits), 1/h and m (FP32),
// one float4 in 1-D, two otherwise; det H = (1/h)^D is formed by the reader.
template <int D> struct DensMixedRec {
  static constexpr int F4 = D == 1 ? 1 : 2;
};
template <int D>
__device__ __forceinline__ void writeDensRecMixed(const double* r, float4* __restrict__ p) {
  using R = RL<true>;
  if constexpr (D == 1) {
    p[0] = make_float4(dlo(r[R::X]), dhi(r[R::X]), float(r[R::HINV]), float(r[R::M]));
  } else {
    const double x1 = r[R::X + 1], x2 = D > 2 ? r[R::X + 2] : 0.0;
    p[0] = make_float4(dlo(r[R::X]), dhi(r[R::X]), dlo(x1), dhi(x1));
    p[1] = make_float4(dlo(x2), dhi(x2), float(r[R::HINV]), float(r[R::M]));
  }
}

// The caller-order fields a record is made from.
struct PackIn {
  const int32_t* perm;     // slot -> caller row (-1: dead slot)
  const double *pos, *vel, *mass, *rho, *P, *cs, *H, *omega;
  const double *fCl, *fCq, *fsh;   // Q multipliers (anisotropic records), or null
};
// Where the records go: rec (FP64 record), sec (SEC bit 1: mixed, bit 2: FP64
// isotropic pair record), sec2 (SEC bit 4: FP64 density record), sec3 (SEC
// bit 8: mixed density record); n slots.
struct PackOut {
  double* rec;
  void* sec;
  void* sec2;
  int64_t n, nInt;
  void* sec3;
  double qInv;     // 1/u of the 3-D mixed record's positions
  double* vel;     // velocities by slot for the dt vote (velStride doubles each), or null
};
// One or two 16-B loads a neighbour in 2-D and 3-D.
constexpr int velStride(int D) { return D == 3 ? 4 : D; }

// A row's fields, as the records take them.
template <int D> struct PackRow {
  V<D> x, v;
  S<D> h;
  double rho, m, P, cs, omega, fcl, fcq, fsh;
};
template <int D, bool ISO>
__device__ __forceinline__ PackRow<D> loadPackRow(int64_t i, const PackIn& in) {
  PackRow<D> w;
  for (int c = 0; c < D; ++c) { w.x.c[c] = in.pos[i * D + c]; w.v.c[c] = in.vel[i * D + c]; }
  for (int c = 0; c < NSym<D>::value; ++c) w.h.c[c] = in.H[i * NSym<D>::value + c];
  w.rho = in.rho[i]; w.m = in.mass[i]; w.P = in.P[i]; w.cs = in.cs[i]; w.omega = in.omega[i];
  w.fcl = w.fcq = w.fsh = 1.0;
  if constexpr (!ISO) {
    if (in.fCl) { w.fcl = in.fCl[i]; w.fcq = in.fCq[i]; w.fsh = in.fsh[i]; }
  }
  return w;
}

template <int D, bool ISO, int SEC>
__device__ __forceinline__ void storeRecords(int64_t k, const double* r, const PackOut& o) {
  static_assert(SEC == 0 || ISO, "the pair kernels' records are isotropic");
  using R = RL<ISO>;
  double2* dst = reinterpret_cast<double2*>(o.rec + k * R::STRIDE);
#pragma unroll
  for (int c = 0; c < R::STRIDE / 2; ++c) dst[c] = make_double2(r[2 * c], r[2 * c + 1]);
  if constexpr ((SEC & 1) != 0) writeMixedRec<D>(r, o.nInt, o.qInv, static_cast<float4*>(o.sec) + k * MixedRec<D>::F4);
  if constexpr ((SEC & 2) != 0)
    writeFast64Rec<D>(r, o.nInt, static_cast<double2*>(o.sec) + k * 6);
  if constexpr ((SEC & 4) != 0) writeDensRec<D>(r, static_cast<double2*>(o.sec2) + k * 3);
  if constexpr ((SEC & 8) != 0) writeDensRecMixed<D>(r, static_cast<float4*>(o.sec3) + k * DensMixedRec<D>::F4);
}

// The records of slot k, which holds caller row i with the fields `w` (from
// memory, or still in the registers of the kernel that wrote them: reading a
// row back right after storing it waits for the stores).  SEC (bits): besides
// the FP64 record also the mixed pair kernel's record (1), the FP64 isotropic
// pair kernel's (2), the FP64 density sum's (4) and the mixed density sum's (8).
template <int D, bool ISO, int SEC>
__device__ __forceinline__ void packRow(int64_t k, int64_t i, const PackRow<D>& w, const PackOut& o) {
  using R = RL<ISO>;
  double r[R::STRIDE];
#pragma unroll
  for (int c = 0; c < R::STRIDE; ++c) r[c] = 0.0;
  for (int c = 0; c < D; ++c) { r[R::X + c] = w.x.c[c]; r[R::V + c] = w.v.c[c]; }
  const double som = safeInv(w.omega, 1.0e-30);
  if constexpr (ISO) {
    r[RL<true>::HINV] = w.h.c[0];
  } else {
    for (int c = 0; c < NSym<D>::value; ++c) r[RL<false>::H + c] = w.h.c[c];
    r[RL<false>::FCL] = w.fcl;
    r[RL<false>::FCQ] = w.fcq;
    r[RL<false>::FSH] = w.fsh;
  }
  r[R::HDET] = sdet(w.h);
  r[R::M] = w.m;
  r[R::ORIG] = double(i);
  r[R::RHO] = w.rho;
  r[R::CS] = w.cs;
  r[R::P] = w.P;
  r[R::SOM] = som;
  r[R::PRHO] = som * w.P / (w.rho * w.rho);
  r[R::MOR] = w.m / w.rho;
  storeRecords<D, ISO, SEC>(k, r, o);
  if (o.vel) {
    double* p = o.vel + k * velStride(D);
    if constexpr (D == 1) {
      p[0] = w.v.c[0];
    } else {
      reinterpret_cast<double2*>(p)[0] = make_double2(w.v.c[0], w.v.c[1]);
      if constexpr (D == 3) reinterpret_cast<double2*>(p)[1] = make_double2(w.v.c[2], 0.0);
    }
  }
}

// The same from the fields in memory; a dead slot (culled ghost, in no row)
// gets an empty record.
template <int D, bool ISO, int SEC>
__device__ __forceinline__ void packSlot(int64_t k, const PackIn& in, const PackOut& o) {
  using R = RL<ISO>;
  const int64_t i = in.perm[k];
  if (i < 0) {
    double r[R::STRIDE];
#pragma unroll
    for (int c = 0; c < R::STRIDE; ++c) r[c] = 0.0;
    r[R::ORIG] = 2147483648.0;
    storeRecords<D, ISO, SEC>(k, r, o);
    return;
  }
  packRow<D, ISO, SEC>(k, i, loadPackRow<D, ISO>(i, in), o);
}

struct Sim;
PackIn packInputs(Sim& s);
// allocates the records that sec asks for; sets recSValid and recSMValid from bits 4 and 8
PackOut packOutputs(Sim& s, int sec);

}  // namespace sphgpu
