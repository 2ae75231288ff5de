// What a captured step's launches hold of the host's state: the key under which its
// graph is kept (integrate.hip replays a graph only under an equal key).  A value
// that reaches a launch as an argument and that anything outside the graph can
// change belongs in it: counts, buffers, parameters, record flags.
#include "internal.hh"
#include <algorithm>
#include <cmath>
#include <cstring>

namespace sphgpu {

double quantInv(const Sim& s) {
  // only the 3-D mixed record holds quantised positions; with no finite search
  // radius there is no pair to difference and any unit serves
  if (s.dim != 3 || !(s.rMax > 0.0) || !std::isfinite(s.rMax)) return 1.0;
  const int e = std::ilogb(s.rMax) + 1 - 30;     // rMax < 2^30 u
  SG_REQUIRE(e > -120 && e < 120, SPHGPU_ERR_UNSUPPORTED,
             "mixed precision: the search radius is outside the FP32 exponent range");
  const double q = std::ldexp(1.0, -e);
  // round(x / u) must fit a 64-bit integer; 2^61 leaves room for the motion
  // of one step beyond the positions the neighbour build saw
  SG_REQUIRE(s.posAbsMax * q < std::ldexp(1.0, 61), SPHGPU_ERR_UNSUPPORTED,
             "mixed precision: positions too far from the origin for the 3-D fixed-point record (|x| >= 2^61 u, "
             "u = largest search radius / 2^30)");
  return q;
}

static void keyBuf(std::vector<uint64_t>& k, const DBuf& b) {
  k.push_back(reinterpret_cast<uint64_t>(b.p));
  k.push_back(uint64_t(b.bytes));
}
template <class T> static void keyBytes(std::vector<uint64_t>& k, const T& v) {
  const unsigned char* c = reinterpret_cast<const unsigned char*>(&v);
  for (size_t i = 0; i < sizeof(T); i += 8) {
    uint64_t w = 0;
    std::memcpy(&w, c + i, std::min<size_t>(8, sizeof(T) - i));
    k.push_back(w);
  }
}
std::vector<uint64_t> stepKey(const Sim& s, const sphgpu_hydro_params& hp, const sphgpu_integrator_params& ip) {
  std::vector<uint64_t> k;
  k.reserve(256);
  for (int64_t v : {int64_t(s.dim), s.nInt, s.nTot, s.nSlots, int64_t(s.ellCap), int64_t(s.nSeg), s.tableVersion,
                    int64_t(s.isotropic), int64_t(s.rowOrder), int64_t(s.precision), int64_t(s.deviceGhosts),
                    int64_t(s.hasMultipliers), int64_t(s.recValid), int64_t(s.recSValid), int64_t(s.recSMValid),
                    int64_t(s.pairRec), int64_t(s.haveDtIn), int64_t(s.derivsValid), int64_t(s.subs.size()),
                    int64_t(s.nLists), int64_t(s.sumAllLists), int64_t(s.listGammaHost.size())})
    k.push_back(uint64_t(v));
  for (int64_t v : s.subStart) k.push_back(uint64_t(v));
  for (const SubBoundary& b : s.subs) keyBytes(k, b);
  keyBytes(k, hp);
  keyBytes(k, ip);
  keyBytes(k, s.dtThreshold);
  // the unit of the mixed records' positions follows the last build's largest search
  // radius, and the captured launches hold it as an argument
  if (hp.precision == SPHGPU_PRECISION_MIXED) keyBytes(k, quantInv(s));
  k.push_back(reinterpret_cast<uint64_t>(s.pinnedOut));
  for (const DBuf* b : {&s.pos, &s.vel, &s.mass, &s.rho, &s.eps, &s.P, &s.cs, &s.H, &s.omega, &s.fCl, &s.fCq,
                        &s.fshear, &s.cellOf, &s.cellCount, &s.cellStart, &s.cellRank, &s.cellMembers, &s.perm, &s.iperm, &s.xs,
                        &s.rowCount, &s.nbr, &s.scanTmp, &s.reduceTmp, &s.flags, &s.rec, &s.recM, &s.recD,
                        &s.recS, &s.recSM, &s.pairDv, &s.compDe, &s.compAcc, &s.compDe0, &s.compRec, &s.out,
                        &s.ghostControl, &s.ghostSub, &s.keep, &s.keepScan, &s.slotKeep, &s.hmaxOf, &s.genDev,
                        &s.work, &s.ghostIsControl, &s.omega0, &s.dtIn, &s.seg, &s.segState, &s.plainSeg,
                        &s.dTable, &s.dTable32, &s.dNperh, &s.dWsum, &s.listGamma, &s.subDev, &s.pairCounts, &s.velS, &s.relV,
                        &s.voteLow, &s.slotList})
    keyBuf(k, *b);
  for (const DBuf& b : s.state0) keyBuf(k, b);
  return k;
}

}  // namespace sphgpu
