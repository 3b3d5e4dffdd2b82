// Threshold records of fp32 and fp16 rows: what sdx_thr.hip's kernels share.
#pragma once

#include "sdx_draw16.hpp"

namespace sdx {

// What decides the final probability of any element of a row: p / totf where
// p = exp_det(x / T - m) / zf is above vf, or equals it with id <= idcut; 0 elsewhere.
// No logit below xcut is kept. Kept in the row's RowStat (kmax, klo and ntbl hold vf,
// idcut and xcut; rstar < gcount marks a partially kept boundary tie group).
struct ThrRow {
  float m, zf, totf, vf, xcut;
  uint32_t idcut;
};
__device__ __forceinline__ ThrRow thr_load_row(const RowStat& st) {
  ThrRow r;
  r.m = st.m;
  r.zf = st.zf;
  r.totf = st.totf;
  r.vf = __uint_as_float((uint32_t)st.kmax);
  r.idcut = (uint32_t)st.klo;
  r.xcut = __uint_as_float((uint32_t)st.ntbl);
  return r;
}
__device__ __forceinline__ float thr_prob(const ThrRow& r, float x, uint32_t id, float T) {
  if (!(x >= r.xcut)) return 0.0f;
  const float p = exp_det(x / T - r.m) / r.zf;
  return p > r.vf || (p == r.vf && id <= r.idcut) ? p / r.totf : 0.0f;
}

// The row's scratch: this, a list of kThrList entries, then kThrBuckets masses (u64) and
// counts (u32).
struct ThrCtl {
  uint32_t tick;       // parts whose sums are in (cleared by the first kernel)
  uint32_t nlist;      // region elements found
  int32_t use_k, use_p;  // filters that the region has to decide
  float m, zf, phi, plo, xcut;
  uint64_t pmass[kThrMaxParts];  // per part: mass and count of the elements above the region
  uint32_t pcnt[kThrMaxParts];
  float pmax[kThrMaxParts], pmin[kThrMaxParts];
  uint32_t pnf[kThrMaxParts];  // fp16: the part holds a +inf or +NaN
  uint64_t z[3];  // the normaliser's 32-bit limbs
};
static_assert(sizeof(ThrCtl) % 8 == 0 && sizeof(ThrCtl) <= kThrCtlBytes, "ThrCtl layout");

}  // namespace sdx
