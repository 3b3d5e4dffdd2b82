// to_probs statistics and outputs of rows whose values are too many to count one by
// one (fp32 and fp16 logits, specdec/sampling.py:34-67), several workgroups per row.
//
// The transform of a row reduces to one record: its final probability is
//   p(id) = exp_det(s - m) / zf,  s = fl32(x / T)
//   kept  = p > vf, or p == vf and id <= idcut      (p / totf where kept, else 0)
// because the reference keeps a prefix of the order (p descending, id ascending).
// The record takes three kernels over several workgroups per row (nlight of them where
// a pass only compares, nparts in the histogram pass) and one with a workgroup per row:
//   1. thr_max_kernel      the row's maximum (and minimum) logit per part;
//   2. thr_hist_kernel     the exact normaliser (96-bit fixed point per thread), and
//                          masses (and, for top-k, counts) of the elements in NB
//                          equal steps of m - s. The part that finishes last
//                          finds the region: the steps that can
//                          hold the boundary element, with a margin of 1e-6 of the
//                          mass on each side (what rounding to p, to fixed point and
//                          to fp32 cumulative sums can move is below 4e-7). As an
//                          interval of p [plo, phi] it holds whole tie groups;
//   3. thr_collect_kernel  count and exact mass of the elements above the region,
//                          and a list (p, id) of the region's;
//   4. thr_resolve_kernel  one workgroup per row sorts the list and walks it with the
//                          reference's test. A region with more than kThrList
//                          elements (a tie group, or a flat row) is refined over the
//                          row itself, a thousand bins of p at a time;
// then thr_output_kernel writes to_probs rows (of up to 32,768 ids and without a filter
// thr_plain_kernel alone), and thr_draw_kernel is the verify's
// accept chain and draw, which evaluates p where it needs it: a verify writes no
// probabilities.
//
// What bounds it: the instructions of the exp of pass 2, which every element needs
// (about 50 per element: the reference division by T as two FMA steps from 1 / T,
// the float64 reduction, nine multiply-adds, and the fixed-point value formed from
// the mantissa and the exponent by one shift); the other passes compare a logit
// with a threshold and evaluate only the few elements above it, compacted to full
// waves. Splitting a row over workgroups keeps the chip full from a few rows on.
// Measured on fp32 rows of 151,936 (one workgroup of 1024 threads per row before, with
// seven IEEE divisions per element and dense probabilities for the draw): verify of 8
// batch rows at k = 4 (72 rows, top-k 50) 283 -> 60 us (kernels 10 + 26 + 11 + 6 and
// the draw 11), to_probs of 256 rows 370 -> 197 us (53 + 56 + 32 + 7 + 54: the exp pass
// issues 54 vector instructions an element, on full SIMDs; the last moves 6.3 TB/s). On
// fp16 rows (one workgroup of 1024 threads and a histogram of 36,864 values per row
// before): verify of 16 batch rows at k = 4, V = 131,072 142 -> 77 us (10 + 30 + 16 + 8
// and the draw 17), of 64 at V = 32,000 165 -> 74 us; to_probs of 64 x 131,072 132 -> 54 us.
// The compare passes keep the evaluation in one place of their code (a loop over a
// queue in LDS): unrolled into every element's place, 16 to 64 copies, the collect
// pass of the fp16 verify took 20 us instead of 17 and its draw 22 instead of 20. The
// queues stay small enough for eight workgroups per CU (twice the queue: 20 us).
#include "sdx_thr.hpp"

#include <cmath>
#include <type_traits>

namespace sdx {

constexpr int TH_NT = 256;
constexpr int TH_NW = TH_NT / kWave;
constexpr int TH_NB = kThrBuckets;
constexpr int TH_BPT = TH_NB / TH_NT;  // buckets per thread

// ---- loads: 16 bytes per lane and step, the elements before the row's first 16-byte
// boundary with part 0, those after the last whole vector with the last part
template <class E>
struct ThrVec {
  static constexpr int N = 16 / (int)sizeof(E);
};
__device__ __forceinline__ float thr_f(float x) { return x; }
__device__ __forceinline__ float thr_f(uint16_t c) { return decode16<SDX_F16>(c); }

// Streams part `part` of the row through f(id, x, valid), every element exactly once:
// every lane of a wave makes every call (valid: the lane has an element), so f may
// vote. UN vectors per thread are in flight; after them, g() runs once (code that
// would otherwise stand once per element: in copies, its first passes wait for the
// instruction cache). With SKIP, whole vectors of a wave below `low` are left out.
template <class E, int UN, bool SKIP = false, class F, class G>
__device__ __forceinline__ void thr_stream(const E* __restrict__ row, int64_t V, int part,
                                           int nparts, int64_t plen, F&& f, G&& g,
                                           float low = 0.0f) {
  constexpr int N = ThrVec<E>::N;
  const int tid = threadIdx.x;
  int64_t head = (int64_t)(((16u - ((uint32_t)(uintptr_t)row & 15u)) & 15u) / sizeof(E));
  if (head > V) head = V;
  const int64_t nv = (V - head) / N;  // whole vectors of the row
  const int64_t v0 = (int64_t)part * (plen / N);
  const int64_t v1 = part == nparts - 1 ? nv : min(nv, v0 + plen / N);
  // the ends, by wave 0: fewer than eight elements each (lanes 0 .. and 32 ..)
  if (tid < kWave && (part == 0 || part == nparts - 1)) {
    const int64_t i = tid < 32 ? tid : head + nv * N + (tid - 32);
    const bool ok = tid < 32 ? part == 0 && i < head : part == nparts - 1 && i < V;
    f(i, ok ? thr_f(row[i]) : 0.0f, ok);
  }
  const uint4* __restrict__ x4 = reinterpret_cast<const uint4*>(row + head);
  // uniform; at least once, for the ends
  for (int64_t b = v0; b == v0 || b < v1; b += (int64_t)UN * TH_NT) {
    uint4 w[UN];
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      const int64_t j = b + (int64_t)u * TH_NT + tid;
      w[u] = j < v1 ? x4[j] : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      if (b + (int64_t)u * TH_NT + (tid & ~(kWave - 1)) >= v1) break;  // uniform per wave
      const int64_t j = b + (int64_t)u * TH_NT + tid;
      const bool ok = j < v1;
      const int64_t i = head + j * N;
      const uint32_t q[4] = {w[u].x, w[u].y, w[u].z, w[u].w};
      float x[N];
#pragma unroll
      for (int e = 0; e < N; ++e) {
        if constexpr (sizeof(E) == 4) x[e] = __uint_as_float(q[e]);
        else x[e] = thr_f((uint16_t)(q[e >> 1] >> (16 * (e & 1))));
      }
      if constexpr (SKIP) {
        float mx = x[0];
#pragma unroll
        for (int e = 1; e < N; ++e) mx = fmaxf(mx, x[e]);
        if (__ballot(ok && mx >= low) == 0) continue;  // uniform
      }
#pragma unroll
      for (int e = 0; e < N; ++e) f(i + e, x[e], ok);
    }
    g();
  }
}
template <class E, int UN, class F>
__device__ __forceinline__ void thr_stream(const E* __restrict__ row, int64_t V, int part,
                                           int nparts, int64_t plen, F&& f) {
  thr_stream<E, UN>(row, V, part, nparts, plen, f, [] {});
}

template <class E>
__device__ __forceinline__ const E* thr_row(const ThrArgs& a, int64_t row) {
  const int g = row < a.nrows[0] ? 0 : 1;
  const int64_t r = g ? row - a.nrows[0] : row;
  return reinterpret_cast<const E*>(a.base[g]) + r * a.ld[g];
}
__device__ __forceinline__ int64_t thr_gid(const ThrArgs& a, int64_t row) {
  const int g = row < a.nrows[0] ? 0 : 1;
  return draft_id_of_row(a.ids, a.tgt_idx, a.k, a.nrows[1], g, g ? row - a.nrows[0] : row);
}
// the row's scratch: ThrCtl, the list, then the masses and the counts
__device__ __forceinline__ ThrCtl* thr_ctl(const ThrArgs& a, int64_t row) {
  const uintptr_t p = (uintptr_t)a.scratch + (uintptr_t)row * (uintptr_t)a.scratch_stride;
  return reinterpret_cast<ThrCtl*>((p + 63) & ~(uintptr_t)63);
}
__device__ __forceinline__ uint64_t* thr_list(ThrCtl* c) {
  return reinterpret_cast<uint64_t*>(c + 1);
}
__device__ __forceinline__ uint64_t* thr_mass(ThrCtl* c) { return thr_list(c) + kThrList; }
__device__ __forceinline__ uint32_t* thr_cnt(ThrCtl* c) {
  return reinterpret_cast<uint32_t*>(thr_mass(c) + TH_NB);
}

// ---------------------------------------------------------------- 1. maximum
// fp16 codes two at a time: as signed keys in value order (negative codes with their
// low 15 bits flipped), maximum and minimum with packed 16-bit operations; -inf (and
// NaNs of negative sign) wrap around above every finite key for the minimum.
__device__ __forceinline__ void thr_max16(const ThrArgs& a, const uint16_t* row, int part,
                                          float& mx, float& mn, bool& nf) {
  typedef short s2 __attribute__((ext_vector_type(2)));
  typedef unsigned short u2 __attribute__((ext_vector_type(2)));
  constexpr short kLow = -31744;  // key of the least finite value
  s2 hi = {-32768, -32768};
  u2 lo = {0xFFFF, 0xFFFF};
  const int tid = threadIdx.x;
  const int64_t nv = a.V / 8;  // rows start 16-byte aligned
  const int64_t v0 = (int64_t)part * (a.llen / 8);
  const int64_t v1 = part == a.nlight - 1 ? nv : min(nv, v0 + a.llen / 8);
  const uint4* const x4 = reinterpret_cast<const uint4*>(row);
  auto fold = [&](uint32_t q) {
    const s2 c = __builtin_bit_cast(s2, q);
    const s2 k = c ^ ((c >> 15) & (s2){0x7FFF, 0x7FFF});
    hi = __builtin_elementwise_max(hi, k);
    lo = __builtin_elementwise_min(lo, __builtin_bit_cast(u2, (s2)(k - (s2){kLow, kLow})));
  };
  // to_probs takes any V: the elements after the last whole vector
  if (part == a.nlight - 1 && nv * 8 + tid < a.V) fold(row[nv * 8 + tid] * 0x10001u);
  constexpr int UN = 4;
  for (int64_t b = v0 + tid; b < v1; b += (int64_t)UN * TH_NT) {
    uint4 w[UN];
#pragma unroll
    for (int u = 0; u < UN; ++u) w[u] = x4[min(b + (int64_t)u * TH_NT, v1 - 1)];  // again: harmless
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      const uint32_t q[4] = {w[u].x, w[u].y, w[u].z, w[u].w};
#pragma unroll
      for (int e = 0; e < 4; ++e) fold(q[e]);
    }
  }
  const int h = max((int)hi[0], (int)hi[1]);
  const int l = min((int)lo[0], (int)lo[1]);
  auto val = [](int k) { return thr_f((uint16_t)(k < 0 ? k ^ 0x7FFF : k)); };
  nf = h >= 0x7C00;
  mx = nf ? INFINITY : val(h);
  mn = l <= 0x7C00 - 1 - kLow ? val(l + kLow) : INFINITY;
}

template <class E>
__global__ void __launch_bounds__(TH_NT) thr_max_kernel(ThrArgs a) {
  __shared__ float sMx[TH_NW], sMn[TH_NW];
  const int64_t row = blockIdx.x / a.nlight;
  const int part = (int)(blockIdx.x % a.nlight);
  const int tid = threadIdx.x;
  ThrCtl* const c = thr_ctl(a, row);
  if (part == 0 && tid == 0) {
    c->tick = 0u; c->nlist = 0u;
    c->z[0] = c->z[1] = c->z[2] = 0ull;
    if (row < a.nzero) a.zero[row] = 0u;
  }
  if (a.nparts > 1)  // the row's histogram, a share per part
    for (int b = part * TH_NT + tid; b < TH_NB; b += a.nlight * TH_NT) {
      thr_mass(c)[b] = 0ull;
      thr_cnt(c)[b] = 0u;
    }
  float mx = -INFINITY, mn = INFINITY;
  bool nf = false;  // fp16: a +inf or a NaN of positive sign (fp32 rows report neither)
  if constexpr (sizeof(E) == 2) thr_max16(a, thr_row<E>(a, row), part, mx, mn, nf);
  else
    thr_stream<E, 8>(thr_row<E>(a, row), a.V, part, a.nlight, a.llen,
                     [&](int64_t, float x, bool ok) {
                       mx = ok ? fmaxf(mx, x) : mx;
                       mn = ok && x > -INFINITY ? fminf(mn, x) : mn;
                     });
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    mx = fmaxf(mx, __shfl_xor(mx, o, kWave));
    mn = fminf(mn, __shfl_xor(mn, o, kWave));
  }
  if ((tid & (kWave - 1)) == 0) { sMx[tid / kWave] = mx; sMn[tid / kWave] = mn; }
  const int any = __syncthreads_or(nf);
  if (tid == 0) {
    for (int w = 1; w < TH_NW; ++w) { mx = fmaxf(mx, sMx[w]); mn = fminf(mn, sMn[w]); }
    c->pmax[part] = mx;
    c->pmin[part] = mn;
    c->pnf[part] = any ? 1u : 0u;
  }
}

// ---------------------------------------------------------------- 2. normaliser, region
// fixed62(exp_det(d)) for d <= 0 (and 0 for NaN): exp_det's steps, then the value
// mant * 2^(k + 39) as a right shift of mant << 39 (k is in [-63, 0] after the clamp at
// -43.5, below which the value is 0). Equal to the two functions over every fp32 d:
// above the clamp p 2^k is normal, so exp_det does not round and fixed62 truncates the
// same 24 bits.
__device__ __forceinline__ uint64_t thr_exp62(float d) {
#pragma clang fp contract(off)
  const double dd = (double)fmaxf(d, -43.5f);
  const double kf = floor(dd * 0x1.71547652b82fep+0);
  const float r = fmaxf((float)(dd - kf * 0x1.62e42fefa39efp-1), 0.0f);
  float p = 0x1.71de3ap-19f;  // 1/9!
  p = p * r + 0x1.a01a02p-16f;
  p = p * r + 0x1.a01a02p-13f;
  p = p * r + 0x1.6c16c2p-10f;
  p = p * r + 0x1.111112p-7f;
  p = p * r + 0x1.555556p-5f;
  p = p * r + 0x1.555556p-3f;
  p = p * r + 0x1p-1f;
  p = p * r + 1.0f;
  p = p * r + 1.0f;
  p = fminf(p, 2.0f);
  const uint32_t mant = __float_as_uint(p) - 0x3F000000u;  // p in [1, 2]: 24-bit mantissa
  return ((uint64_t)(mant << 7) << 32) >> (uint32_t)(-(int)kf);
}

// How s = x / T is formed: T == 1; two Newton steps on x * (1 / T) with FMAs, which
// round correctly where no step under- or overflows (the first leaves the quotient
// within an ulp, the second is Markstein's); or the division itself.
enum ThrDiv { kDivOne, kDivFma, kDivIeee };
template <int DIV>
__device__ __forceinline__ float thr_div(float x, float T, float rT) {
  if constexpr (DIV == kDivOne) return x;
  if constexpr (DIV == kDivIeee) return x / T;
  const float q0 = x * rT;
  const float q1 = __builtin_fmaf(__builtin_fmaf(-T, q0, x), rT, q0);
  return __builtin_fmaf(__builtin_fmaf(-T, q1, x), rT, q1);
}

__device__ __forceinline__ ThrDiv thr_div_kind(float T, float xmax) {
  const float a = fabsf(xmax);
  if (T == 1.0f) return kDivOne;
  return T >= 0x1p-20f && T <= 0x1p20f && a <= 0x1p100f && (a >= 0x1p-90f || a == 0.0f) ? kDivFma
                                                                                       : kDivIeee;
}
// Steps of m - s per unit, 2^e: the row's range, as far as it can hold the boundary
// (a.dmax), over at most TH_NB steps; a quarter of them where a nucleus bounds the range
// and a small top-k the elements of a step: each step that is not empty is an atomic or
// two per part (fp32 verify of 16 rows, V = 32,000, top_p 0.9, top-k 50: histogram pass
// 20.5 us with up to all steps, 16.3 with a quarter).
__device__ __forceinline__ float thr_scale(const ThrArgs& a, float m, float xmn) {
  const float range = fminf(m - xmn / a.T, a.dmax);  // NaN (no finite logit): the most
  static_assert(104 * 8 <= TH_NB - 2 && 32 * 32 <= TH_NB, "the widest range fits the steps");
  const bool few = a.use_k && a.dmax <= 32.0f && a.top_k <= 1024;
  const float steps = few ? (float)(TH_NB / 4) : (float)(TH_NB - 2);
  const float q = fminf(steps / fmaxf(range, 0x1p-10f), 0x1p20f);
  const float least = a.dmax > 32.0f ? 8.0f : few ? 1.0f : 32.0f;
  return fmaxf(__uint_as_float(__float_as_uint(q) & 0x7F800000u), least);
}
// The first step that is left out of the histogram: the last one, or the first past
// a.dmax.
__device__ __forceinline__ uint32_t thr_steps(const ThrArgs& a, float scale) {
  return (uint32_t)fminf(a.dmax * scale + 1.0f, (float)(TH_NB - 1));
}
// Logits below this have no part in the histogram pass: m - s is past the steps and
// past 43.5, below which the fixed-point exp is 0.
__device__ __forceinline__ float thr_xskip(float m, float scale, uint32_t steps, float T) {
  const float d = fmaxf(43.5f, (float)steps / scale);
  float x = ((m - d) - (4e-6f * (fabsf(m) + d) + 2e-5f)) * T;  // as xcut below
  x -= 4e-6f * fabsf(x);
  return fabsf(x) < INFINITY ? x : -INFINITY;
}
// One element of the histogram pass: its mass where the filter is a nucleus, its count
// where it is a top-k (each an LDS atomic). What lies past `steps` is left out: a
// boundary that no step holds is there, and much of a row can be, most of it at low
// temperatures (64 lanes at one LDS address go one after the other: fp16 verify of 16
// rows, V = 131,072, T = 0.1, top-k 20 97 us with it, 74 without).
// `steps` is past every element (ALL) with both filters, where the range holds them and
// T does not press them together: the comparison costs such a pass 2%.
template <int DIV, bool MASS, bool CNT, bool ALL = false>
__device__ __forceinline__ void thr_hist_one(float x, bool ok, float T, float rT, float m,
                                             float scale, uint32_t steps, uint64_t* mass,
                                             uint32_t* cnt, uint64_t& zlo, uint32_t& zhi) {
  const float d = ok ? thr_div<DIV>(x, T, rT) - m : -INFINITY;
  // NaN (-inf logits through the FMA steps): the last step; d > 0 never, and
  // v_cvt_u32_f32 would take it to 0
  const uint32_t b = (uint32_t)fminf(-d * scale, (float)(TH_NB - 1));
  const uint64_t f = thr_exp62(d);
  zlo += f;
  zhi += zlo < f ? 1u : 0u;
  const bool in = ALL ? ok : b < steps;  // (not ok: never)
  if (CNT && in) atomicAdd(&cnt[b], 1u);
  // 2^-44 units: sums of 2^18 elements fit 64 bits
  const uint64_t fm = ALL || in ? f >> 18 : 0ull;  // (not ok: f is 0)
  if (MASS && fm) atomicAdd((unsigned long long*)&mass[b], (unsigned long long)fm);
}
// What a region of steps [b0, b1] (and the step bk of the k-th largest) decides.
struct ThrCut {
  float phi, plo, xcut;
  bool use_k, use_p;
};
__device__ __forceinline__ ThrCut thr_cut(const ThrArgs& a, float m, float zf, float scale, int b0,
                                          int b1, int bk) {
  ThrCut c;
  c.use_k = a.use_k;
  c.use_p = a.use_p;
  if (c.use_k && !c.use_p) {
    b0 = b1 = bk;
  } else if (c.use_k) {
    if (b1 < bk) c.use_k = false;  // the nucleus ends above the k-th largest
    else { b0 = min(b0, bk); b1 = bk; }
  }
  const float inv = 1.0f / scale;  // a power of two
  c.phi = -1.0f;                   // no filter: everything is above
  c.plo = 0x1p-149f;
  float dlo = -104.0f;
  if (c.use_k || c.use_p) {
    // edges of the steps: p at m - s = b0 / scale and (b1 + 1) / scale
    c.phi = b0 == 0 ? 2.0f : exp_det(-(float)b0 * inv) / zf;
    if (b1 < TH_NB - 1) {
      dlo = -(float)(b1 + 1) * inv;
      c.plo = exp_det(dlo) / zf;
      // a subnormal p can be the same over a whole unit of s: every positive p then
      if (!(c.plo >= 0x1p-126f)) {
        c.plo = 0x1p-149f;
        dlo = -104.0f;
      }
    }
  }
  // no logit below xcut has p >= plo: a normal p drops by more than its rounding within
  // 1e-5 of s, and the fp32 rounding of (m + dlo) T is within 1e-6 of its terms
  c.xcut = ((m + dlo) - (4e-6f * (fabsf(m) + fabsf(dlo)) + 2e-5f)) * a.T;
  c.xcut -= 4e-6f * fabsf(c.xcut);
  if (!(fabsf(c.xcut) < INFINITY)) c.xcut = -INFINITY;
  return c;
}
// The region's steps from running sums: this step's mass (and count) between rm and nm
// (rc and nc) of the row's, zu the row's normaliser in the masses' units. One writer
// each, as the running sums grow (the step before has not reached the bound).
__device__ __forceinline__ void thr_mark(const ThrArgs& a, int b, uint64_t rm, uint64_t nm,
                                         uint64_t rc, uint64_t nc, double zu, int32_t* b0,
                                         int32_t* b1, int32_t* bk) {
  const double tlo = ((double)a.top_p - 1e-6) * zu, thi = ((double)a.top_p + 1e-6) * zu;
  if ((double)nm >= tlo && !(b > 0 && (double)rm >= tlo)) *b0 = b;
  if ((double)nm >= thi && !(b > 0 && (double)rm >= thi)) *b1 = b;
  if (a.use_k && nc >= (uint64_t)a.top_k && rc < (uint64_t)a.top_k) *bk = b;
}

struct ThrHistLds {
  uint64_t mass[TH_NB];
  uint32_t cnt[TH_NB];
  uint64_t s64[TH_NW];
  uint64_t zl[TH_NW];
  uint32_t zh[TH_NW];
  int32_t last, b0, b1, bk;
};

// Exclusive scan over a workgroup of NW waves; `s` holds NW words.
template <int NW = TH_NW>
__device__ __forceinline__ uint64_t thr_excl_u64(uint64_t v, uint64_t* s) {
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
  const uint64_t incl = wave_incl_scan_u64(v, lane);
  __syncthreads();
  if (lane == kWave - 1) s[w] = incl;
  __syncthreads();
  uint64_t off = 0;
  for (int i = 0; i < NW; ++i) off += i < w ? s[i] : 0ull;
  return off + incl - v;
}

// f(DIV, MASS, CNT) as integral constants, for the row's division and the call's filters.
template <class F>
__device__ __forceinline__ void thr_hist_kind(const ThrArgs& a, ThrDiv div, F&& f) {
  auto kind = [&](auto mass, auto cnt) {
    if (div == kDivOne) f(std::integral_constant<int, kDivOne>{}, mass, cnt);
    else if (div == kDivFma) f(std::integral_constant<int, kDivFma>{}, mass, cnt);
    else f(std::integral_constant<int, kDivIeee>{}, mass, cnt);
  };
  if (a.use_p && a.use_k) kind(std::true_type{}, std::true_type{});
  else if (a.use_p) kind(std::true_type{}, std::false_type{});
  else if (a.use_k) kind(std::false_type{}, std::true_type{});
  else kind(std::false_type{}, std::false_type{});
}

// SKIP: whole vectors of logits that have no part in the pass are left out. They are
// most of a row at low temperatures, but the test ends the overlap of one vector's
// chains with the next's: fp16 verify of 16 rows, V = 131,072, top-k 20 at T = 0.1 74 ->
// 65 us with it; fp32 verify of 16 rows, V = 32,000 at T = 0.7 44 -> 49 us.
template <class E, bool SKIP>
__global__ void __launch_bounds__(TH_NT) thr_hist_kernel(ThrArgs a) {
  __shared__ ThrHistLds L;
  const int64_t row = blockIdx.x / a.nparts;
  const int part = (int)(blockIdx.x % a.nparts);
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wv = tid / kWave;
  ThrCtl* const c = thr_ctl(a, row);
  const E* const x = thr_row<E>(a, row);
  for (int b = tid; b < TH_NB; b += TH_NT) { L.mass[b] = 0ull; L.cnt[b] = 0u; }
  float xmx = lane < a.nlight ? c->pmax[lane] : -INFINITY;
  float xmn = lane < a.nlight ? c->pmin[lane] : INFINITY;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    xmx = fmaxf(xmx, __shfl_xor(xmx, o, kWave));
    xmn = fminf(xmn, __shfl_xor(xmn, o, kWave));
  }
  const float T = a.T;
  const float m = xmx / T;  // the division is monotone: the maximum of fl32(x / T)
  const float scale = thr_scale(a, m, xmn);
  const ThrDiv div = thr_div_kind(T, xmx);
  __syncthreads();
  uint64_t zlo = 0;
  uint32_t zhi = 0;
  const float rT = 1.0f / T;
  const uint32_t steps = thr_steps(a, scale);
  const float low = thr_xskip(m, scale, steps, T);
  thr_hist_kind(a, div, [&](auto DIV, auto MASS, auto CNT) {
    auto one = [&](int64_t, float xv, bool ok) {
      thr_hist_one<DIV.value, MASS.value, CNT.value, MASS.value && CNT.value && !SKIP>(
          xv, ok, T, rT, m, scale, steps, L.mass, L.cnt, zlo, zhi);
    };
    thr_stream<E, 4, SKIP>(x, a.V, part, a.nparts, a.plen, one, [] {}, low);
  });
  U128 z = wave_sum_u128(U128{zlo, (uint64_t)zhi});
  if (lane == 0) { L.zl[wv] = z.lo; L.zh[wv] = (uint32_t)z.hi; }
  __syncthreads();  // and the histogram is complete
  z = U128{0, 0};
  for (int w = 0; w < TH_NW; ++w) z = u128_add(z, U128{L.zl[w], L.zh[w]});
  if (a.nparts > 1) {
    // The row's sums by device-coherent atomics, step tid + 256 i per thread (a wave's
    // land in a few lines): nothing waits for them but the ticket. The part that
    // finishes last then reads one histogram; adding the parts' up there instead, four
    // in flight, took 8 to 10 us of dependent loads that miss the L2 at 15 parts.
    uint64_t* const gm = thr_mass(c);
    uint32_t* const gc = thr_cnt(c);
#pragma unroll
    for (int i = 0; i < TH_BPT; ++i) {
      const int b = tid + i * TH_NT;
      const uint64_t v = L.mass[b];
      if (v)
        __hip_atomic_fetch_add(gm + b, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (a.use_k && L.cnt[b])
        __hip_atomic_fetch_add(gc + b, L.cnt[b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (tid < 3)  // 32-bit limbs in 64-bit words
      __hip_atomic_fetch_add(&c->z[tid], tid == 2 ? z.hi : tid == 1 ? z.lo >> 32 : z.lo & 0xFFFFFFFFu,
                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0x0F70);  // gfx9 encoding: vmcnt(0)
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __syncthreads();
    if (tid == 0)
      L.last = __hip_atomic_fetch_add(&c->tick, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
               (uint32_t)(a.nparts - 1);
    __syncthreads();
    if (!L.last) return;  // uniform
    uint64_t tm[TH_BPT];
    uint32_t tc[TH_BPT];
#pragma unroll
    for (int i = 0; i < TH_BPT; ++i) {
      tm[i] = __hip_atomic_load(gm + tid + i * TH_NT, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      tc[i] = a.use_k ? __hip_atomic_load(gc + tid + i * TH_NT, __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_AGENT)
                      : 0u;
    }
    const uint64_t z0 = __hip_atomic_load(&c->z[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint64_t z1 = __hip_atomic_load(&c->z[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint64_t z2 = __hip_atomic_load(&c->z[2], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    z = u128_add(u128_add(U128{z0, 0}, U128{z1 << 32, z1 >> 32}), U128{0, z2});
#pragma unroll
    for (int i = 0; i < TH_BPT; ++i) {
      L.mass[tid + i * TH_NT] = tm[i];
      L.cnt[tid + i * TH_NT] = tc[i];
    }
    __syncthreads();
  }
  uint64_t mass[TH_BPT];
  uint32_t cnt[TH_BPT];
#pragma unroll
  for (int i = 0; i < TH_BPT; ++i) {
    mass[i] = L.mass[tid * TH_BPT + i];
    cnt[i] = L.cnt[tid * TH_BPT + i];
  }
  // ---- the region, step indexes [b0, b1] (0 at the maximum)
  const float zf = rn32_u128(z);
  if (tid == 0) { L.b0 = TH_NB - 1; L.b1 = TH_NB - 1; L.bk = TH_NB - 1; }
  uint64_t sm = 0, sc = 0;
#pragma unroll
  for (int i = 0; i < TH_BPT; ++i) { sm += mass[i]; sc += cnt[i]; }
  uint64_t rm = thr_excl_u64(sm, L.s64);
  uint64_t rc = a.use_k ? thr_excl_u64(sc, L.s64) : 0ull;
  __syncthreads();
  const double zu = ((double)z.hi * 0x1p64 + (double)z.lo) * 0x1p-18;
#pragma unroll
  for (int i = 0; i < TH_BPT; ++i) {
    const uint64_t nm = rm + mass[i], nc = rc + cnt[i];
    thr_mark(a, tid * TH_BPT + i, rm, nm, rc, nc, zu, &L.b0, &L.b1, &L.bk);
    rm = nm;
    rc = nc;
  }
  __syncthreads();
  if (tid != 0) return;
  const ThrCut t = thr_cut(a, m, zf, scale, L.b0, L.b1, L.bk);
  c->m = m;
  c->zf = zf;
  c->phi = t.phi;
  c->plo = t.plo;
  c->xcut = t.xcut;
  c->use_k = t.use_k ? 1 : 0;
  c->use_p = t.use_p ? 1 : 0;
}

// ---------------------------------------------------------------- 3. collect
// Per wave: ids that pass the threshold are compacted into LDS and evaluated 64 at a
// time by full waves, in one place of the code.
template <int N>
struct ThrQueue {
  uint2 e[kWave - 1 + N * kWave];  // bits of x, id
};
__device__ __forceinline__ void thr_lds_sync() {  // within one wave
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_wave_barrier();
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}
// Appends the lanes' (x, id) with `take`.
template <int N>
__device__ __forceinline__ void thr_push(ThrQueue<N>& q, uint32_t& n, float x, uint32_t id,
                                         bool take) {
  const uint64_t bm = __ballot(take);
  if (bm == 0) return;  // uniform
  if (take) {
    const uint32_t at = n + __builtin_amdgcn_mbcnt_hi((uint32_t)(bm >> 32),
                                                      __builtin_amdgcn_mbcnt_lo((uint32_t)bm, 0u));
    q.e[at] = make_uint2(__float_as_uint(x), id);
  }
  n += (uint32_t)__popcll(bm);
}
// g(x, id, ok) for the queue's last 64 entries while it holds at least 64, or any with
// `all`; fewer than 64 are left, so N more pushes fit.
template <int N, class G>
__device__ __forceinline__ void thr_drain(ThrQueue<N>& q, uint32_t& n, bool all, G&& g) {
  const uint32_t lane = threadIdx.x & (kWave - 1);
#pragma nounroll
  while (n >= (uint32_t)kWave || (all && n > 0)) {  // uniform
    thr_lds_sync();
    const uint32_t c = min(n, (uint32_t)kWave);
    n -= c;
    const bool ok = lane < c;
    const uint2 e = ok ? q.e[n + lane] : make_uint2(0xFF800000u, 0u);  // -inf
    thr_lds_sync();  // read before the next pushes
    g(__uint_as_float(e.x), e.y, ok);
  }
}

template <class E>
__global__ void __launch_bounds__(TH_NT) thr_collect_kernel(ThrArgs a) {
  constexpr int UN = 8 / ThrVec<E>::N;  // 8 elements a lane between two drains
  __shared__ ThrQueue<UN * ThrVec<E>::N + 1> sq[TH_NW];  // and the row's ends
  __shared__ uint32_t s_cnt[TH_NW];
  __shared__ uint64_t s_mass[TH_NW];
  const int64_t row = blockIdx.x / a.nlight;
  const int part = (int)(blockIdx.x % a.nlight);
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wv = tid / kWave;
  ThrCtl* const c = thr_ctl(a, row);
  const float m = c->m, zf = c->zf, phi = c->phi, plo = c->plo, xcut = c->xcut, T = a.T;
  uint64_t* const list = thr_list(c);
  uint64_t mass = 0;
  uint32_t cnt = 0;
  auto eval = [&](float x, uint32_t id, bool ok) {
    const float p = ok ? exp_det_sel(x / T - m) / zf : 0.0f;
    const bool above = ok && p > phi;
    mass += above ? fixed62(p) : 0ull;
    cnt += above ? 1u : 0u;
    const bool in = ok && !above && p >= plo;
    const uint64_t bm = __ballot(in);
    if (bm == 0) return;  // uniform
    uint32_t at = 0;
    if (lane == 0) at = atomicAdd(&c->nlist, (uint32_t)__popcll(bm));
    at = rdlane(at, 0) + __builtin_amdgcn_mbcnt_hi((uint32_t)(bm >> 32),
                                                   __builtin_amdgcn_mbcnt_lo((uint32_t)bm, 0u));
    if (in && at < (uint32_t)kThrList)
      list[at] = ((uint64_t)(~__float_as_uint(p)) << 32) | id;  // ascending: p down, id up
  };
  uint32_t n = 0;
  thr_stream<E, UN>(
      thr_row<E>(a, row), a.V, part, a.nlight, a.llen,
      [&](int64_t i, float x, bool ok) { thr_push(sq[wv], n, x, (uint32_t)i, ok && x >= xcut); },
      [&] { thr_drain(sq[wv], n, false, eval); });
  thr_drain(sq[wv], n, true, eval);
  mass = wave_sum_u64(mass);
  cnt = wave_sum_u32(cnt);
  if (lane == 0) { s_mass[wv] = mass; s_cnt[wv] = cnt; }
  __syncthreads();
  if (tid != 0) return;
  for (int w = 1; w < TH_NW; ++w) { mass += s_mass[w]; cnt += s_cnt[w]; }
  c->pmass[part] = mass;
  c->pcnt[part] = cnt;
}

// ---------------------------------------------------------------- 4. resolve
// kept = p > vf, or p == vf and id <= idcut; partial: the group of vf keeps a part of
// its members; tot: the kept mass.
struct ThrEnd {
  float vf = -1.0f;
  uint32_t idcut = 0xFFFFFFFFu;
  bool partial = false;
  uint64_t tot = 0;
};
struct ThrWalkLds {
  uint32_t first;
  uint64_t sum;
};
// The list's entries (e[0, n), any order, ~0 from there to NC or the next power of two)
// sorted ascending: up to NC of them by counting the smaller entries (into t), else in
// place. Returns where they are.
template <int NT, int NC>
__device__ __forceinline__ const uint64_t* thr_sort(uint64_t* e, uint64_t* t, uint32_t n) {
  const uint32_t tid = threadIdx.x;
  static_assert(NC == NT || NC == 2 * NT, "one or two entries per thread");
  if (n <= (uint32_t)NC) {  // uniform
    const uint64_t k0 = tid < n ? e[tid] : ~0ull;
    const uint64_t k1 = NC > NT && tid + NT < n ? e[tid + NT] : ~0ull;
    if (tid < n) {
      uint32_t r0 = 0, r1 = 0;
      for (uint32_t i = 0; i < n; i += 16) {  // ~0 past n: never smaller
        uint64_t v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) v[u] = e[i + u];
#pragma unroll
        for (int u = 0; u < 16; ++u) {
          r0 += v[u] < k0 ? 1u : 0u;
          if (NC > NT) r1 += v[u] < k1 ? 1u : 0u;
        }
      }
      t[r0] = k0;
      if (NC > NT && tid + NT < n) t[r1] = k1;
    }
    __syncthreads();
    return t;
  }
  uint32_t S = NT;
  while (S < n) S <<= 1;
  for (uint32_t size = 2; size <= S; size <<= 1)
    for (uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
      for (uint32_t i = tid; i < S; i += NT) {
        const uint32_t j = i ^ stride;
        if (j > i) {
          const bool up = (i & size) == 0;
          const uint64_t ai = e[i], aj = e[j];
          if ((ai > aj) == up) { e[i] = aj; e[j] = ai; }
        }
      }
      __syncthreads();
    }
  return e;
}
// The reference's walk over the sorted region: `above` and `nabove` are the mass and
// count of the elements above it, phi its upper edge.
template <int NT>
__device__ __forceinline__ ThrEnd thr_walk(const ThrArgs& a, const uint64_t* e, uint32_t n,
                                           bool use_k, bool use_p, uint64_t above, uint64_t nabove,
                                           float phi, ThrWalkLds& L, uint64_t* s64) {
  const uint32_t tid = threadIdx.x;
  ThrEnd r;
  auto pof = [&](uint32_t i) { return __uint_as_float(~(uint32_t)(e[i] >> 32)); };
  // the k-th largest p (0: not among the positive ones, nothing is zeroed)
  float kth = 0.0f;
  if (use_k && (uint64_t)a.top_k > nabove && (uint64_t)a.top_k - nabove <= n)
    kth = pof((uint32_t)((uint64_t)a.top_k - nabove) - 1u);
  if (tid == 0) { L.first = n; L.sum = 0ull; }
  // entries per * tid ..: their masses, then the first that fails
  const uint32_t per = (n + NT - 1) / NT;
  const uint32_t i0 = min(n, tid * per), i1 = min(n, i0 + per);
  uint64_t s = 0;
  for (uint32_t i = i0; i < i1; ++i) s += fixed62(pof(i));
  const uint64_t ex = above + thr_excl_u64<NT / kWave>(s, s64);
  uint64_t run = ex;
  uint32_t mine = n;
  for (uint32_t i = i0; i < i1; ++i) {
    const float p = pof(i);
    const uint64_t nr = run + fixed62(p);
    bool keep = !(p < kth);
    if (use_p) keep = keep && (((rn32_u64(nr) - p) < a.top_p) || (nabove + i == 0));
    if (!keep) { mine = i; break; }
    run = nr;
  }
  __syncthreads();
  // one LDS atomic per wave (a wave's lanes at one address go one after the other)
  const uint64_t fail = __ballot(mine < n);
  if (fail && (int)(tid & (kWave - 1)) == __ffsll((unsigned long long)fail) - 1)
    atomicMin(&L.first, mine);  // the wave's first: entries go up with the thread
  __syncthreads();
  const uint32_t f = L.first;  // entries [0, f) are kept
  const uint64_t part = wave_sum_u64(i0 < f ? run - ex : 0ull);
  if ((tid & (kWave - 1)) == 0 && part)
    atomicAdd((unsigned long long*)&L.sum, (unsigned long long)part);
  __syncthreads();
  r.tot = above + L.sum;
  if (f == 0) {
    r.vf = __uint_as_float(__float_as_uint(phi) + 1u);  // everything above the region
  } else {
    r.vf = pof(f - 1);
    r.partial = f < n && pof(f) == r.vf && !(r.vf < kth);
    if (r.partial) r.idcut = (uint32_t)e[f - 1];
  }
  return r;
}
// The row's record, with the final probability of its gathered token (one thread).
__device__ __forceinline__ RowStat thr_record(const ThrEnd& r, float m, float zf, float xcut,
                                              int64_t gid, int64_t V, float xg, float T,
                                              bool nonfinite) {
  const float totf = fmaxf(rn32_u64(r.tot), 1e-12f);
  const bool bad = !(zf > 0.0f);  // no finite maximum: every probability is 0 / 0
  const ThrRow row{m, zf, totf, r.vf, xcut, r.idcut};
  RowStat st = {};
  bool gtie = false;
  if (gid >= 0 && gid < V) {
    st.pgather = bad ? __builtin_nanf("") : thr_prob(row, xg, (uint32_t)gid, T);
    gtie = r.partial && exp_det(xg / T - m) / zf == r.vf;
  }
  st.m = m; st.zf = zf; st.totf = totf; st.mass = r.tot;
  st.kmax = (int32_t)__float_as_uint(r.vf);
  st.klo = (int32_t)r.idcut;
  st.glo = 1; st.ghi = 0;
  st.rstar = r.partial ? 1 : 0;
  st.gcount = r.partial ? 2 : 0;
  st.ntbl = (int32_t)__float_as_uint(xcut);
  st.argmax = -1;
  st.flags = (gtie ? (uint32_t)kRowGatherTie : 0u) | (bad ? (uint32_t)kRowNoMass : 0u) |
             (nonfinite ? (uint32_t)kRowNonfinite : 0u);
  return st;
}

// ---- refinement: a region with more elements than its list holds (a tie group, or many
// logits within a step) is split by p's bits, TH_NB bins a pass over the row, until the
// bin that holds the boundary fits the list or is one value.
struct ThrSpan {
  uint32_t lo, hi;     // bits of p: the boundary is in [lo, hi]
  uint64_t above;      // mass and count of the elements above hi
  uint64_t nabove;
  uint32_t n;          // elements in [lo, hi]
  bool use_k, use_p;   // filters that [lo, hi] has to decide
};
struct ThrPickLds {
  uint32_t fk, fp;
  uint64_t mass, count, total;
  uint32_t n;
};
__device__ __forceinline__ uint32_t thr_bin_shift(const ThrSpan& r) {
  uint32_t sh = 0;
  while (((r.hi - r.lo) >> sh) >= (uint32_t)TH_NB) ++sh;
  return sh;
}
// r narrowed to the bin (2^sh values of p each, bin 0 at r.hi; their masses, counts and
// least bits) that holds the boundary: the first in which the count from the top
// reaches top_k, or whose last element fails the nucleus test, whichever comes first.
// False: none does, everything in r is kept (r.above: with its mass).
template <int NT>
__device__ __forceinline__ bool thr_pick(const ThrArgs& a, const uint64_t* mass,
                                         const uint32_t* cnt, const uint32_t* low, uint32_t sh,
                                         ThrSpan& r, ThrPickLds& L, uint64_t* s64) {
  constexpr int BPT = TH_NB / NT;
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  if (tid == 0) L.fk = L.fp = ~0u;
  uint64_t sm = 0, sc = 0;
#pragma unroll
  for (int i = 0; i < BPT; ++i) { sm += mass[tid * BPT + i]; sc += cnt[tid * BPT + i]; }
  const uint64_t m0 = r.above + thr_excl_u64<NT / kWave>(sm, s64);
  const uint64_t c0 = r.nabove + thr_excl_u64<NT / kWave>(sc, s64);
  uint64_t rm = m0, rc = c0;
  uint32_t mk = ~0u, mp = ~0u;
#pragma unroll
  for (int i = 0; i < BPT; ++i) {
    const int b = tid * BPT + i;
    const uint32_t n = cnt[b];
    rm += mass[b];
    rc += n;
    if (n == 0) continue;
    if (mk == ~0u && rc >= (uint64_t)a.top_k) mk = (uint32_t)b;
    if (mp == ~0u && !((rn32_u64(rm) - __uint_as_float(low[b])) < a.top_p)) mp = (uint32_t)b;
  }
  if (tid == NT - 1) L.total = rm;
  const uint64_t vk = __ballot(mk != ~0u), vp = __ballot(mp != ~0u);  // bins go up with the lane
  if (vk && lane == __ffsll((unsigned long long)vk) - 1) atomicMin(&L.fk, mk);
  if (vp && lane == __ffsll((unsigned long long)vp) - 1) atomicMin(&L.fp, mp);
  __syncthreads();
  const uint32_t fk = r.use_k ? L.fk : ~0u, fp = r.use_p ? L.fp : ~0u, f = min(fk, fp);
  if (f == ~0u) {  // uniform
    r.above = L.total;
    __syncthreads();
    return false;
  }
  if ((uint32_t)tid == f / BPT) {
    rm = m0;
    rc = c0;
    for (uint32_t b = (uint32_t)tid * BPT; b < f; ++b) { rm += mass[b]; rc += cnt[b]; }
    L.mass = rm;
    L.count = rc;
    L.n = cnt[f];
  }
  __syncthreads();
  // the filter that ends in a later bin has no say
  r.use_k = fk == f;
  r.use_p = fp == f;
  r.above = L.mass;
  r.nabove = L.count;
  r.n = L.n;
  r.hi -= f << sh;
  r.lo = max(r.lo, r.hi - (1u << sh) + 1u);
  __syncthreads();
  return true;
}
// How many members of the tie group of p = v pass the nucleus test, of n below mass
// `above` and count `nabove` (a prefix; every wave the same search, 64 candidates a step).
__device__ __forceinline__ uint64_t thr_tie_kept(float v, uint64_t above, uint64_t nabove,
                                                 uint64_t n, float tp) {
  const int lane = threadIdx.x & (kWave - 1);
  const uint64_t P = fixed62(v);
  uint64_t lo = 0, hi = n;
  while (lo < hi) {
    const uint64_t step = (hi - lo + kWave - 1) / kWave;
    const uint64_t cand = lo + (uint64_t)lane * step;
    const bool keep = cand < hi && (((rn32_u64(above + (cand + 1) * P) - v) < tp) ||
                                    (nabove + cand == 0));  // the row's first is always kept
    const int nk = __popcll(__ballot(keep));
    if (nk == 0) break;
    const uint64_t last = lo + (uint64_t)(nk - 1) * step;
    lo = last + 1;
    hi = min(hi, last + step);
  }
  return lo;
}
// The end at a single value of p, of which `kept` members are.
__device__ __forceinline__ ThrEnd thr_tie_end(const ThrSpan& r, uint64_t kept) {
  ThrEnd e;
  e.vf = __uint_as_float(kept > 0 ? r.lo : r.lo + 1u);  // none: everything above
  e.tot = r.above + kept * fixed62(__uint_as_float(r.lo));
  e.partial = kept > 0 && kept < r.n;
  return e;
}
// One region element's share of the bins, where `in`; lanes that hold one value (a
// tie group) add it once.
__device__ __forceinline__ void thr_bin_add(bool in, uint32_t bits, uint32_t hi, uint32_t sh,
                                            uint64_t* mass, uint32_t* cnt, uint32_t* low) {
  const uint64_t bm = __ballot(in);
  if (bm == 0) return;  // uniform
  const int src = __ffsll((unsigned long long)bm) - 1;
  const uint32_t first = rdlane(bits, src);
  const bool one = __ballot(in && bits != first) == 0;
  if (one ? (int)(threadIdx.x & (kWave - 1)) == src : in) {
    const uint32_t b = (hi - bits) >> sh, n = one ? (uint32_t)__popcll(bm) : 1u;
    atomicAdd((unsigned long long*)&mass[b], (unsigned long long)(n * fixed62(__uint_as_float(bits))));
    atomicAdd(&cnt[b], n);
    atomicMin(&low[b], bits);
  }
}

constexpr int kThrCount = 2 * TH_NT;  // lists up to here are sorted by TH_NT threads, by counting
template <int NT>
struct ThrResLds {
  uint64_t e[kThrList];  // the list; the refinement's masses
  uint32_t cnt[TH_NB], low[TH_NB];
  uint64_t s64[NT / kWave];
  ThrWalkLds w;
  ThrPickLds pick;
  uint32_t n, idcut;
  union {
    uint64_t t[NT > TH_NT ? kThrList : kThrCount];  // a list sorted by counting
    ThrQueue<4> q[NT / kWave];
  };
};
static_assert(kThrList >= kThrCount && kThrList >= TH_NB, "the refinement's masses use the list's space");

// Logits that can have p in [lo, hi] (bits): m - s = -ln(p zf), with the margins of xcut;
// a subnormal bound does not cut.
struct ThrWindow {
  float lo, hi;
  __device__ __forceinline__ ThrWindow(const ThrCtl* c, float T, uint32_t pl, uint32_t ph) {
    const float m = c->m, lz = logf(c->zf);
    auto at = [&](uint32_t bits, float sgn) {
      const float d = logf(__uint_as_float(bits)) + lz;
      const float x = ((m + d) + sgn * (4e-6f * (fabsf(m) + fabsf(d)) + 2e-5f)) * T;
      return x + sgn * 4e-6f * fabsf(x);
    };
    lo = pl >= 0x00800000u ? fmaxf(at(pl, -1.0f), c->xcut) : c->xcut;
    hi = ph >= 0x00800000u ? at(ph, 1.0f) : INFINITY;
    if (!(fabsf(lo) < INFINITY)) lo = c->xcut;
    if (!(fabsf(hi) < INFINITY)) hi = INFINITY;
  }
  __device__ __forceinline__ bool has(float x) const { return x >= lo && x <= hi; }
};
// p of an element, the lanes' where `ok`; a wave whose logits are all the last one's
// (a tie group) keeps its p.
struct ThrEval {
  float m, zf, T, lx = __builtin_nanf(""), lp = 0.0f;
  __device__ __forceinline__ float operator()(float x, bool ok) {
    if (__ballot(ok && x != lx) == 0) return lp;  // uniform
    const float p = exp_det_sel(x / T - m) / zf;
    const uint64_t bm = __ballot(ok);
    const int src = __ffsll((unsigned long long)bm) - 1;
    const float x0 = __uint_as_float(rdlane(__float_as_uint(x), src));
    if (__ballot(ok && x != x0) == 0) {
      lx = x0;
      lp = __uint_as_float(rdlane(__float_as_uint(p), src));
    }
    return p;
  }
};
// Every element of the row in the window through g(x, id, ok) by full waves of the
// NT threads; 16 elements a lane in flight.
template <class E, int NT, class G>
__device__ __forceinline__ void thr_scan(const E* __restrict__ row, int64_t V, const ThrWindow& w,
                                         ThrQueue<4>& q, G&& g) {
  constexpr int N = ThrVec<E>::N, UN = 16 / N;
  const int tid = threadIdx.x;
  uint32_t n = 0;
  int64_t head = (int64_t)(((16u - ((uint32_t)(uintptr_t)row & 15u)) & 15u) / sizeof(E));
  if (head > V) head = V;
  const int64_t nv = (V - head) / N;
  if (tid < kWave) {  // the ends, as in thr_stream
    const int64_t i = tid < 32 ? tid : head + nv * N + (tid - 32);
    const bool ok = tid < 32 ? i < head : i < V;
    const float x = ok ? thr_f(row[i]) : 0.0f;
    thr_push(q, n, x, (uint32_t)i, ok && w.has(x));
  }
  const uint4* __restrict__ x4 = reinterpret_cast<const uint4*>(row + head);
  for (int64_t b = 0; b < nv; b += (int64_t)UN * NT) {  // uniform
    uint4 v[UN];
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      const int64_t j = b + (int64_t)u * NT + tid;
      v[u] = j < nv ? x4[j] : make_uint4(0, 0, 0, 0);
    }
#pragma nounroll
    for (int h = 0; h < 4; ++h) {  // four elements of each lane, by selects (see the output)
      const int u = h * UN / 4;
      uint4 y = v[0];
#pragma unroll
      for (int k = 1; k < UN; ++k) {
        y.x = u == k ? v[k].x : y.x;
        y.y = u == k ? v[k].y : y.y;
        y.z = u == k ? v[k].z : y.z;
        y.w = u == k ? v[k].w : y.w;
      }
      const int64_t j = b + (int64_t)u * NT + tid;
      const int64_t i = head + j * N + (N > 4 ? 4 * (h & 1) : 0);
      if constexpr (N > 4) {
        y.x = h & 1 ? y.z : y.x;
        y.y = h & 1 ? y.w : y.y;
      }
      const uint32_t c[4] = {y.x, y.y, y.z, y.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float x;
        if constexpr (sizeof(E) == 4) x = __uint_as_float(c[e]);
        else x = thr_f((uint16_t)(c[e >> 1] >> (16 * (e & 1))));
        thr_push(q, n, x, (uint32_t)(i + e), j < nv && w.has(x));
      }
      thr_drain(q, n, false, g);
    }
  }
  thr_drain(q, n, true, g);
}
// The id of member `k` (from 0, by id) of the tie group of p = v: the ids are split over
// the waves, which count their members, then the part that holds it again.
template <class E, int NT>
__device__ __forceinline__ uint32_t thr_member(const ThrArgs& a, ThrResLds<NT>& L, const E* row,
                                               const ThrWindow& w, ThrEval ev, float v, uint64_t k) {
  constexpr int NW = NT / kWave;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wv = tid / kWave;
  int64_t lo = 0, hi = a.V;
  auto members = [&](float x, bool ok) {
    const bool c = ok && w.has(x);
    return __ballot(c) == 0 ? 0ull : __ballot(ev(x, c) == v && c);
  };
  while (hi - lo > kWave) {  // uniform
    const int64_t per = ((hi - lo + NW - 1) / NW + kWave - 1) / kWave * kWave;
    const int64_t i0 = lo + wv * per, i1 = min(hi, i0 + per);
    uint32_t n = 0;
    for (int64_t i = i0; i < i1; i += 8 * kWave) {
      E c[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) c[u] = row[min(i + u * kWave + lane, hi - 1)];
#pragma unroll
      for (int u = 0; u < 8; ++u)
        n += (uint32_t)__popcll(members(thr_f(c[u]), i + u * kWave + lane < i1));
    }
    __syncthreads();
    if (lane == 0) L.s64[wv] = n;
    __syncthreads();
    int s = 0;
    while (s < NW - 1 && k >= L.s64[s]) k -= L.s64[s++];
    lo += s * per;
    hi = min(hi, lo + per);
  }
  const bool ok = lo + lane < hi;
  const uint64_t bm = members(ok ? thr_f(row[lo + lane]) : 0.0f, ok);
  const uint32_t at = __builtin_amdgcn_mbcnt_hi((uint32_t)(bm >> 32),
                                                __builtin_amdgcn_mbcnt_lo((uint32_t)bm, 0u));
  if (wv == 0 && ((bm >> lane) & 1u) && at == (uint32_t)k) L.idcut = (uint32_t)(lo + lane);
  __syncthreads();
  return L.idcut;
}
// True: e is the end. False: r is narrowed to at most kThrList elements, which are in
// L.e. A pass takes about 15 us at 151,936 elements: the row by one CU, compared with the
// window, the elements in it evaluated by full waves.
template <class E, int NT>
__device__ __forceinline__ bool thr_refine(const ThrArgs& a, ThrResLds<NT>& L, const E* x,
                                           const ThrCtl* c, ThrSpan& r, ThrEnd& e) {
  const int tid = threadIdx.x, wv = tid / kWave;
  ThrEval ev{c->m, c->zf, a.T};
  while (true) {  // at most four rounds: [lo, hi] shrinks by TH_NB
    const ThrWindow w(c, a.T, r.lo, r.hi);
    __syncthreads();
    if (r.n <= (uint32_t)kThrList) {
      if (tid == 0) L.n = 0u;
      __syncthreads();
      thr_scan<E, NT>(x, a.V, w, L.q[wv], [&](float xv, uint32_t id, bool ok) {
        const uint32_t bits = __float_as_uint(ev(xv, ok));
        const bool in = ok && bits >= r.lo && bits <= r.hi;
        const uint64_t bm = __ballot(in);
        if (bm == 0) return;  // uniform
        uint32_t at = 0;
        if ((tid & (kWave - 1)) == 0) at = atomicAdd(&L.n, (uint32_t)__popcll(bm));
        at = rdlane(at, 0) + __builtin_amdgcn_mbcnt_hi((uint32_t)(bm >> 32),
                                                       __builtin_amdgcn_mbcnt_lo((uint32_t)bm, 0u));
        if (in && at < (uint32_t)kThrList) L.e[at] = ((uint64_t)(~bits) << 32) | id;
      });
      __syncthreads();
      return false;
    }
    if (r.lo == r.hi) {
      const float v = __uint_as_float(r.lo);
      const uint64_t kept = r.use_p ? thr_tie_kept(v, r.above, r.nabove, r.n, a.top_p) : r.n;
      e = thr_tie_end(r, kept);
      if (e.partial) e.idcut = thr_member<E, NT>(a, L, x, w, ev, v, kept - 1);
      return true;
    }
    for (int b = tid; b < TH_NB; b += NT) { L.e[b] = 0ull; L.cnt[b] = 0u; L.low[b] = ~0u; }
    __syncthreads();
    const uint32_t sh = thr_bin_shift(r);
    thr_scan<E, NT>(x, a.V, w, L.q[wv], [&](float xv, uint32_t, bool ok) {
      const uint32_t bits = __float_as_uint(ev(xv, ok));
      thr_bin_add(ok && bits >= r.lo && bits <= r.hi, bits, r.hi, sh, L.e, L.cnt, L.low);
    });
    __syncthreads();
    if (!thr_pick<NT>(a, L.e, L.cnt, L.low, sh, r, L.pick, L.s64)) {
      e.vf = __uint_as_float(r.lo);
      e.tot = r.above;
      return true;
    }
  }
}

// One workgroup per row. Only a refinement and lists of more than kThrCount entries use
// more than the first TH_NT threads (a list of 2,048 by counting with 1,024 threads, 15
// us less than a bitonic sort with 256); the others end at once otherwise. NT 1,024 where every row has a CU of its own (a row of
// 131,072 equal logits, T = 0.7, top_p 0.9, top-k 50 231 us against 546 with 256), 256
// for more rows (fp16 to_probs of 576 rows of 32,000 85 us, 89 with 1,024).
template <class E, int NT>
__global__ void __launch_bounds__(NT) thr_resolve_kernel(ThrArgs a) {
  __shared__ ThrResLds<NT> L;
  const int64_t row = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const ThrCtl* const c = thr_ctl(a, row);
  // everything that needs no other is loaded before the first wait
  const uint32_t n = c->nlist;
  const E* const x = thr_row<E>(a, row);
  const float m = c->m, zf = c->zf, T = a.T;
  const uint64_t pm = lane < a.nlight ? c->pmass[lane] : 0ull;
  const uint32_t pc = lane < a.nlight ? c->pcnt[lane] : 0u;
  const uint32_t pnf = lane < a.nlight ? c->pnf[lane] : 0u;
  const int64_t gid = thr_gid(a, row);
  ThrSpan sp;
  sp.use_k = c->use_k != 0;
  sp.use_p = c->use_p != 0;
  float phi = c->phi;
  if (NT > TH_NT && n <= (uint32_t)kThrCount && tid >= TH_NT) return;  // whole waves
  const float xg = gid >= 0 && gid < a.V ? thr_f(x[gid]) : 0.0f;
  sp.above = wave_sum_u64(pm);
  sp.nabove = wave_sum_u32(pc);
  sp.n = n;
  ThrEnd r;
  r.tot = sp.above;
  bool done = !(sp.use_k || sp.use_p);
  if (__builtin_expect(n > (uint32_t)kThrList, 0)) {  // uniform
    sp.lo = __float_as_uint(c->plo);
    sp.hi = __float_as_uint(fminf(phi, 1.0f));
    done = thr_refine<E, NT>(a, L, x, c, sp, r);
    phi = __uint_as_float(sp.hi);
  } else if (!done) {
    const uint64_t* const list = reinterpret_cast<const uint64_t*>(c + 1);
    for (uint32_t i = tid; i < n; i += n > (uint32_t)kThrCount ? NT : TH_NT) L.e[i] = list[i];
  }
  if (!done) {  // uniform
    auto walk = [&](auto nt, auto count) {
      uint32_t S = kThrCount;
      while (S < sp.n) S <<= 1;
      for (uint32_t i = sp.n + tid; i < S; i += nt.value) L.e[i] = ~0ull;
      __syncthreads();
      r = thr_walk<nt.value>(a, thr_sort<nt.value, count.value>(L.e, L.t, sp.n), sp.n, sp.use_k,
                             sp.use_p, sp.above, sp.nabove, phi, L.w, L.s64);
    };
    if (NT > TH_NT && sp.n > (uint32_t)kThrCount) {  // uniform
      walk(std::integral_constant<int, NT>{}, std::integral_constant<int, NT == TH_NT ? kThrCount : kThrList>{});
    } else {
      if (tid >= TH_NT) return;  // whole waves
      walk(std::integral_constant<int, TH_NT>{}, std::integral_constant<int, kThrCount>{});
    }
  }
  const bool nonfinite = __ballot(pnf != 0) != 0;
  if (tid == 0) a.stats[row] = thr_record(r, m, zf, c->xcut, gid, a.V, xg, T, nonfinite);
}

// ---------------------------------------------------------------- short rows
// Rows of at most kThrSmall elements: the same in one launch, a workgroup per row that
// holds the row in registers (PER elements a thread: 256 threads for rows of up to
// 2,048, 512 up to 4,096, 1,024 above, so that short rows share a CU). A region of more
// than a list of NT is refined as above, from the registers. With `out`, also the
// to_probs row. Bound by the latency of its chain of block reductions. to_probs of 64
// fp32 rows of 4,096: 13 us against 69 us for a bitonic sort of the row in LDS, of 256
// of 8,192 21 against 131 us, of 20,000 of 64 148 against 1,141 us.
template <int NT>
struct ThrSmallLds {
  uint64_t e[NT];  // the region's list
  union {
    struct {
      uint64_t mass[TH_NB];
      uint32_t cnt[TH_NB], low[TH_NB];
    } h;
    uint64_t t[NT];
  };
  uint64_t s64[NT / kWave], t64[NT / kWave];
  uint32_t u32[NT / kWave];
  float mx[NT / kWave], mn[NT / kWave];
  ThrWalkLds w;
  ThrPickLds pick;
  uint32_t n, idcut;
  int32_t b0, b1, bk, nf;
};
// Appends the lanes' (p, id) with `in` to the list of NT, counting all.
template <int NT>
__device__ __forceinline__ void thr_small_list(ThrSmallLds<NT>& L, bool in, float p, uint32_t id) {
  const uint64_t bm = __ballot(in);
  if (bm == 0) return;  // uniform per wave
  uint32_t at = 0;
  if ((threadIdx.x & (kWave - 1)) == 0) at = atomicAdd(&L.n, (uint32_t)__popcll(bm));
  at = rdlane(at, 0) + __builtin_amdgcn_mbcnt_hi((uint32_t)(bm >> 32),
                                                 __builtin_amdgcn_mbcnt_lo((uint32_t)bm, 0u));
  if (in && at < (uint32_t)NT) L.e[at] = ((uint64_t)(~__float_as_uint(p)) << 32) | id;
}
// The refinement: as thr_refine, over the p of the workgroup's elements u NT + thread
// (0 past the row).
template <int NT, int PER>
__device__ __forceinline__ bool thr_small_refine(const ThrArgs& a, ThrSmallLds<NT>& L,
                                                 const float (&p)[PER], ThrSpan& r, ThrEnd& e) {
  constexpr int NW = NT / kWave;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wv = tid / kWave;
  static_assert(PER * NW <= TH_NB, "the members' counts use the bins' space");
  while (true) {  // at most four rounds: [lo, hi] shrinks by TH_NB
    __syncthreads();
    if (r.n <= (uint32_t)NT) {
      if (tid == 0) L.n = 0u;
      __syncthreads();
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        const uint32_t bits = __float_as_uint(p[u]);
        thr_small_list<NT>(L, bits >= r.lo && bits <= r.hi, p[u], (uint32_t)(u * NT + tid));
      }
      __syncthreads();
      return false;
    }
    if (r.lo == r.hi) {
      const uint64_t kept =
          r.use_p ? thr_tie_kept(__uint_as_float(r.lo), r.above, r.nabove, r.n, a.top_p) : r.n;
      e = thr_tie_end(r, kept);
      if (!e.partial) return true;  // uniform
      // the id of member kept - 1: members by (u, wave, lane)
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        const uint64_t bm = __ballot(__float_as_uint(p[u]) == r.lo);
        if (lane == 0) L.h.cnt[u * NW + wv] = (uint32_t)__popcll(bm);
      }
      __syncthreads();
      uint32_t k = (uint32_t)kept - 1u, s = 0;
      while (s < (uint32_t)(PER * NW - 1) && k >= L.h.cnt[s]) k -= L.h.cnt[s++];
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        const bool mem = __float_as_uint(p[u]) == r.lo;
        const uint64_t bm = __ballot(mem);
        const uint32_t at = __builtin_amdgcn_mbcnt_hi((uint32_t)(bm >> 32),
                                                      __builtin_amdgcn_mbcnt_lo((uint32_t)bm, 0u));
        if (s == (uint32_t)(u * NW + wv) && mem && at == k) L.idcut = (uint32_t)(u * NT + tid);
      }
      __syncthreads();
      e.idcut = L.idcut;
      return true;
    }
    for (int b = tid; b < TH_NB; b += NT) { L.h.mass[b] = 0ull; L.h.cnt[b] = 0u; L.h.low[b] = ~0u; }
    __syncthreads();
    const uint32_t sh = thr_bin_shift(r);
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const uint32_t bits = __float_as_uint(p[u]);
      thr_bin_add(bits >= r.lo && bits <= r.hi, bits, r.hi, sh, L.h.mass, L.h.cnt, L.h.low);
    }
    __syncthreads();
    if (!thr_pick<NT>(a, L.h.mass, L.h.cnt, L.h.low, sh, r, L.pick, L.s64)) {
      e.vf = __uint_as_float(r.lo);
      e.tot = r.above;
      return true;
    }
  }
}

template <class E, int NT, int PER>
__global__ void __launch_bounds__(NT) thr_small_kernel(ThrArgs a, float* out, int64_t ld_out) {
  constexpr int NW = NT / kWave;
  constexpr int BPT = TH_NB / NT;  // steps per thread
  __shared__ ThrSmallLds<NT> L;
  const int64_t row = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wv = tid / kWave;
  const E* const xr = thr_row<E>(a, row);
  const int V = (int)a.V;
  const float T = a.T;
  const int64_t gid = thr_gid(a, row);
  float xg = 0.0f;
  if (tid == 0) {
    if (row < a.nzero) a.zero[row] = 0u;
    if (gid >= 0 && gid < V) xg = thr_f(xr[gid]);
    L.n = 0u;
    L.b0 = L.b1 = L.bk = TH_NB - 1;
    L.nf = 0;
  }
#pragma unroll
  for (int i = 0; i < BPT; ++i) {
    L.h.mass[tid + i * NT] = 0ull;
    L.h.cnt[tid + i * NT] = 0u;
  }
  float x[PER];
  E raw[PER];  // all loads first
  float mx = -INFINITY, mn = INFINITY;
  bool nf = false;
#pragma unroll
  for (int u = 0; u < PER; ++u) raw[u] = xr[min(u * NT + tid, V - 1)];
#pragma unroll
  for (int u = 0; u < PER; ++u) x[u] = u * NT + tid < V ? thr_f(raw[u]) : -INFINITY;
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    if (sizeof(E) == 2) nf |= (int32_t)__float_as_uint(x[u]) >= 0x7F800000;
    mx = fmaxf(mx, x[u]);
    mn = x[u] > -INFINITY ? fminf(mn, x[u]) : mn;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    mx = fmaxf(mx, __shfl_xor(mx, o, kWave));
    mn = fminf(mn, __shfl_xor(mn, o, kWave));
  }
  if (lane == 0) { L.mx[wv] = mx; L.mn[wv] = mn; }
  const uint64_t nfw = __ballot(nf);
  __syncthreads();
  if (lane == 0 && nfw) atomicOr(&L.nf, 1);
#pragma unroll
  for (int w = 0; w < NW; ++w) { mx = fmaxf(mx, L.mx[w]); mn = fminf(mn, L.mn[w]); }
  const float m = mx / T;
  const float scale = thr_scale(a, m, mn);
  const uint32_t steps = thr_steps(a, scale);
  const ThrDiv div = thr_div_kind(T, mx);
  uint64_t zlo = 0;
  uint32_t zhi = 0;
  const float rT = 1.0f / T;
  thr_hist_kind(a, div, [&](auto DIV, auto MASS, auto CNT) {
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      if (u * NT >= V) break;  // uniform
      thr_hist_one<DIV.value, MASS.value, CNT.value>(x[u], u * NT + tid < V, T, rT, m, scale,
                                                     steps, L.h.mass, L.h.cnt, zlo, zhi);
    }
  });
  U128 z = wave_sum_u128(U128{zlo, (uint64_t)zhi});
  if (lane == 0) { L.s64[wv] = z.lo; L.t64[wv] = z.hi; }
  __syncthreads();  // and the histogram is complete
  z = U128{0, 0};
  for (int w = 0; w < NW; ++w) z = u128_add(z, U128{L.s64[w], L.t64[w]});
  const float zf = rn32_u128(z);
  const bool bad = !(zf > 0.0f);
  ThrEnd r;
  ThrCut c;
  if (!a.use_k && !a.use_p) {  // uniform: everything is above
    c = thr_cut(a, m, zf, scale, 0, 0, 0);
  } else {
    uint64_t ms[BPT], ct[BPT], sm = 0, sc = 0;
#pragma unroll
    for (int i = 0; i < BPT; ++i) {
      ms[i] = L.h.mass[tid * BPT + i];
      ct[i] = L.h.cnt[tid * BPT + i];
      sm += ms[i];
      sc += ct[i];
    }
    uint64_t rm = thr_excl_u64<NW>(sm, L.s64);
    uint64_t rc = a.use_k ? thr_excl_u64<NW>(sc, L.s64) : 0ull;
    const double zu = ((double)z.hi * 0x1p64 + (double)z.lo) * 0x1p-18;
#pragma unroll
    for (int i = 0; i < BPT; ++i) {
      thr_mark(a, tid * BPT + i, rm, rm + ms[i], rc, rc + ct[i], zu, &L.b0, &L.b1, &L.bk);
      rm += ms[i];
      rc += ct[i];
    }
    __syncthreads();
    c = thr_cut(a, m, zf, scale, L.b0, L.b1, L.bk);
  }
  // p of this thread's elements; what lies above the region, and the region's list
  float p[PER];
  uint64_t mass = 0;
  uint32_t cnt = 0;
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    p[u] = 0.0f;
    if (u * NT >= V) continue;  // uniform
    const int i = u * NT + tid;
    const bool take = i < V && x[u] >= c.xcut;
    if (__ballot(take)) p[u] = take ? exp_det_sel(x[u] / T - m) / zf : 0.0f;
    const bool above = take && p[u] > c.phi;
    mass += above ? fixed62(p[u]) : 0ull;
    cnt += above ? 1u : 0u;
    thr_small_list<NT>(L, take && !above && p[u] >= c.plo, p[u], (uint32_t)i);
  }
  mass = wave_sum_u64(mass);
  cnt = wave_sum_u32(cnt);
  __syncthreads();  // the scans' words are read, the list is complete
  if (lane == 0) { L.s64[wv] = mass; L.u32[wv] = cnt; }
  __syncthreads();
  uint64_t above = 0, nabove = 0;
  for (int w = 0; w < NW; ++w) { above += L.s64[w]; nabove += L.u32[w]; }
  ThrSpan sp;
  sp.above = above;
  sp.nabove = nabove;
  sp.n = L.n;
  sp.use_k = c.use_k;
  sp.use_p = c.use_p;
  r.tot = above;
  bool done = !(c.use_k || c.use_p);
  float phi = c.phi;
  if (__builtin_expect(sp.n > (uint32_t)NT, 0)) {  // uniform
    sp.lo = __float_as_uint(c.plo);
    sp.hi = __float_as_uint(fminf(phi, 1.0f));
    done = thr_small_refine<NT, PER>(a, L, p, sp, r);
    phi = __uint_as_float(sp.hi);
  }
  if (!done) {  // uniform
    for (uint32_t i = sp.n + tid; i < (uint32_t)NT; i += NT) L.e[i] = ~0ull;
    __syncthreads();
    r = thr_walk<NT>(a, thr_sort<NT, NT>(L.e, L.t, sp.n), sp.n, sp.use_k, sp.use_p, sp.above,
                     sp.nabove, phi, L.w, L.s64);
  }
  if (tid == 0 && a.stats)
    a.stats[row] = thr_record(r, m, zf, c.xcut, gid, V, xg, T, L.nf != 0);
  if (!out) return;
  const float totf = fmaxf(rn32_u64(r.tot), 1e-12f);
  float* const o = out + row * ld_out;
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int i = u * NT + tid;
    const bool kept = p[u] > r.vf || (p[u] == r.vf && (uint32_t)i <= r.idcut);
    if (i < V) o[i] = bad ? __builtin_nanf("") : kept ? p[u] / totf : 0.0f;
  }
}

// ---------------------------------------------------------------- rows without a filter
// softmax alone, a workgroup per row and one launch: maximum, exact normaliser, p and its
// exact sum (p waits in the output row), division. The row's later passes come from the
// L2. Bound by the instructions of two exps per element. fp32 to_probs at T = 0.7, us, the
// kernels above | this: 1 row of 8,200 38 | 13, of 32,000 39 | 33, of 40,000 39 | 42; 256
// rows of 8,200 47 | 15, of 32,000 83 | 44; 1,024 rows of 32,000 228 | 135. fp16: 1 row of
// 32,000 40 | 37, 256 rows 85 | 47.
constexpr int TP_NT = 1024, TP_NW = TP_NT / kWave;
template <class E>
__global__ void __launch_bounds__(TP_NT) thr_plain_kernel(ThrArgs a, float* out, int64_t ld_out) {
  constexpr int N = ThrVec<E>::N;
  __shared__ uint64_t s64[TP_NW], t64[TP_NW];
  __shared__ float s_mx[TP_NW];
  const int64_t row = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wv = tid / kWave;
  const E* const x = thr_row<E>(a, row);
  float* const o = out + row * ld_out;
  const int64_t V = a.V;
  int64_t head = (int64_t)(((16u - ((uint32_t)(uintptr_t)x & 15u)) & 15u) / sizeof(E));
  if (head > V) head = V;
  const int64_t nv = (V - head) / N;
  // the elements before the first and after the last whole vector: one a thread
  const int64_t ie = tid < N ? (tid < head ? tid : -1)
                             : tid < 2 * N && head + nv * N + (tid - N) < V
                                   ? head + nv * N + (tid - N) : -1;
  const float xe = ie >= 0 ? thr_f(x[ie]) : 0.0f;
  const uint4* const x4 = reinterpret_cast<const uint4*>(x + head);
  auto elem = [](const uint4& w, int e) {
    const uint32_t q[4] = {w.x, w.y, w.z, w.w};
    if constexpr (sizeof(E) == 4) return __uint_as_float(q[e]);
    else return thr_f((uint16_t)(q[e >> 1] >> (16 * (e & 1))));
  };
  float mx = ie >= 0 ? xe : -INFINITY;
  for (int64_t j = tid; j < nv; j += TP_NT) {
    const uint4 w = x4[j];
#pragma unroll
    for (int e = 0; e < N; ++e) mx = fmaxf(mx, elem(w, e));
  }
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) mx = fmaxf(mx, __shfl_xor(mx, d, kWave));
  if (lane == 0) s_mx[wv] = mx;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < TP_NW; ++w) mx = fmaxf(mx, s_mx[w]);
  const float T = a.T, m = mx / T;
  uint64_t zlo = 0;
  uint32_t zhi = 0;
  auto add = [&](float v) {
    const uint64_t f = thr_exp62(v / T - m);
    zlo += f;
    zhi += zlo < f ? 1u : 0u;
  };
  if (ie >= 0) add(xe);
#pragma unroll 2
  for (int64_t j = tid; j < nv; j += TP_NT) {
    const uint4 w = x4[j];
#pragma unroll
    for (int e = 0; e < N; ++e) add(elem(w, e));
  }
  U128 z = wave_sum_u128(U128{zlo, (uint64_t)zhi});
  if (lane == 0) { s64[wv] = z.lo; t64[wv] = z.hi; }
  __syncthreads();
  z = U128{0, 0};
  for (int w = 0; w < TP_NW; ++w) z = u128_add(z, U128{s64[w], t64[w]});
  const float zf = rn32_u128(z);
  const bool bad = !(zf > 0.0f);  // no finite maximum: every probability is 0 / 0
  const bool vec = ((uintptr_t)(o + head) & 15u) == 0;  // uniform
  uint64_t mass = 0;
  auto prob = [&](float v) {  // a NaN logit has no mass, as above
    const float p = v == v ? exp_det_sel(v / T - m) / zf : 0.0f;
    mass += fixed62(p);
    return bad ? __builtin_nanf("") : p;
  };
  if (ie >= 0) o[ie] = prob(xe);
#pragma unroll 2
  for (int64_t j = tid; j < nv; j += TP_NT) {
    const uint4 w = x4[j];
    float* const d = o + head + j * N;
#pragma unroll
    for (int h = 0; h < N; h += 4) {
      const float4 p = make_float4(prob(elem(w, h)), prob(elem(w, h + 1)), prob(elem(w, h + 2)),
                                   prob(elem(w, h + 3)));
      if (vec) {
        *reinterpret_cast<float4*>(d + h) = p;
      } else {
        d[h] = p.x; d[h + 1] = p.y; d[h + 2] = p.z; d[h + 3] = p.w;
      }
    }
  }
  mass = wave_sum_u64(mass);
  __syncthreads();  // the normaliser's words are read
  if (lane == 0) s64[wv] = mass;
  __syncthreads();
  uint64_t tot = 0;
  for (int w = 0; w < TP_NW; ++w) tot += s64[w];
  const float totf = fmaxf(rn32_u64(tot), 1e-12f);
  // a thread's own elements again
  if (ie >= 0) o[ie] = o[ie] / totf;
#pragma unroll 2
  for (int64_t j = tid; j < nv; j += TP_NT) {
    float* const d = o + head + j * N;
#pragma unroll
    for (int h = 0; h < N; h += 4) {
      if (vec) {
        float4 p = *reinterpret_cast<const float4*>(d + h);
        p.x /= totf; p.y /= totf; p.z /= totf; p.w /= totf;
        *reinterpret_cast<float4*>(d + h) = p;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) d[h + e] /= totf;
      }
    }
  }
}

// ---------------------------------------------------------------- to_probs output
// Wave by wave: zeros first, 16 bytes a lane, then the kept elements, compacted and
// evaluated by full waves, over them (the wave waits for its zeros).
constexpr int TH_OUT = 8192;  // ids per workgroup: 32 a thread

template <class E>
__global__ void __launch_bounds__(TH_NT) thr_output_kernel(ThrArgs a, float* out, int64_t ld_out,
                                                           int nchunk) {
  constexpr int N = ThrVec<E>::N;
  constexpr int UN = TH_OUT / (TH_NT * N);
  constexpr int GR = 16 / N;  // vectors between two drains
  __shared__ ThrQueue<GR * N> sq[TH_NW];
  const int64_t row = blockIdx.x / nchunk;
  const int ch = (int)(blockIdx.x % nchunk);
  const int tid = threadIdx.x, wv = tid / kWave;
  const E* const x = thr_row<E>(a, row);
  float* const o = out + row * ld_out;
  const ThrRow r = thr_load_row(a.stats[row]);
  const bool bad = (a.stats[row].flags & kRowNoMass) != 0;
  const float T = a.T;
  int64_t head = (int64_t)(((16u - ((uint32_t)(uintptr_t)x & 15u)) & 15u) / sizeof(E));
  if (head > a.V) head = a.V;
  const int64_t nv = (a.V - head) / N;
  const int64_t v0 = (int64_t)ch * (TH_OUT / N), v1 = min(nv, v0 + TH_OUT / N);
  const uint4* const x4 = reinterpret_cast<const uint4*>(x + head);
  uint4 w[UN];
#pragma unroll
  for (int u = 0; u < UN; ++u) {
    const int64_t j = v0 + (int64_t)u * TH_NT + tid;
    w[u] = j < v1 ? x4[j] : make_uint4(0, 0, 0, 0);
  }
  const float fill = bad ? __builtin_nanf("") : 0.0f;
  const bool vec = ((uintptr_t)(o + head) & 15u) == 0;  // uniform
  auto one = [&](int64_t i) {  // the row's ends, one element a lane
    o[i] = bad ? fill : thr_prob(r, thr_f(x[i]), (uint32_t)i, T);
  };
  if (ch == 0 && tid < head) one(tid);
  if (ch == nchunk - 1 && head + nv * N + tid < a.V) one(head + nv * N + tid);
#pragma unroll
  for (int u = 0; u < UN; ++u) {
    const int64_t j = v0 + (int64_t)u * TH_NT + tid;
    if (j >= v1) continue;
    float* const d = o + head + j * N;
    if (vec) {
#pragma unroll
      for (int q = 0; q < N / 4; ++q)
        reinterpret_cast<float4*>(d)[q] = make_float4(fill, fill, fill, fill);
    } else {
#pragma unroll
      for (int e = 0; e < N; ++e) d[e] = fill;
    }
  }
  if (bad) return;  // uniform
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0x0F70);  // gfx9 encoding: vmcnt(0)
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  auto put = [&](float xv, uint32_t id, bool ok) {
    const float p = thr_prob(r, xv, id, T);
    if (ok && p != 0.0f) o[id] = p;
  };
  uint32_t n = 0;
#pragma nounroll
  for (int g = 0; g < UN / GR; ++g) {
#pragma unroll
    for (int u = 0; u < GR; ++u) {
      // group g's vectors by selects: an index known at run time would put w in memory
      uint4 wu = w[u];
#pragma unroll
      for (int h = 1; h < UN / GR; ++h) {
        const uint4 y = w[h * GR + u];
        wu.x = g == h ? y.x : wu.x;
        wu.y = g == h ? y.y : wu.y;
        wu.z = g == h ? y.z : wu.z;
        wu.w = g == h ? y.w : wu.w;
      }
      const int64_t j = v0 + (int64_t)(g * GR + u) * TH_NT + tid;
      const bool ok = j < v1;
      const int64_t i = head + j * N;
      const uint32_t q[4] = {wu.x, wu.y, wu.z, wu.w};
#pragma unroll
      for (int e = 0; e < N; ++e) {
        float xv;
        if constexpr (sizeof(E) == 4) xv = __uint_as_float(q[e]);
        else xv = thr_f((uint16_t)(q[e >> 1] >> (16 * (e & 1))));
        thr_push(sq[wv], n, xv, (uint32_t)(i + e), ok && xv >= r.xcut);
      }
    }
    thr_drain(sq[wv], n, g == UN / GR - 1, put);
  }
}

// ---------------------------------------------------------------- draw
// The verify's accept chain and draw (or, with acc.k = 0, a draft step's draw): a wave
// per record of kThrRec ids reduces it to its p and residual masses, which need only
// the ids where p is kept; the workgroup that completes a batch row's records adds
// them up, picks the one that holds floor(u * total) and walks its ids. Members of a
// boundary tie group are decided by their ids, so nothing depends on earlier records.
struct ThrDrawLds {
  ThrQueue<kThrRec / kWave> q[TH_NW];
  RowStat st[2];
  SampleJob job;
  uint32_t fl;
  int32_t last;
  uint64_t s64[TH_NW], t64[TH_NW];
  int64_t pick, found;
  uint64_t at;
};
constexpr int TH_RV = kThrRec / TH_NT;  // ids per thread of the walk (4)
static_assert(TH_RV * TH_NT == kThrRec, "the walk takes a record with the workgroup");

template <class E>
__global__ void __launch_bounds__(TH_NT) thr_draw_kernel(ThrDrawArgs a) {
  __shared__ ThrDrawLds S;
  const int64_t j = blockIdx.x / a.nblk;
  const int bi = (int)(blockIdx.x % a.nblk);
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wv = tid / kWave;
  if (tid < kWave) {
    SampleJob jb;
    uint32_t fl;
    int64_t n;
    if (a.acc.k <= 31) {  // uniform: the 2k + 1 rows' records at once, one per lane
      // (no row here is left for the chain to rank, so the row source is not read)
      n = chain16_wave<SDX_F16, false>(a.acc, Eval16<SDX_F16>{}, j, &jb, &fl, S.st);
    } else {
      n = accept_chain_wave(a.acc, j, &jb, &fl);
      if (lane == 0) {
        S.st[0] = a.acc.stats[jb.prow];
        S.st[1] = a.acc.stats[jb.qrow >= 0 ? jb.qrow : jb.prow];
      }
    }
    if (lane == 0) {
      if (bi == 0 && a.acc.n_acc) a.acc.n_acc[j] = n;
      S.job = jb;
      S.fl = fl;
      S.pick = -1;
      S.found = -1;
    }
  }
  __syncthreads();
  const SampleJob job = S.job;
  const bool hasq = job.qrow >= 0;
  auto rowp = [&](int64_t row) {
    const int g = row < a.nrows0 ? 0 : 1;
    return reinterpret_cast<const E*>(a.base[g]) + (g ? row - a.nrows0 : row) * a.ld[g];
  };
  const E* const xp = rowp(job.prow);
  const E* const xq = hasq ? rowp(job.qrow) : xp;
  const RowStat sp = S.st[0];
  const RowStat sq = S.st[hasq ? 1 : 0];
  const ThrRow rp = thr_load_row(sp), rq = thr_load_row(sq);
  const float T = a.T;
  const int64_t V = a.V;
  // ---- records
  const int rec = bi * TH_NW + wv;
  uint64_t mp = 0, mr = 0;
  if (rec < a.nrec) {  // uniform per wave
    const int64_t r0 = (int64_t)rec * kThrRec;
    constexpr int RN = kThrRec / kWave;
    // codes first, unconditionally: an element's bounds check and conversion between
    // the loads made each wait for the one before (fp16: 5 us for the 16)
    E raw[RN];
#pragma unroll
    for (int u = 0; u < RN; ++u) raw[u] = xp[min(r0 + u * kWave + lane, V - 1)];
    float x[RN];
#pragma unroll
    for (int u = 0; u < RN; ++u) x[u] = thr_f(raw[u]);
    auto add = [&](float xv, uint32_t id, bool ok) {
      const float qx = hasq && ok ? thr_f(xq[id]) : 0.0f;
      const float p = ok ? thr_prob(rp, xv, id, T) : 0.0f;
      const float q = hasq && ok ? thr_prob(rq, qx, id, T) : 0.0f;
      mp += fixed62(p);
      mr += hasq ? fixed62(fmaxf(p - q, 0.0f)) : 0ull;
    };
    uint32_t n = 0;
#pragma unroll
    for (int u = 0; u < RN; ++u) {
      const int64_t i = r0 + u * kWave + lane;
      thr_push(S.q[wv], n, x[u], (uint32_t)i, i < V && x[u] >= rp.xcut);
    }
    thr_drain(S.q[wv], n, true, add);
    mp = wave_sum_u64(mp);
    mr = wave_sum_u64(mr);
    if (lane == 0) {
      uint64_t* const d = a.recs + 2 * (j * a.nrec + rec);
      __hip_atomic_store(d, mp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(d + 1, mr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  // ---- the workgroup whose count completes the records goes on (stores done first)
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0x0F70);  // gfx9 encoding: vmcnt(0)
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __syncthreads();
  if (tid == 0)
    S.last = __hip_atomic_fetch_add(&a.counters[j], 1u, __ATOMIC_RELAXED,
                                    __HIP_MEMORY_SCOPE_AGENT) == (uint32_t)(a.nblk - 1);
  __syncthreads();
  if (!S.last) return;  // uniform
  static_assert(kF32MaxVocab <= (int64_t)TH_NT * kThrRec, "one record per thread");
  mp = mr = 0;
  if (tid < a.nrec) {
    const uint64_t* const d = a.recs + 2 * (j * a.nrec + tid);
    mp = __hip_atomic_load(d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    mr = __hip_atomic_load(d + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  const uint64_t ip = wave_incl_scan_u64(mp, lane), ir = wave_incl_scan_u64(mr, lane);
  if (lane == kWave - 1) { S.s64[wv] = ip; S.t64[wv] = ir; }
  __syncthreads();
  uint64_t ep = ip - mp, er = ir - mr, totp = 0, totr = 0;
  for (int w = 0; w < TH_NW; ++w) {
    ep += w < wv ? S.s64[w] : 0ull;
    er += w < wv ? S.t64[w] : 0ull;
    totp += S.s64[w];
    totr += S.t64[w];
  }
  const bool use_r = hasq && rn32_u64(totr) > 1e-9f;  // sampling.py:85-88
  const uint64_t tot = use_r ? totr : totp, e0 = use_r ? er : ep, mine = use_r ? mr : mp;
  const uint64_t t = uniform_threshold(job.u, tot);
  if (tot > 0 && e0 <= t && t - e0 < mine) {  // exactly one thread
    S.pick = tid;
    S.at = e0;
  }
  __syncthreads();
  const int64_t pick = S.pick;
  float pw = 0.0f;  // p of this thread's ids, the found one's kept
  if (pick >= 0) {  // uniform
    const int64_t i0 = pick * kThrRec + (int64_t)tid * TH_RV;
    uint64_t w[TH_RV], sum = 0;
    float pv[TH_RV];
    E pc[TH_RV], qc[TH_RV];
#pragma unroll
    for (int u = 0; u < TH_RV; ++u) {  // all loads first
      pc[u] = xp[min(i0 + u, V - 1)];
      qc[u] = xq[min(i0 + u, V - 1)];
    }
#pragma unroll
    for (int u = 0; u < TH_RV; ++u) {
      const int64_t i = i0 + u;
      const float p = i < V ? thr_prob(rp, thr_f(pc[u]), (uint32_t)i, T) : 0.0f;
      const float q = use_r && i < V ? thr_prob(rq, thr_f(qc[u]), (uint32_t)i, T) : 0.0f;
      pv[u] = p;
      w[u] = fixed62(use_r ? fmaxf(p - q, 0.0f) : p);
      sum += w[u];
    }
    const uint64_t st = S.at + thr_excl_u64(sum, S.s64);
    if (st <= t && t - st < sum) {  // exactly one thread
      uint64_t acc = st;
      int64_t f = -1;
#pragma unroll
      for (int u = 0; u < TH_RV; ++u) {
        acc += w[u];
        if (f < 0 && acc > t) { f = i0 + u; pw = pv[u]; }
      }
      S.found = f;
      if (a.qx) a.qx[j] = pw;
    }
    __syncthreads();
  }
  if (tid != 0) return;
  const int64_t y = S.found;
  a.y[j] = y;
  if (a.qx && y < 0) a.qx[j] = 0.0f;
  if (a.acc.flags) {
    uint32_t fl = S.fl;
    auto tie = [&](const ThrRow& r, const RowStat& st, const E* x) {
      return st.rstar > 0 && st.rstar < st.gcount &&
             exp_det(thr_f(x[y]) / T - r.m) / r.zf == r.vf;
    };
    if (y >= 0 && (tie(rp, sp, xp) || (use_r && tie(rq, sq, xq)))) fl |= SDX_FLAG_TIE_ORDER;
    a.acc.flags[j] = (uint8_t)fl;
  }
}

// ---------------------------------------------------------------- launches

// How far below the maximum (in s) the steps reach. The k-th largest can be anywhere p is
// above 0 (104 units); alone, in the thousands and at ordinary temperatures it is within
// 32, and finite mask values do not widen the steps (where it is not, the last step is
// refined: fp16 to_probs of 72 rows of 131,072, N(0, 1) with a -1e4 mask, T = 2, top-k
// 5000 102 -> 86 us with the lists below). A nucleus ends where less than 1 - top_p of the mass is left,
// and D units below the maximum that is at most V e^-D of it (of at least 1): within 15
// units for V = 151,936 and top_p 0.95, so that a row's finite mask values do not widen
// the steps; 32 units where top_p is so near 1 that its rounding counts. With a top-k
// too, the nucleus bounds the range only at low temperatures (see thr_hist_one).
constexpr float TH_LOWT = 0.25f;
static float thr_dmax(const ThrArgs& a) {
  const bool near = !a.use_k || (!a.use_p && a.top_k > 1024 && a.T >= 0.7f);
  const double most = near ? 32.0 : 104.0;
  const double rest = 1.0 - (double)a.top_p - 2e-6;  // the region's margin of 1e-6, and roundings
  if (!a.use_p || rest < 2e-6 || (a.use_k && a.T > TH_LOWT)) return (float)most;
  return (float)fmin(most, log((double)a.V) - log(rest) + 0.25);
}

// Parts per row: about four workgroups per CU over the call, parts of at least 4,096
// elements (below that a part's histogram costs more than its stream), and no more
// than the first pass has words for.
static int thr_parts(int64_t rows, int64_t V) {
  const int64_t want = (1024 + rows - 1) / rows;
  int64_t p = want < V / 4096 ? want : V / 4096;
  if (p > kThrMaxParts) p = kThrMaxParts;
  return (int)(p < 1 ? 1 : p);
}


// Of the passes that only compare: as many workgroups as the chip holds waves for.
static int thr_light_parts(int64_t rows, int64_t V) {
  const int64_t want = (2048 + rows - 1) / rows, most = V / 4096;
  const int64_t p = want < most ? want : most;
  return (int)(p < 1 ? 1 : p > kThrMaxParts ? kThrMaxParts : p);
}

template <class E>
static hipError_t thr_stats(const ThrArgs& a, int64_t rows, hipStream_t s) {
  const dim3 grid((unsigned)(rows * a.nparts)), light((unsigned)(rows * a.nlight));
  hipLaunchKernelGGL(thr_max_kernel<E>, light, dim3(TH_NT), 0, s, a);
  if (a.T <= TH_LOWT) hipLaunchKernelGGL((thr_hist_kernel<E, true>), grid, dim3(TH_NT), 0, s, a);
  else hipLaunchKernelGGL((thr_hist_kernel<E, false>), grid, dim3(TH_NT), 0, s, a);
  hipLaunchKernelGGL(thr_collect_kernel<E>, light, dim3(TH_NT), 0, s, a);
  if (rows <= 256)
    hipLaunchKernelGGL((thr_resolve_kernel<E, 1024>), dim3((unsigned)rows), dim3(1024), 0, s, a);
  else
    hipLaunchKernelGGL((thr_resolve_kernel<E, 256>), dim3((unsigned)rows), dim3(256), 0, s, a);
  return hipGetLastError();
}

template <class E>
static hipError_t thr_small(const ThrArgs& a, int64_t rows, float* out, int64_t ld_out,
                            hipStream_t s) {
  const dim3 grid((unsigned)rows);
  if (a.V <= 8 * 256)
    hipLaunchKernelGGL((thr_small_kernel<E, 256, 8>), grid, dim3(256), 0, s, a, out, ld_out);
  else if (a.V <= 8 * 512)
    hipLaunchKernelGGL((thr_small_kernel<E, 512, 8>), grid, dim3(512), 0, s, a, out, ld_out);
  else
    hipLaunchKernelGGL((thr_small_kernel<E, 1024, 8>), grid, dim3(1024), 0, s, a, out, ld_out);
  return hipGetLastError();
}

hipError_t launch_thr_small(int dtype, ThrArgs a, int64_t rows, float* out, int64_t ld_out,
                            hipStream_t s) {
  a.dmax = thr_dmax(a);
  if (a.V > kThrSmall || (!a.stats && !out)) return hipErrorInvalidValue;
  return dtype == SDX_F32 ? thr_small<float>(a, rows, out, ld_out, s)
                          : thr_small<uint16_t>(a, rows, out, ld_out, s);
}

// Above this a row is too long for one workgroup of a call with few (see the kernel).
bool thr_plain(int64_t V, int use_k, int use_p) { return !use_k && !use_p && V <= 32768; }

hipError_t launch_thr_plain(int dtype, const ThrArgs& a, int64_t rows, float* out, int64_t ld_out,
                            hipStream_t s) {
  const dim3 grid((unsigned)rows);
  if (dtype == SDX_F32)
    hipLaunchKernelGGL(thr_plain_kernel<float>, grid, dim3(TP_NT), 0, s, a, out, ld_out);
  else
    hipLaunchKernelGGL(thr_plain_kernel<uint16_t>, grid, dim3(TP_NT), 0, s, a, out, ld_out);
  return hipGetLastError();
}

hipError_t launch_thr_stats(int dtype, ThrArgs a, int64_t rows, hipStream_t s) {
  if (a.V <= kThrSmall) return launch_thr_small(dtype, a, rows, nullptr, 0, s);
  if (!a.scratch || a.scratch_bytes < kThrScratchMin || a.scratch_stride < a.scratch_bytes || !a.stats || a.V > kF32MaxVocab)
    return hipErrorInvalidValue;
  a.dmax = thr_dmax(a);
  a.nparts = thr_parts(rows, a.V);
  const int64_t per = (a.V + a.nparts - 1) / a.nparts;
  a.plen = (per + 7) / 8 * 8;  // whole vectors of either element size
  a.nlight = thr_light_parts(rows, a.V);
  const int64_t lper = (a.V + a.nlight - 1) / a.nlight;
  a.llen = (lper + 7) / 8 * 8;
  return dtype == SDX_F32 ? thr_stats<float>(a, rows, s) : thr_stats<uint16_t>(a, rows, s);
}

hipError_t launch_thr_output(int dtype, const ThrArgs& a, int64_t rows, float* out, int64_t ld_out,
                             hipStream_t s) {
  const int nchunk = (int)((a.V + TH_OUT - 1) / TH_OUT);
  const dim3 grid((unsigned)(rows * nchunk));
  if (dtype == SDX_F32)
    hipLaunchKernelGGL(thr_output_kernel<float>, grid, dim3(TH_NT), 0, s, a, out, ld_out, nchunk);
  else
    hipLaunchKernelGGL(thr_output_kernel<uint16_t>, grid, dim3(TH_NT), 0, s, a, out, ld_out, nchunk);
  return hipGetLastError();
}

hipError_t launch_thr_draw(int dtype, ThrDrawArgs a, int64_t jobs, hipStream_t s) {
  a.nrec = (int32_t)((a.V + kThrRec - 1) / kThrRec);
  a.nblk = (a.nrec + TH_NW - 1) / TH_NW;
  const dim3 grid((unsigned)(jobs * a.nblk));
  if (dtype == SDX_F32) hipLaunchKernelGGL(thr_draw_kernel<float>, grid, dim3(TH_NT), 0, s, a);
  else hipLaunchKernelGGL(thr_draw_kernel<uint16_t>, grid, dim3(TH_NT), 0, s, a);
  return hipGetLastError();
}

}  // namespace sdx
