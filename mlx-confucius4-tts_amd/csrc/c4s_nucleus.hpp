// One nucleus step (top_k off, 0 < p < 1) of a row staged in LDS, by the waves
// of one workgroup: the exact steps of the stream's full-vocabulary chain,
// whose rows of more than kListLarge kept ids (flat rows: top_p 0.9 at a
// temperature of 1.2) have no other path. One pass takes the reference's
// masses exp((double)fl(z - m)) (sampling.cpp:55) into LDS and a histogram of
// them on buckets of 1/32; the boundary's few entries are sorted and the cut
// (sampling.cpp:60-65) and the draw (text2semantic.cpp:150-165) decided with
// margins, as the other one-pass paths do. The multi-pass chain it stands in
// front of takes four radix passes with an exponential and two LDS atomics a
// value: 70 us a step of 8194 ids on six waves.

#pragma once

#include "c4s_chain.hpp"

namespace c4s {
namespace {

constexpr int kNucNB = 1024;             // buckets of 1 / kNucScale below the maximum
constexpr float kNucScale = 32.0f;
constexpr int kNucX = 256;               // boundary entries
constexpr int kNucU = 4;                 // ids of a thread taken together

template <int NWX>
struct NucSh {
  unsigned long long hist[kNucNB];       // masses, 2^-31 units
  unsigned long long list[kNucX], sorted[kNucX];
  double wd[2][NWX];
  uint32_t wu[2][NWX];
  float wf[NWX];
  uint32_t xlo, xhi, n;
  unsigned long long kthr;
  int tok;
};
template <int NWX>
__host__ __device__ __forceinline__ size_t nucleus_bytes(int V) { return 8 * (size_t)V + sizeof(NucSh<NWX>); }

// Exclusive and inclusive prefix of v and the total over the workgroup, and the
// total of u, one barrier (`set` alternates between calls).
struct NucScan {
  double ex, in, tot;
  uint32_t utot;
};
template <int NWX>
__device__ __forceinline__ NucScan nuc_scan(double v, uint32_t u, NucSh<NWX>& sh, int set) {
  const int w = wave_id();
  const double inc = wave_scan_f64(v);
  const uint32_t ui = wave_scan_u32(u);
  if (lane_id() == kWave - 1) { sh.wd[set][w] = inc; sh.wu[set][w] = ui; }
  __syncthreads();
  NucScan r;
  double base = 0.0, run = 0.0;
  uint32_t ut = 0;
#pragma unroll
  for (int i = 0; i < NWX; ++i) {
    if (i == w) base = run;
    run += sh.wd[set][i];
    ut += sh.wu[set][i];
  }
  r.ex = base + wave_shr1_f64(inc, 0.0);
  r.in = base + inc;
  r.tot = run;
  r.utot = ut;
  return r;
}

// X: the penalised row (not changed), area: nucleus_bytes(V) of LDS. True with
// the token, the statistics and the RNG advanced when the step is decided;
// false (uniform, nothing changed but the area) otherwise. Barriers on entry
// and exit are the caller's.
template <int NWX>
__device__ __forceinline__ bool nucleus_lds(const float* X, const RowCfg& c, unsigned char* area, uint64_t& rng, int& tok,
                                            uint32_t* stats) {
  constexpr int NTX = NWX * kWave;
  static_assert(NTX >= kNucX, "a thread an entry");
  double* E = reinterpret_cast<double*>(area);
  NucSh<NWX>& sh = *reinterpret_cast<NucSh<NWX>*>(area + 8 * (size_t)c.V);
  const int V = c.V, t = threadIdx.x, lane = lane_id(), w = wave_id();
  const double thr = 1.0 - (double)c.p;   // sampling.cpp:64 removes while cum <= 1 - p
  if (!c.draw || c.topk_on || !(thr > 0.0) || !(thr < 1.0)) return false;
  const double rt = 1.0 / (double)c.temp;
  auto z_of = [&](float y) { return c.temp_on ? div_rcp(y, rt) : y; };
  const int P = odd_chunk<NTX>(V);        // consecutive ids a thread: id order is thread order
  static_assert((kLdsVocabMax + NTX - 1) / NTX < kWave, "a thread's ids, one a lane");
  const int lo = min(V, t * P), hi = min(V, lo + P);
  for (int i = t; i < kNucNB; i += NTX) sh.hist[i] = 0ull;
  if (t == 0) { sh.xlo = kNucNB; sh.xhi = kNucNB; sh.n = 0u; sh.tok = -1; }
  // the loops over a thread's ids go kNucU at a time: reads in bounds (index
  // clamped) and issued together, what lies past the ids selected away
  float lm = neg_inf();
  for (int i = lo; i < hi; i += kNucU) {
    float x[kNucU];
#pragma unroll
    for (int u = 0; u < kNucU; ++u) x[u] = X[min(i + u, hi - 1)];
#pragma unroll
    for (int u = 0; u < kNucU; ++u) lm = fmaxf(lm, x[u]);
  }
  lm = wave_max_dpp(lm);
  if (lane == 0) sh.wf[w] = lm;
  __syncthreads();
  float my = neg_inf();
#pragma unroll
  for (int i = 0; i < NWX; ++i) my = fmaxf(my, sh.wf[i]);
  const float m = z_of(my);               // the quotient is monotone in y
  if (!(fabsf(m) < 0x1p18f)) return false;   // the grid's differences are exact below; uniform
  const float fQ = floorf(m * kNucScale);
  // the masses, their sum, the histogram
  double s = 0.0;
  for (int i = lo; i < hi; i += kNucU) {
    float x[kNucU];
#pragma unroll
    for (int u = 0; u < kNucU; ++u) x[u] = X[min(i + u, hi - 1)];
#pragma unroll
    for (int u = 0; u < kNucU; ++u) {
      const float z = i + u < hi ? z_of(x[u]) : neg_inf();
      const double e = exp_neg((double)(z - m));   // 0 for -inf
      if (i + u < hi) E[i + u] = e;
      s += e;
      const float d = fQ - floorf(z * kNucScale);
      if (d < (float)(kNucNB - 1)) atomicAdd(&sh.hist[(int)d], (unsigned long long)(uint32_t)(e * 0x1p31));
    }
  }
  const double S = nuc_scan<NWX>(s, 0u, sh, 0).tot;
  // the buckets in which the kept mass S - thr S is reached: four a thread
  // (truncation: 2^-31 a value; values more than 32 below the maximum are left out)
  const double B = S - thr * S, err = S * 0x1p-40 + (double)V * 0x1p-30;
  {
    double h4[4], loc = 0.0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      h4[q] = 4 * t + q < kNucNB ? (double)sh.hist[min(4 * t + q, kNucNB - 1)] * 0x1p-31 : 0.0;
      loc += h4[q];
    }
    const NucScan sc = nuc_scan<NWX>(loc, 0u, sh, 1);
    double run = sc.ex;
    uint32_t a = kNucNB, b = kNucNB;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      run += h4[q];
      if (a == kNucNB && run >= B - err) a = 4 * t + q;
      if (b == kNucNB && run >= B + err) b = 4 * t + q;
    }
    // the first of each wave (the prefixes do not decrease)
    const uint64_t ba = __ballot(a < kNucNB), bb = __ballot(b < kNucNB);
    if (ba && lane == __ffsll((unsigned long long)ba) - 1) atomicMin(&sh.xlo, a);
    if (bb && lane == __ffsll((unsigned long long)bb) - 1) atomicMin(&sh.xhi, b);
  }
  __syncthreads();
  const float xlo = (float)sh.xlo, xhi = (float)sh.xhi;
  if (!(xhi < (float)(kNucNB - 1))) return false;   // uniform
  // the mass above X, and X's entries
  double ab = 0.0;
  uint32_t nab = 0;
  for (int i = lo; i < hi; i += kNucU) {
    float x[kNucU];
    double ei[kNucU];
#pragma unroll
    for (int u = 0; u < kNucU; ++u) {
      x[u] = X[min(i + u, hi - 1)];
      ei[u] = E[min(i + u, hi - 1)];
    }
#pragma unroll
    for (int u = 0; u < kNucU; ++u) {
      const float z = i + u < hi ? z_of(x[u]) : neg_inf();
      const float d = fQ - floorf(z * kNucScale);
      ab += d < xlo ? ei[u] : 0.0;
      nab += d < xlo ? 1u : 0u;
      if (!(d < xlo) && d <= xhi) {
        const uint32_t slot = atomicAdd(&sh.n, 1u);
        if (slot < (uint32_t)kNucX) sh.list[slot] = ((uint64_t)fkey(z) << 32) | (uint32_t)~(uint32_t)(i + u);
      }
    }
  }
  const NucScan as = nuc_scan<NWX>(ab, nab, sh, 0);
  const double Ma = as.tot;
  nab = as.utot;
  const int nX = (int)sh.n;   // every push came before the scan's barrier
  if (nX > kNucX) return false;   // uniform
  // by (value desc, id asc): each key's place is the count of keys above it, the
  // four lanes of a quad counting over every fourth entry
  for (int b = 0; b < nX; b += NTX / 4) {
    const int i = b + (t >> 2), q = t & 3;
    const uint64_t mine = sh.list[min(i, nX - 1)];
    uint32_t r = 0;
    int j = 0;
    for (; j + 16 <= nX; j += 16) {
      uint64_t o[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) o[u] = sh.list[j + 4 * u + q];
#pragma unroll
      for (int u = 0; u < 4; ++u) r += o[u] > mine ? 1u : 0u;
    }
    for (; j < nX; j += 4) r += (j + q < nX && sh.list[min(j + q, nX - 1)] > mine) ? 1u : 0u;
    r += xor_lane_u32<1>(r);
    r += xor_lane_u32<2>(r);
    if (q == 0 && i < nX) sh.sorted[r] = mine;
  }
  __syncthreads();
  // entry j is removed iff the mass at or below it in ascending order,
  // M = S - (mass above it), is <= thr S (sampling.cpp:60-65)
  const uint64_t ent = sh.sorted[min(t, kNucX - 1)];
  const double e = t < nX ? E[(int)~(uint32_t)ent] : 0.0;
  const NucScan xs = nuc_scan<NWX>(e, 0u, sh, 1);
  const int mk = max(0, c.min_keep);
  const double A = thr * S, M = S - (Ma + xs.ex);
  const bool kept = t < nX && M > A;
  const bool unsure = t < nX && !(fabs(M - A) > rel_eps(V) * S) && nab + (uint32_t)t >= (uint32_t)mk;
  const NucScan ks = nuc_scan<NWX>(0.0, (kept ? 1u : 0u) | (unsure ? 1u << 16 : 0u), sh, 0);
  if (ks.utot >> 16) return false;   // uniform
  uint32_t nk = ks.utot;
  if (nab + nk < (uint32_t)mk) {   // sampling.cpp:67-68: the top min_keep positions stay
    if ((uint32_t)mk > nab + (uint32_t)nX) return false;
    nk = (uint32_t)mk - nab;
  }
  if (nX == 0 || nab + nk == 0u) return false;
  const uint64_t kthr = nk > 0u ? (uint64_t)sh.sorted[nk - 1u] : (uint64_t)sh.sorted[0] + 1ull;
  // subnormal kept masses (libm implementations may disagree), and the draw's floor of -1e30 (far above)
  if (kfloat((uint32_t)(kthr >> 32)) - m < -690.0f) return false;
  // the kept masses in id order; a removed id's mass becomes 0
  double kd = 0.0;
  for (int i = lo; i < hi; i += kNucU) {
    float x[kNucU];
    double ei[kNucU];
#pragma unroll
    for (int u = 0; u < kNucU; ++u) {
      x[u] = X[min(i + u, hi - 1)];
      ei[u] = E[min(i + u, hi - 1)];
    }
#pragma unroll
    for (int u = 0; u < kNucU; ++u) {
      const uint64_t key = ((uint64_t)fkey(z_of(x[u])) << 32) | (uint32_t)~(uint32_t)(i + u);
      const double ek = i + u < hi && key >= kthr ? ei[u] : 0.0;
      if (i + u < hi) E[i + u] = ek;   // the thread's own ids
      kd += ek;
    }
  }
  const NucScan ds = nuc_scan<NWX>(kd, 0u, sh, 1);
  const uint64_t st2 = xorshift64(rng);
  const double r = unit_from_state(st2) * ds.tot, mg = 2.0 * rel_eps(V) * ds.tot;
  if (r > 0.0) {
    const uint64_t own = __ballot(ds.ex < r && r <= ds.in);
    if (own) {   // the owner's wave: the owner's ids one a lane, their sums by a wave scan
      const int ol = __ffsll((unsigned long long)own) - 1;
      const int lo_o = (int)readlane_u32((uint32_t)lo, ol), n_o = (int)readlane_u32((uint32_t)(hi - lo), ol);
      const double ex_o = readlane_f64(ds.ex, ol);
      const double el = lane < n_o ? E[lo_o + lane] : 0.0;
      const double al = ex_o + wave_scan_f64(el);
      const uint64_t hit = __ballot(el > 0.0 && al >= r);
      if (hit) {
        const int f = __ffsll((unsigned long long)hit) - 1;
        const double af = readlane_f64(al, f), pf = af - readlane_f64(el, f);
        if (lane == 0 && af - r > mg && r - pf > mg) sh.tok = lo_o + f;
      }
    }
    __syncthreads();
    tok = sh.tok;
    if (tok < 0) return false;   // uniform
  } else {
    tok = 0;   // r == 0: the first id satisfies r <= acc (text2semantic.cpp:161-162)
  }
  rng = st2;
  if (stats && t == 0) {
    stats[0] = 1u | 4u;
    stats[1] = 0u;
    stats[2] = 0u;
    stats[3] = nab + nk;
  }
  return true;
}

}  // namespace
}  // namespace c4s
