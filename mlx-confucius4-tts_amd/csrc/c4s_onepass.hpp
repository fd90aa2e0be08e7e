// The parts of the one-AR-step kernels (k_rows_step and its form for many
// rows): the row's outputs, the draw, the tie cut, the fallback chain, the
// candidate-list step and the one pass of a sampled row.

#pragma once

#include "c4s_list.hpp"
#include "c4s_step.hpp"

namespace c4s {
namespace {

// Writes one row's result: token, RNG state, history set (text2semantic.cpp:
// 333-334: the stop token does not join), statistics.
__device__ __forceinline__ void step_out(const StepIO& io, int V, int tok, uint64_t rng, bool draw,
                                         uint32_t s0, uint32_t s1, uint32_t s2, uint32_t s3) {
  *io.out_tok = tok;
  if (draw && io.rng) *io.rng = rng;
  if (io.join && tok >= 0 && tok < V && tok != io.stop_token) atomicOr(&io.join[tok >> 5], 1u << (tok & 31));
  if (io.stats) { io.stats[0] = s0; io.stats[1] = s1; io.stats[2] = s2; io.stats[3] = s3; }
}

// The draw of the one-pass step (text2semantic.cpp:150-165) once the kept set
// is known: the kept fp32 masses of each thread and ds, the workgroup scan of
// their sums with the error bound in tot2. The thread whose interval holds r
// decides. When it cannot (r within the bound of one end of its entry: on a
// flat row of thousands of kept entries a few percent of rows a call), the
// masses are taken again in double: at most 64 kept ids go in id order (kl, by
// the scan's kept counts) to one wave, which draws on them and replays the
// sums sequentially if that is too close (lane_draw); otherwise every thread
// recomputes its kept masses, the workgroup scans them (bound rel_eps, about
// 1e-11 relative) and the owner's wave walks the owner's ids, one a lane; only
// if that still does not decide does one wave replay the draw sequentially
// over the row (draw_replay).
// The row's configuration and I/O as one LDS copy for the workgroup: the
// out-of-line helpers take them by reference, and a reference to a copy in
// registers would make the compiler keep that copy in per-lane scratch memory
// for the whole kernel (about 120 bytes a lane written at entry).
struct StepRowSh {
  RowCfg cfg;
  StepIO io;
  uint32_t tp_exact_first;   // 1: the one pass's top_p test missed its margin in double
};

template <int PT, bool kCached>
__device__ __forceinline__ void draw_finish(const StepIO& io, const RowCfg& c, const KeptRule& kr, const float (&z)[PT],
                                            int lo, int n, float m, const Scan2& ds, uint32_t n_kept,
                                            uint32_t st_path, uint32_t st_exact, StepSh& ss, const StepRowSh& rs,
                                            const float* em, uint64_t* kl) {
  const int t = threadIdx.x;
  const uint64_t st2 = xorshift64(*io.rng);
  const double u = unit_from_state(st2);
  const double K = ds.tot;
  const double r = u * K;
  const double margin = 2.0 * ds.tot2 + rel_eps(c.V) * K;
  if (!(r > 0.0)) {   // r == 0: the first id satisfies r <= acc (text2semantic.cpp:161-162)
    if (t == 0) step_out(io, c.V, 0, st2, true, st_path, st_exact, 0u, n_kept);
    return;
  }
  const bool owner = (ds.ex < r && r <= ds.in) || (t == kStepThreads - 1 && r > ds.in);
  int found = -1;
  bool certain = false;
  C4S_PHASE_IF(owner, 18);
  const uint64_t obw = __ballot(owner);
  if (obw) {
    // the owner's wave: lane j takes the owner's id lo + j and its kept fp32
    // mass (independent loads and tests, one a lane), the running sums in id
    // order by a wave scan in double from the owner's exclusive prefix (its
    // rounding, about 2^-53 relative a step, lies far inside the margin), then
    // the first kept id whose sum reaches r and the sums on both sides of it
    const int ol = __ffsll((unsigned long long)obw) - 1, l = lane_id();
    float zl = neg_inf();
#pragma unroll
    for (int j = 0; j < PT; ++j) {
      const float zj = readlane_f32(z[j], ol);
      zl = (l == j) ? zj : zl;
    }
    const int lo_o = (int)readlane_u32((uint32_t)lo, ol);
    const double ex_o = readlane_f64(ds.ex, ol);
    float el;   // lanes past the owner's ids hold -inf: not kept
    if constexpr (kCached) {
      const float ec = em[min(lo_o + l, c.V - 1)];
      el = ((int)(zl != neg_inf()) & (int)kept_in(kr, zl, m, lo_o + l)) ? ec : 0.0f;
    } else {
      bool kp;
      el = kept_mass32(kr, zl, m, lo_o + l, kp);
    }
    const double al = ex_o + wave_scan_f64((double)el);
    const uint64_t hit = __ballot(el > 0.0f && al >= r);
    if (hit) {
      const int f = __ffsll((unsigned long long)hit) - 1;
      const double af = readlane_f64(al, f);
      const double pf = f > 0 ? readlane_f64(al, max(f - 1, 0)) : ex_o;
      found = lo_o + f;
      certain = (af - r > margin) && (r - pf > margin);
    }
  }
  C4S_PHASE_IF(owner, 19);
  if (!__syncthreads_or(owner && !certain)) {
    if (owner) step_out(io, c.V, found, st2, true, st_path, st_exact, 0u, n_kept);
    return;
  }
  // the kept masses in double. The kept test is the one pass's (kept_in): a
  // dense row reaches this draw only without values whose double mass lies
  // near underflow, so `z - m > -745` there is exactly `exp((double)(z - m)) > 0`.
  C4S_PHASE(24);
  if (n_kept <= (uint32_t)kWave) {
    // at most 64 kept ids: in id order (thread order, then the thread's own)
    // to one wave, which draws on them in double and replays the sums
    // sequentially when that is too close (lane_draw)
    uint32_t km = 0;
#pragma unroll
    for (int j = 0; j < PT; ++j)
      km |= ((int)(j < n) & (int)(z[j] != neg_inf()) & (int)kept_in(kr, z[j], m, lo + j)) ? 1u << j : 0u;
#pragma unroll
    for (int j = 0; j < PT; ++j)
      if ((km >> j) & 1u)
        kl[ds.uex + (uint32_t)__popc(km & ((1u << j) - 1u))] = ((uint64_t)__float_as_uint(z[j]) << 32) | (uint32_t)(lo + j);
    __syncthreads();
    if (wave_id() == 0) {
      const int l = lane_id();
      const bool in = l < (int)n_kept;
      const uint64_t ent = kl[in ? l : 0];
      const double e = in ? exp((double)(__uint_as_float((uint32_t)(ent >> 32)) - m)) : 0.0;
      uint32_t ex2 = 0;
      const int tk = lane_draw<6>(in, (int)(uint32_t)ent, l, e, u, c.V, ex2);
      if (l == 0) step_out(io, c.V, tk, st2, true, st_path, st_exact, 1u + ex2, n_kept);
    }
    return;
  }
  double dk = 0.0;
#pragma unroll
  for (int j = 0; j < PT; ++j)
    if (j < n && z[j] != neg_inf() && kept_in(kr, z[j], m, lo + j)) dk += exp((double)(z[j] - m));
  const Scan2 d2 = block_scan2(dk, 0.0, 0u, ss.wa, ss.wb, ss.wu);
  C4S_PHASE(25);
  const double r2 = u * d2.tot;
  const double m2 = 2.0 * rel_eps(c.V) * d2.tot;
  const bool own2 = (d2.ex < r2 && r2 <= d2.in) || (t == kStepThreads - 1 && r2 > d2.in);
  found = -1;
  certain = false;
  const uint64_t ob = __ballot(own2);
  if (ob) {   // the owner's wave: lane j takes the owner's id lo + j, the prefix by a wave scan
    const int ol = __ffsll((unsigned long long)ob) - 1, l = lane_id();
    float zl = neg_inf();
#pragma unroll
    for (int j = 0; j < PT; ++j) {
      const float zj = readlane_f32(z[j], ol);
      zl = (l == j) ? zj : zl;
    }
    const int lo_o = readlane_u32((uint32_t)lo, ol), n_o = readlane_u32((uint32_t)n, ol);
    const double ex_o = readlane_f64(d2.ex, ol);
    const bool kp = ((int)(l < n_o) & (int)(zl != neg_inf()) & (int)kept_in(kr, zl, m, lo_o + l)) != 0;
    const double el = kp ? exp((double)(zl - m)) : 0.0;
    const double al = ex_o + wave_scan_f64(el);
    const uint64_t hit = __ballot(el > 0.0 && al >= r2);
    if (r2 > 0.0 && hit) {
      const int f = __ffsll((unsigned long long)hit) - 1;
      const double af = readlane_f64(al, f), pf = af - readlane_f64(el, f);
      found = lo_o + f;
      certain = (af - r2 > m2) && (r2 - pf > m2);
    }
  }
  C4S_PHASE(26);
  if (!__syncthreads_or(own2 && !certain)) {
    if (own2) step_out(io, c.V, found, st2, true, st_path, st_exact, 1u, n_kept);
    return;
  }
  if (wave_id() == 0) {   // the reference's sequential sums, one wave
    const int tk = draw_replay(rs.io, rs.cfg, kr, m, u);
    if (lane_id() == 0) step_out(io, c.V, tk, st2, true, st_path, st_exact, 2u, n_kept);
  }
}

// sampling.cpp:52-65 replayed for a row whose top group X (nX entries at the
// maximum, mass 1 each) is preceded in ascending order by entries of total
// mass B (known within relative `re` of the reference's sequential sum):
// total = B + 1 + ... + 1 and cum = sum of prob / total, both sequential. The
// sums over the entries below X reach the sequence only through B and B /
// total; each enters one add (B + 1, then B / total + 1 / total), which rounds
// every value of its interval to one double, or the replay gives up (-1).
// Returns the members of X kept (cum > thr), the rest removed in order.
__device__ __forceinline__ int tie_top_exact(double B, int nX, double thr, double re) {
  const double t_lo = B * (1.0 - 2.0 * re) + 1.0, t_hi = B * (1.0 + 2.0 * re) + 1.0;
  if (t_lo != t_hi) return -1;
  const double tot = repeat_add(t_lo, 1.0, nX - 1, -1.0, true).x;
  const double q = 1.0 / tot;
  const double cb = B / tot, cb_hi = cb * (1.0 + 3.0 * re);
  if (!(cb_hi <= thr)) return -1;   // some entry below X could be kept
  const double c_lo = cb * (1.0 - 3.0 * re) + q, c_hi = cb_hi + q;
  if (c_lo != c_hi) return -1;
  return nX - repeat_add(c_lo, q, nX - 1, thr, false).le;
}

// The cut when the boundary entries X (more than one sort takes) all hold one
// value z*: each has the mass e = exp(z* - m), and in the chain's order (value
// descending, lower id first) X is ordered by id, which is thread order here,
// so a member's rank is a prefix count. Member i is kept iff the mass at or
// below it, M_i = S - (mass above X) - i e, exceeds thr S (sampling.cpp:60-65;
// top_k rows: every member survives top_k, S = the survivors' mass); kept
// members are ranks 0 .. k-1. A decision within the margin is taken again with
// S and the mass above X summed in double, and, when X holds the maximum, by
// replaying the reference's sums over X (tie_top_exact). Sets ss.kthr;
// returns 1 decided, 3 decided with the double sums or the replay, 4 neither
// settles it (the multi-pass chain decides, by the exact emulation), 0 the
// multi-pass chain decides (X holds more than one value; top-k rows;
// min_tokens_to_keep).
template <int PT>
__device__ __noinline__ int tie_cut(const RowCfg& c, const float* val, int lo, int n, const SideRule sr, int nX,
                                    double thr, double S, double errS, double Ma, double eMa, uint32_t n_above,
                                    StepSh& ss) {
  const int lane = lane_id(), w = wave_id();
  const float ninf = neg_inf();
  const bool topk = c.topk_on;
  // z = fl(y / T) by the exact reciprocal division; every read unconditional
  // (index clamped); the loops rolled (code size: this path is rare)
  const double rt = 1.0 / (double)c.temp;
  float zmax = ninf, zmin = -ninf;
  uint32_t cnt = 0;
#pragma unroll 1
  for (int j = 0; j < PT; ++j) {
    const float y = val[min(lo + j, c.V - 1)];
    const float z = c.temp_on ? div_rcp(y, rt) : y;
    const bool inx = ((int)(j < n) & (int)(sr.side(z) == 0)) != 0;
    zmax = inx ? fmaxf(zmax, z) : zmax;
    zmin = inx ? fminf(zmin, z) : zmin;
    cnt += inx ? 1u : 0u;
  }
  zmax = wave_max_dpp(zmax);
  zmin = -wave_max_dpp(-zmin);
  if (lane == 0) { ss.wmax[w] = zmax; ss.wmin[w] = zmin; }
  const Scan2 rk = block_scan2((double)cnt, 0.0, 0u, ss.we, ss.wf, ss.ww);   // includes a barrier
  float zs = ninf, zl = -ninf;
#pragma unroll
  for (int i = 0; i < kStepWaves; ++i) { zs = fmaxf(zs, ss.wmax[i]); zl = fminf(zl, ss.wmin[i]); }
  if (!(zs == zl) || zs == ninf) return 0;   // not one value (or nothing finite)
  C4S_PHASE(24);
  const double e = exp((double)(zs - sr.m));
  const double N = (double)nX;
  const uint32_t mk = (uint32_t)max(0, c.min_keep);
  double Sx = topk ? N * e : S, base = topk ? 0.0 : Ma, err = topk ? 0.0 : 2.0 * errS + eMa;
  double nB = 0.0;   // the mass below X, in double (pass 1)
  int k = 0, verdict = 1;
  for (int pass = 0; pass < 2; ++pass) {
    if (thr <= 0.0) {   // p >= 1: only zero-mass positions can go
      k = (thr < 0.0 || e > 0.0) ? nX : 0;
      break;
    }
    const double A = thr * Sx;
    // k = the members with M_i > A, M_i = Sx - base - i e decreasing in i
    const double q = (Sx - base - A) / e;
    k = q <= 0.0 ? 0 : (q >= N ? nX : (int)ceil(q));
    while (k > 0 && !(Sx - base - (double)(k - 1) * e > A)) --k;
    while (k < nX && Sx - base - (double)k * e > A) ++k;
    const double mg = rel_eps(c.V) * Sx + err;
    const bool sure = (k == 0 || fabs(Sx - base - (double)(k - 1) * e - A) > mg) &&
                      (k == nX || fabs(Sx - base - (double)k * e - A) > mg);
    if (sure) break;
    if (topk) return 0;
    if (pass == 1) {
      // X holds the maximum and nothing lies above it: the reference's sums
      // in ascending order are the entries below X, then X's nX masses of 1.
      // The entries below enter only through their sums, known within
      // rel_eps, which the first add of a mass of 1 (or of 1 / total) rounds
      // to one double unless the interval straddles a rounding boundary; from
      // there the sums over X are replayed exactly.
      if (n_above != 0u || zs != sr.m) return 4;
      C4S_PHASE(25);
      if (threadIdx.x == 0) ss.bsel[0] = tie_top_exact(nB, nX, thr, rel_eps(c.V));   // one thread; the rest wait
      __syncthreads();
      k = ss.bsel[0];
      C4S_PHASE(26);
      if (k < 0) return 4;
      break;
    }
    // decide again with S and the mass above X in double (and the mass below
    // X). X holds the one value zs and side() is monotone in z, so the entries
    // above X are those above zs and the entries below X those below it; z is
    // -inf past the thread's ids (exp(-inf) = 0)
    double se = 0.0, sa = 0.0, sb = 0.0;
#pragma unroll 1
    for (int j = 0; j < PT; ++j) {
      const float y = val[min(lo + j, c.V - 1)];
      const float z = (j < n) ? (c.temp_on ? div_rcp(y, rt) : y) : ninf;
      const double ed = exp((double)(z - sr.m));
      se += ed;
      sa += z > zs ? ed : 0.0;
      sb += z < zs ? ed : 0.0;
    }
    se = wave_sum_dpp(se);
    sa = wave_sum_dpp(sa);
    sb = wave_sum_dpp(sb);
    if (lane == 0) { ss.wc[w] = se; ss.wd[w] = sa; ss.wa[w] = sb; }
    __syncthreads();
    Sx = 0.0;
    base = 0.0;
#pragma unroll
    for (int i = 0; i < kStepWaves; ++i) { Sx += ss.wc[i]; base += ss.wd[i]; nB += ss.wa[i]; }
    err = 0.0;
    verdict = 3;
  }
  // min_tokens_to_keep (sampling.cpp:67-68): the top min_keep positions stay
  if (topk) {
    if ((uint32_t)k < mk) k = (int)min(mk, (uint32_t)nX);
  } else if (n_above + (uint32_t)k < mk) {
    if (mk > n_above + (uint32_t)nX) return 0;
    k = (int)(mk - n_above);
  }
  // the last kept member's key (rank k - 1), or with none kept, one above
  // every member (the lowest id's key + 1)
  C4S_PHASE(27);
  const int want = k > 0 ? k - 1 : 0;
  const int r0 = (int)rk.ex;
  if (cnt > 0 && want >= r0 && want < r0 + (int)cnt) {
    int rank = r0;
    for (int j = 0; j < n; ++j) {
      const float y = val[lo + j];
      const float z = c.temp_on ? y / c.temp : y;
      if (sr.side(z) == 0) {
        if (rank == want) ss.kthr = key64(zs, lo + j) + (k > 0 ? 0ull : 1ull);
        ++rank;
      }
    }
  }
  __syncthreads();
  return verdict;
}

// The multi-pass chain (c4s_chain.hpp) on the penalised row staged in LDS
// (`val`), for the rows the one pass leaves; kept out of line so that its
// registers do not weigh on the one-pass path.
[[maybe_unused]] __device__ __noinline__ void chain_fallback(const StepIO& io, const RowCfg& c, unsigned char* work, float* val,
                                            StepScratch& sh, bool tp_exact_first) {
  const int V = c.V, t = threadIdx.x;
  uint64_t rng = *io.rng;
  LdsRow src{val, reinterpret_cast<double*>(work), V, 0u, false};
  const int tok = run_chain<kStepWaves, LdsRow, true>(src, sh, c, rng, io.masked, sh.step_stats, tp_exact_first);
  if (t == 0) {
    const uint32_t* sp = sh.step_stats;
    step_out(io, V, tok, rng, true, sp[0], sp[1], sp[2], sp[3]);
  }
}

// ---- top-k rows on a candidate list --------------------------------------------------
//
// A sampled row with top_k in [1, 64] is decided by its largest values alone
// (sampling.cpp:30-40 keeps the k largest and their ties; top_p and the draw,
// :42-71 and text2semantic.cpp:150-165, then read the kept entries only). So
// the step takes a candidate list as the AR stream's scan makes it, from the
// penalised values y each thread holds (ids [lo, lo + n), thread order is id
// order): a key L0 at or below the 112th largest of the threads' top-2 keys
// (two 11-bit histogram passes), every value with key(y) >= L0 in id order
// (one workgroup scan), the temperature on those alone (fl(y / T) is monotone
// in y), their sort by (z desc, id asc), and a bound on every value outside.
// One wave then decides the step on the first 128 entries (list_step). When
// the list cannot settle it (a boundary tie group past the list, a cut inside
// the error bound, ...), nothing has been written but the work area, and the
// row takes the one-pass step.
constexpr int kFastList = kListSmall;           // list entries the decision sees
constexpr int kFastSel = kListSmall - 16;       // thread-top keys at or above L0
constexpr int kFastCands = 256;                 // candidates the list step sorts
constexpr int kFastOneBin = 64;                 // thread-top keys from the first pass's bin up: no second pass
static_assert(kStepThreads * 4 == 2048, "four histogram bins a thread");

struct NoHit {   // no id drawn since the list was made
  __device__ __forceinline__ bool hit(int) const { return false; }
};

struct FastSh {
  uint32_t hist[2][2048];      // the two histogram passes; the first then holds the sorted head (uint64)
  uint64_t cand[kFastCands];   // candidates as entries (key of z, id, candidate position)
  uint32_t red[4][kStepWaves];   // one set per workgroup scan (no barrier between reuses)
  uint32_t redm[kStepWaves];
  uint32_t bu[8];
  LSpecCS cs;
};
static_assert(sizeof(FastSh) <= kStepWorkBytes, "the list step's area lies in the one pass's work area");
static_assert(offsetof(FastSh, hist) == 0 && sizeof(FastSh::hist) <= 3 * kHistBytes,
              "the list step's histograms lie in the area the step clears before staging");

// Exclusive scan of v over the workgroup (thread order); total in `tot`. One
// barrier: each call uses its own `red`.
__device__ __forceinline__ uint32_t fast_scan(uint32_t v, uint32_t* red, uint32_t& tot) {
  const uint32_t inc = wave_scan_u32(v);
  if (lane_id() == kWave - 1) red[wave_id()] = inc;
  __syncthreads();
  uint32_t pre = 0;
  tot = 0;
#pragma unroll
  for (int w = 0; w < kStepWaves; ++w) {
    const uint32_t x = red[w];
    pre += (w < wave_id()) ? x : 0u;
    tot += x;
  }
  return pre + inc - v;
}

// Bin of hist (2048 bins, scanned from the top) holding the m-th largest
// counted key, and the count above it, through bu[0..1] of this pick; false
// when fewer than m keys were counted.
__device__ __forceinline__ bool fast_pick(const uint32_t* hist, uint32_t* red, uint32_t* bu, uint32_t m,
                                          uint32_t& bin, uint32_t& above) {
  const int t = threadIdx.x;
  uint32_t cb[4], loc = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) { cb[i] = hist[2047 - 4 * t - i]; loc += cb[i]; }
  uint32_t total;
  const uint32_t ex = fast_scan(loc, red, total);
  if (total < m) return false;   // uniform
  if (ex < m && ex + loc >= m) {
    uint32_t run = ex;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (run < m && run + cb[i] >= m) { bu[0] = 2047 - 4 * t - i; bu[1] = run; }
      run += cb[i];
    }
  }
  __syncthreads();
  bin = bu[0];
  above = bu[1];
  return true;
}

template <int PT>
__device__ __forceinline__ bool list_fast(const StepIO& io, const RowCfg& c, int V, const float (&y)[PT], int lo,
                                          int n, const float* val, FastSh& fs) {
  const int t = threadIdx.x, lane = lane_id(), wv = wave_id();
  const double rt = 1.0 / (double)c.temp;   // used only when the temperature applies
  uint32_t ky[PT];
#pragma unroll
  for (int j = 0; j < PT; ++j) ky[j] = fkey(y[j]);
  if (n < PT) {   // the last threads: 0 past the row, below every key of a value
#pragma unroll
    for (int j = 0; j < PT; ++j) ky[j] = j < n ? ky[j] : 0u;
  }
  uint32_t t1 = 0, t2 = 0;
#pragma unroll
  for (int j = 0; j < PT; ++j) {
    t2 = max(t2, min(t1, ky[j]));
    t1 = max(t1, ky[j]);
  }
  // L0: two 11-bit passes over the threads' top-2 keys, on histograms that are
  // zero on entry (the caller clears the one-pass histogram area, which they lie in)
  C4S_PHASE(20);
  C4S_PHASE(21);
  if (t1) atomicAdd(&fs.hist[0][t1 >> 21], 1u);
  if (t2) atomicAdd(&fs.hist[0][t2 >> 21], 1u);
  __syncthreads();
  // L0 lies at or below the msel-th largest of those keys, so at least msel
  // values are candidates: for k < kFastSel the k-th largest and the next one
  const uint32_t msel = min((uint32_t)kFastSel, (uint32_t)c.k + 1u);
  uint32_t L0 = 0;
  {
    uint32_t b1, ab1;
    C4S_PHASE(22);
    if (fast_pick(fs.hist[0], fs.red[0], fs.bu, msel, b1, ab1)) {
      C4S_PHASE(23);
      if (ab1 + fs.hist[0][b1] <= (uint32_t)kFastOneBin) {
        L0 = b1 << 21;   // few keys from b1 up: its floor bounds them closely enough (uniform)
      } else {
        if (t1 && (t1 >> 21) == b1) atomicAdd(&fs.hist[1][(t1 >> 10) & 2047u], 1u);
        if (t2 && (t2 >> 21) == b1) atomicAdd(&fs.hist[1][(t2 >> 10) & 2047u], 1u);
        __syncthreads();
        uint32_t b2, ab2;
        fast_pick(fs.hist[1], fs.red[1], fs.bu + 2, msel - ab1, b2, ab2);
        L0 = (b1 << 21) | (b2 << 10);
      }
    }
  }
  L0 = max(L0, 1u);   // the same values; excludes the zero keys past the row
  C4S_PHASE(11);
  // candidates in id order; the largest key under L0 bounds everything else
  uint32_t cnt = 0, below = 0;
#pragma unroll
  for (int j = 0; j < PT; ++j) {
    cnt += (ky[j] >= L0) ? 1u : 0u;
    below = max(below, ky[j] < L0 ? ky[j] : 0u);
  }
  {
    const uint32_t bm = wave_max_u32_dpp(below);   // every lane of the workgroup is here
    if (lane == 0) fs.redm[wv] = bm;
  }
  uint32_t C;
  const uint32_t pos = fast_scan(cnt, fs.red[2], C);   // its barrier also publishes redm
  C4S_PHASE(26);
  uint32_t tout = 0;
#pragma unroll
  for (int w = 0; w < kStepWaves; ++w) tout = max(tout, fs.redm[w]);
  if (tout != 0u && c.temp_on) tout = fkey(div_rcp(kfloat(tout), rt));   // the quotient is monotone in y
  // uniform; past kFastCands the rank sort costs more than the one pass
  // (a tie group of hundreds at the k-th value, which the list cannot take anyway)
  if (C > (uint32_t)kFastCands || C == 0u) return false;
  {
    // this thread's candidates as entries: z = fl(y / T) (sampling.cpp:16), the
    // id, and the candidate's position (pos + the candidates before it), which
    // is the id order: the draw's order key
    // (the set bits only: a wave takes as many rounds as its lane with the
    // most candidates, each value read again from the row in LDS)
    uint32_t cm = 0;
#pragma unroll
    for (int j = 0; j < PT; ++j) cm |= (ky[j] >= L0) ? 1u << j : 0u;
    uint32_t i = pos;
    for (uint32_t bits = cm; bits != 0u; bits &= bits - 1u, ++i) {
      const int j = __ffs(bits) - 1;
      const float yv = val[lo + j];
      fs.cand[i] = make_entry(c.temp_on ? div_rcp(yv, rt) : yv, lo + j, (int)i);
    }
  }
  static_assert(kFastCands % 16 == 0 && kFastCands <= 1024, "padding to 16 entries stays in the candidate array; "
                "positions fit the entry's rank field");
  const int C16 = __builtin_amdgcn_readfirstlane(((int)C + 15) & ~15);   // uniform: scalar loop control below
  if (t < C16 - (int)C) fs.cand[C + t] = 0ull;   // every entry is positive
  C4S_PHASE(27);
  __syncthreads();
  C4S_PHASE(12);
  // sort by rank counting (entries are distinct: their ids are); the first
  // kFastList + 1 places are kept
  uint64_t* srt = reinterpret_cast<uint64_t*>(fs.hist[0]);
  static_assert(sizeof(FastSh::hist[0]) >= (kFastList + 1) * sizeof(uint64_t), "the sorted head fits");
  const int Cs = __builtin_amdgcn_readfirstlane((int)C);
  for (int base = 0; base < Cs; base += kStepThreads) {
    const int i = base + t;
    const uint64_t mine = (i < Cs) ? fs.cand[i] : ~0ull;
    uint32_t r = 0;
    if (base + __builtin_amdgcn_readfirstlane(wv) * kWave < Cs)   // waves without an entry skip the count
      for (int j = 0; j < C16; j += 16) {   // 16 broadcast reads in flight a round
        uint64_t o[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) o[q] = fs.cand[j + q];
#pragma unroll
        for (int q = 0; q < 16; ++q) r += (o[q] > mine) ? 1u : 0u;
      }
    if (i < Cs && r < (uint32_t)(kFastList + 1)) srt[r] = mine;
  }
  __syncthreads();
  C4S_PHASE(13);
  if (wv == 0) {
    // the list: the leading entries above the bound (a prefix), at most kFastList
    const int nl = min((int)C, kFastList + 1);
    const bool a0 = lane < nl, a1 = lane + kWave < nl;
    uint64_t e0 = srt[a0 ? lane : 0], e1 = srt[a1 ? lane + kWave : 0];
    const uint64_t e2 = srt[nl > 2 * kWave ? 2 * kWave : 0];
    const int n_all = __popcll(__ballot(a0 && ent_key(e0) > tout)) + __popcll(__ballot(a1 && ent_key(e1) > tout)) +
                      ((nl > 2 * kWave && ent_key(e2) > tout) ? 1 : 0);
    const int nlist = min(n_all, kFastList);
    if (n_all > kFastList) tout = max(tout, ent_key(e2));
    const float ztop = kfloat(ent_key(srt[0]));   // C >= 1
    // the draw starts its maximum at -1e30 (text2semantic.cpp:150): below it the one pass decides
    bool ok = nlist > 0 && ztop >= -1e30f;
    C4S_PHASE(24);
    if (ok) {
      // each entry keeps its candidate position as its id-order key (8 bits)
      e0 = lane < nlist ? e0 : 0ull;
      e1 = lane + kWave < nlist ? e1 : 0ull;
      SumHdr h{};
      h.n = nlist;
      h.tout = tout;
      h.flags = 0u;
      uint64_t r = io.rng ? *io.rng : 0ull;
      StepOut o{0, 0u, 0u, 0u, 0u};
      static_assert(kFastCands <= 256, "candidate positions in 8 bits");
      ok = list_step<8, true>(h, e0, e1, 0.0f, 0.0f, c, V, NoHit{}, r, fs.cs, o);
      C4S_PHASE(25);
      if (ok && lane == 0) step_out(io, V, o.tok, r, true, 1u | 2u | 4u | 16u | 32u, 0u, o.dex, o.kept);
    }
    if (lane == 0) fs.bu[4] = ok ? 1u : 0u;
  }
  __syncthreads();
  C4S_PHASE(15);
  return fs.bu[4] != 0u;
}

// The one pass of a sampled row, specialised by the row's kind (top_k on; top_p
// with p < 1; p >= 1, a dense draw) so that the per-value loops carry no tests
// of the kind. Returns true when the row is finished; false leaves the row to
// the multi-pass chain (nothing written but the work area).
constexpr int kKindTopK = 0, kKindTopP = 1, kKindDense = 2;

template <int PT, int kKind>
__device__ __forceinline__ bool sampled_step(const StepIO& io, const RowCfg& c, const float (&y)[PT], int lo, int n,
                                             float* val, uint32_t* hc, unsigned long long* hm, uint64_t* sbuf,
                                             uint64_t* list, float* em, StepSh& ss, StepRowSh& rs) {
  const int t = threadIdx.x, lane = lane_id(), w = wave_id();
  const float ninf = neg_inf();
  // ---- sampled rows: temperature (sampling.cpp:14-17) and the maximum ----
  float z[PT];
  const double rt = 1.0 / (double)c.temp;   // used only when the temperature applies
#pragma unroll
  for (int j = 0; j < PT; ++j) z[j] = c.temp_on ? div_rcp(y[j], rt) : y[j];
  if (n < PT) {   // the last threads: the padding past the row stays -inf whatever the temperature
#pragma unroll
    for (int j = 0; j < PT; ++j) z[j] = j < n ? z[j] : ninf;
  }
  {
    float lm = ninf;
#pragma unroll
    for (int j = 0; j < PT; ++j) lm = fmaxf(lm, z[j]);
    lm = wave_max_dpp(lm);
    if (lane == 0) ss.wmax[w] = lm;
  }
  C4S_PHASE(2);
  __syncthreads();
  C4S_PHASE(3);
  float m = ninf;
#pragma unroll
  for (int i = 0; i < kStepWaves; ++i) m = fmaxf(m, ss.wmax[i]);
  const double thr = 1.0 - (double)c.p;   // sampling.cpp:64 removes while cum <= 1 - p
  constexpr bool topk = kKind == kKindTopK;
  constexpr bool dense = kKind == kKindDense;
  // The draw's maximum starts from -1e30f (text2semantic.cpp:150): below it, or
  // for an all -inf row, or with p <= 0, the multi-pass chain decides.
  bool one_pass = !(m < -1e30f) && thr < 1.0;
  int verdict = 0;
  bool tp_exact = false;
  if (one_pass) {
    // fp32 masses; the dense rows' kept set; the histogram (counts for top_k,
    // masses for top_p). Sums per thread in fp32: bound (2^-20 + PT 2^-24)
    // relative (terms and summation) + 2^-125 a term (underflow).
    // Every value goes through the same instructions (no branch a value): z is
    // -inf past the thread's ids, and an entry of the unbounded last bucket
    // adds to a word of its own thread instead (in the boundary list, unused
    // until the compaction): on a wide row most values lie there, and lanes
    // adding to one LDS word take turns.
    // The error bound counts every id of the thread (at least its finite ones).
    float s32 = 0.0f;
    uint32_t flags = 0, kc = 0;
#pragma unroll
    for (int j = 0; j < PT; ++j) {
      const float tt = z[j] - m;
      if (topk) {
        const int b = bucket_of_diff(-tt);   // the last bucket for -inf
        atomicAdd(b < kNB - 1 ? &hc[w * kNB + b] : reinterpret_cast<uint32_t*>(list) + t, 1u);
      } else {
        // 0 for -inf without a select: below about -150 the fp32 exp2 is 0
        // and mass32 returns +0, so clamping at -1000 changes no mass
        float ej = mass32(fmaxf(tt, -1000.0f));
        if (j < n) em[lo + j] = ej;   // read again by the kept sums and the draw
        if (dense) {
          // p == 1 removes the zero-mass positions: exp((double)tt) == 0 below
          // about -745.13; near that, and for subnormal kept masses, the chain decides
          const bool fin = z[j] != ninf;
          const bool kp = fin && (thr < 0.0 || tt > -745.0f);
          if (fin && ((thr == 0.0 && tt <= -745.0f && tt >= -745.25f) || (kp && tt < -690.0f))) flags = 1u;
          ej = kp ? ej : 0.0f;
          kc += kp ? 1u : 0u;
        } else {
          // 2^-31 fixed point, truncated (ej <= 1)
          const int b = bucket_of_diff(-tt);
          const uint32_t q = (uint32_t)(ej * 0x1p31f);
          atomicAdd(b < kNB - 1 ? &hm[w * kNB + b] : reinterpret_cast<unsigned long long*>(list) + t,
                    (unsigned long long)q + kHistOne);
        }
        s32 += ej;
      }
    }
    const double s = (double)s32;
    const double er = s * (0x1p-20 + PT * 0x1p-24) + (double)max(n, 0) * 0x1p-125;
    C4S_PHASE(4);
    const Scan2 sc = block_scan2(s, er, kc | (flags << 16), ss.wa, ss.wb, ss.wu);
    C4S_PHASE(5);
    const uint32_t n_pos = sc.utot & 0xFFFFu;   // dense rows: kept ids with a finite value
    // p == 1 with min_keep above the positive-mass count keeps zero-mass values
    // unmasked (sampling.cpp:67-68): the multi-pass chain handles that
    if ((sc.utot >> 16) || (dense && thr == 0.0 && n_pos < (uint32_t)max(0, c.min_keep))) {
      one_pass = false;
    } else if (dense) {
      // nothing to cut: the draw over the fp32 masses scanned above
      const KeptRule kr{true, thr < 0.0, 0ull};
      if (io.masked)
#pragma unroll
        for (int j = 0; j < PT; ++j)
          if (j < n) io.masked[lo + j] = (thr < 0.0 || (z[j] != ninf && z[j] - m > -745.0f)) ? z[j] : ninf;
      C4S_PHASE(10);
      draw_finish<PT, true>(io, c, kr, z, lo, n, m, sc, n_pos, 1u | 4u | 16u, 0u, ss, rs, em, list);
      C4S_PHASE(15);
      return true;
    } else {
      const double S = sc.tot, errS = sc.tot2;
      // boundary buckets: threads 0..255 merge one bucket each over the waves,
      // then wave 0 scans them (lane l holds buckets 4l .. 4l+3)
      uint32_t* bcnt = reinterpret_cast<uint32_t*>(sbuf);           // sort buffers are free here
      double* bmass = reinterpret_cast<double*>(sbuf) + kNB;
      if (t < kNB) {
        uint32_t cn = 0;
        unsigned long long ms = 0ull;
#pragma unroll
        for (int i = 0; i < kStepWaves; ++i) {
          const unsigned long long h = hm[i * kNB + t];
          cn += hc[i * kNB + t] + (uint32_t)(h >> 48);
          ms += h & (kHistOne - 1ull);
        }
        bcnt[t] = cn;
        bmass[t] = (double)ms * 0x1p-31;
      }
      __syncthreads();
      const double B = S - thr * S;   // the mass the kept entries hold
      const double Blo = B * (1.0 - 1e-3) - errS, Bhi = B * (1.0 + 1e-3) + errS;
      if (w == 0) {
        const Boundary bd = boundary_scan(bcnt, bmass, topk, (uint32_t)c.k, Blo, Bhi, 0u, 0.0);
        if (lane == 0) {
          ss.bsel[0] = bd.lo;
          ss.bsel[1] = bd.hi;
          ss.bsel[2] = (int)bd.above;
          ss.thru = bd.thru;
          ss.mab = bd.mabove;
          ss.mabx = topk ? 0.0 : bd.mabove;   // top_k: nothing lies above X
          ss.nabx = topk ? 0u : bd.above;
          ss.nx = 0u;
        }
      }
      __syncthreads();
      C4S_PHASE(6);
      const int blo = ss.bsel[0], bhi = ss.bsel[1];
      // the sub-window of the boundary buckets (all of them unless refined)
      int slo = 0, shi = kNB - 1, lo2 = 0;
      float sc2 = 0.0f;
      bool refine = false;
      if (blo >= 0 && bhi >= 0) {
        // More boundary entries than one sort takes (flat rows): histogram the
        // boundary buckets again, kNB sub-buckets over them (top_k: over the
        // k-th entry's bucket), and keep the sub-buckets where the boundary
        // falls. Not for the unbounded last bucket.
        const uint32_t nest = topk ? ss.thru : ss.thru - (uint32_t)ss.bsel[2];
        refine = nest > (uint32_t)kSortCap && bhi < kNB - 1;
        if (refine) {
          lo2 = topk ? bhi : blo;
          sc2 = (float)kNB / (float)(bhi + 1 - lo2);
          for (int i = t; i < (int)(3 * kHistBytes / 4); i += kStepThreads) hc[i] = 0u;
          __syncthreads();
          // Per value: no branch, and the fp32 mass the first pass cached (the
          // same mass32), read unconditionally (index clamped). -inf and the
          // padding past the thread's ids lie in the last bucket, never in the
          // window (bhi < kNB - 1); entries outside it add to a word of the
          // thread's own (the boundary list, unused until the compaction).
#pragma unroll
          for (int j = 0; j < PT; ++j) {
            const int b = bucket_of(z[j], m);
            const bool inw = ((int)(b >= lo2) & (int)(b <= bhi)) != 0;
            const int sb = sub_bucket_of(z[j], m, lo2, sc2);
            if (topk) {
              atomicAdd(inw ? &hc[w * kNB + sb] : reinterpret_cast<uint32_t*>(list) + t, 1u);
            } else {
              const float ec = em[min(lo + j, c.V - 1)];
              atomicAdd(inw ? &hm[w * kNB + sb] : reinterpret_cast<unsigned long long*>(list) + t,
                        (unsigned long long)(uint32_t)(ec * 0x1p31f) + kHistOne);
            }
          }
          __syncthreads();
          if (t < kNB) {
            uint32_t cn = 0;
            unsigned long long ms = 0ull;
#pragma unroll
            for (int i = 0; i < kStepWaves; ++i) {
              const unsigned long long h = hm[i * kNB + t];
              cn += hc[i * kNB + t] + (uint32_t)(h >> 48);
              ms += h & (kHistOne - 1ull);
            }
            bcnt[t] = cn;
            bmass[t] = (double)ms * 0x1p-31;
          }
          __syncthreads();
          if (w == 0) {
            const Boundary b2 = boundary_scan(bcnt, bmass, topk, (uint32_t)c.k, Blo, Bhi, (uint32_t)ss.bsel[2],
                                              ss.mab);
            if (lane == 0) {
              ss.sub[0] = topk ? 0 : b2.lo;   // top_k: every entry above the k-th stays in the sort
              ss.sub[1] = b2.hi;
              if (!topk) {
                ss.mabx = b2.mabove;
                ss.nabx = b2.above;
              }
            }
          }
          __syncthreads();
          slo = ss.sub[0];
          shi = ss.sub[1];
        }
      }
      C4S_PHASE(16);
      C4S_PHASE_VAL(21, refine ? 1 : 0);
      if (blo < 0 || bhi < 0 || slo < 0 || shi < 0) {
        one_pass = false;
      } else {
        // X: the entries to sort. top_k: every entry up to the k-th value's
        // (sub-)bucket (the survivors then are a prefix of X). top_p: the
        // boundary (sub-)buckets; every entry above them is kept, every entry
        // below removed. side(): -1 above X, 0 in X, 1 below (monotone in z).
        const int xlo = topk ? 0 : blo, xhi = bhi;
        const SideRule sr{m, sc2, xlo, xhi, lo2, slo, shi, refine};
        auto side = [&](float zj) { return sr.side(zj); };
        // X's entries go to `list`, each wave taking one block of slots with
        // one atomic (slot order is arbitrary: the sort orders them)
        static_assert(PT < 32, "a thread's X entries as one bit mask");
        uint32_t xm = 0;   // this thread's X entries (its ids only: the -inf padding may lie in the last bucket)
        if (!refine) {
          // uniform: X is whole buckets xlo .. xhi. With q = (m - z) 4 (exact:
          // a power of two; q >= 0, +inf for -inf) bucket_of is trunc(q) below
          // 255, else 255: b >= xlo iff !(q < xlo) (NaN in the last bucket), and
          // b <= xhi iff q < xhi + 1 unless xhi is the last bucket
          const float qlo = (float)xlo, qhi = xhi >= kNB - 1 ? __builtin_inff() : (float)(xhi + 1);
          const bool last = xhi >= kNB - 1;
#pragma unroll
          for (int j = 0; j < PT; ++j) {
            const float q = (m - z[j]) * kBucketScale;
            xm |= ((int)!(q < qlo) & (int)(last || q < qhi)) ? 1u << j : 0u;
          }
        } else {
#pragma unroll
          for (int j = 0; j < PT; ++j) xm |= (side(z[j]) == 0) ? 1u << j : 0u;
        }
        xm &= (1u << n) - 1u;
        {
          const uint32_t cx = (uint32_t)__popc(xm);
          const uint32_t inc = wave_scan_u32(cx);
          uint32_t wb = 0;
          if (lane == kWave - 1 && inc > 0u) wb = atomicAdd(&ss.nx, inc);
          const uint32_t base = readlane_u32(wb, kWave - 1) + inc - cx;
          // the set bits only, in id order (a wave takes as many rounds as its
          // lane with the most X entries: usually one or two), each value read
          // again from the row in LDS (z = fl(y / T), the same division)
          uint32_t slot = base;
          for (uint32_t bits = xm; bits != 0u; bits &= bits - 1u, ++slot) {
            const int j = __ffs(bits) - 1;
            const float yv = val[lo + j];
            if (slot < (uint32_t)kSortCap) list[slot] = key64(c.temp_on ? div_rcp(yv, rt) : yv, lo + j);
          }
        }
        C4S_PHASE(17);
        __syncthreads();
        C4S_PHASE(7);
        const int nX = (int)ss.nx;
        C4S_PHASE_VAL(20, nX);
        // The mass above X and its count, from the histogram: the fixed-point
        // masses of the (sub-)buckets above X. Against the exact masses each
        // entry is off by its fp32 mass error (2^-20 relative + 2^-125) and
        // the truncation (below 2^-31); the bucket sums are exact integers and
        // the scan's double prefix adds a few 2^-53 relative.
        const double Ma = ss.mabx;
        const uint32_t n_above = ss.nabx;
        const double eMa = Ma * (0x1p-20 + 0x1p-40) + (double)n_above * 0x1p-30;
        if (nX > kSortCap) {
          // more boundary entries than one sort takes: one_pass only if they
          // all hold one value (ties), which needs no sort
          verdict = tie_cut<PT>(rs.cfg, val, lo, n, sr, nX, thr, S, errS, Ma, eMa, n_above, ss);
          C4S_PHASE(28);
          tp_exact = verdict == 3;
          if (verdict != 1 && verdict != 3) one_pass = false;
          if (verdict == 4 && t == 0) rs.tp_exact_first = 1u;
        } else {
          int P2 = 1;
          while (P2 < nX) P2 <<= 1;
          const bool block = P2 > kWave;
          uint64_t v = 0ull;
          if (block) {
            // up to 256 entries by rank counting (two to four threads a key,
            // two barriers); more by the bitonic network (six barriers)
            if (nX <= 128) {
              v = rank_sort_desc<128>(list, nX, reinterpret_cast<uint32_t*>(sbuf));
            } else if (nX <= 256) {
              v = rank_sort_desc<256>(list, nX, reinterpret_cast<uint32_t*>(sbuf));
            } else {
              v = t < nX ? list[t] : 0ull;
              v = sort_desc_block(v, P2, sbuf);
              if (t < nX) list[t] = v;
              __syncthreads();
            }
            C4S_PHASE(8);
            if (t == 0) ss.zx = key_value(v);   // X's largest value (read after the barriers below)
            decide_cut<true>(rs.cfg, v, nX, m, thr, S, errS, Ma, eMa, n_above, list, ss);
          } else if (w == 0) {
            v = lane < nX ? list[lane] : 0ull;
            v = sort_desc_wave(v, P2);
            C4S_PHASE(8);
            if (t == 0) ss.zx = key_value(v);
            decide_cut<false>(rs.cfg, v, nX, m, thr, S, errS, Ma, eMa, n_above, list, ss);
          }
          __syncthreads();
          verdict = ss.verdict;
          if (verdict == 2) {
            // decide again with every mass in double (S and the mass above the boundary)
            tp_exact = true;
            // every value through the same instructions, so that the exps
            // interleave: z is -inf past the thread's ids and exp(-inf) = 0.
            // side() is monotone in z and equal values share a side, so the
            // entries above X are exactly those above X's largest value.
            double se = 0.0, sa = 0.0;
            if (nX > 0) {
              const float zx = ss.zx;
#pragma unroll
              for (int j = 0; j < PT; ++j) {
                const double ed = exp((double)(z[j] - m));
                se += ed;
                sa += z[j] > zx ? ed : 0.0;
              }
            } else {
#pragma unroll
              for (int j = 0; j < PT; ++j) {
                const double ed = exp((double)(z[j] - m));
                se += ed;
                sa += side(z[j]) < 0 ? ed : 0.0;
              }
            }
            se = wave_sum_dpp(se);
            sa = wave_sum_dpp(sa);
            if (lane == 0) { ss.wc[w] = se; ss.wd[w] = sa; }
            __syncthreads();
            double Se = 0.0, Mae = 0.0;
#pragma unroll
            for (int i = 0; i < kStepWaves; ++i) { Se += ss.wc[i]; Mae += ss.wd[i]; }
            if (block) decide_cut<true>(rs.cfg, v, nX, m, thr, Se, 0.0, Mae, 0.0, n_above, list, ss);
            else if (w == 0) decide_cut<false>(rs.cfg, v, nX, m, thr, Se, 0.0, Mae, 0.0, n_above, list, ss);
            __syncthreads();
            verdict = ss.verdict;
          }
          C4S_PHASE(9);
          C4S_PHASE_VAL(22, verdict);
          if (verdict != 1) one_pass = false;
          if (verdict == 4 && t == 0) rs.tp_exact_first = 1u;
        }
      }
    }
  }
  if (one_pass) {
    // the draw over the kept set: key >= the last kept key
    const uint64_t kthr = ss.kthr;
    const KeptRule kr{false, false, kthr};
    float ks32 = 0.0f;
    uint32_t kc = 0, flags = 0;
    float ecs[PT];   // top_p: the masses cached by the histogram pass (0 for -inf)
    if (!topk) read_row(em, lo, n, c.V, ecs);
#pragma unroll
    for (int j = 0; j < PT; ++j) {   // z is -inf past the thread's ids: never kept with a mass
      bool kp;
      float ej;
      if (topk) {
        ej = kept_mass32(kr, z[j], m, lo + j, kp);
      } else {
        const float ec = ecs[j];
        kp = ((int)(z[j] != ninf) & (int)kept_in(kr, z[j], m, lo + j)) != 0;   // z is -inf past the thread's ids
        ej = kp ? ec : 0.0f;
      }
      const bool kf = kp && z[j] != ninf;
      kc += kf ? 1u : 0u;
      ks32 += ej;
    }
    // subnormal kept masses (libm implementations may disagree): the smallest
    // kept value is the last kept key's (a -inf there also sends the row on)
    flags = (t == 0 && key_value(kthr) - m < -690.0f) ? 1u : 0u;
    if (io.masked)
#pragma unroll
      for (int j = 0; j < PT; ++j) {
        bool kp;
        kept_mass32(kr, z[j], m, lo + j, kp);
        if (j < n) io.masked[lo + j] = kp ? z[j] : ninf;
      }
    C4S_PHASE(27);
    const double ks = (double)ks32;
    const double ek = ks * (0x1p-20 + PT * 0x1p-24) + (double)kc * 0x1p-125;
    const Scan2 ds = block_scan2(ks, ek, kc | (flags << 16), ss.wa, ss.wb, ss.wu);
    C4S_PHASE(10);
    if ((ds.utot >> 16) == 0u) {
      draw_finish<PT, !topk>(io, c, kr, z, lo, n, m, ds, ds.utot & 0xFFFFu, 1u | (topk ? 2u : 0u) | 4u | 16u,
                             tp_exact ? 1u : 0u, ss, rs, em, list);
      C4S_PHASE(15);
      return true;
    }
  }
  return false;
}

}  // namespace
}  // namespace c4s
