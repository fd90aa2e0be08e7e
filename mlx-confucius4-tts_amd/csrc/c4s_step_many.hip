// The one-pass step (k_rows_step, sampled_step) in the form for many more rows
// than CUs: two workgroups share a CU.
//
// The step is a chain of short barrier-separated phases; one workgroup of eight
// waves leaves its CU idle most of the time, and with 228 registers a thread
// and 108 KB of LDS it is alone there, so 1000 rows take four rounds. This form
// fits 128 registers and 76 KB at 8194 ids: the values are read again from the
// row in LDS by every pass, kManyU of a thread's ids at a time, instead of held
// in registers over the calls (the unrolled passes at 128 registers spilled 44
// of them: 46 us for 1000 nucleus rows against 47.7 for the other form and 38.4
// rolled), and the fp32 masses are taken again instead of kept in LDS. One
// workgroup alone takes longer this way, so kManyRows is where the line lies.
// 1000 rows of 8194 ids, microseconds a call (other form / this): assorted
// 44.6 / 34.8, pipeline defaults 35.7 / 23.4, nucleus bf16 47.7 / 38.4,
// greedy 24.9 / 16.2, 1024 rows of ties 138.4 / 105.4.
//
// The decisions, margins and fallbacks are sampled_step's.

#include "c4s_onepass.hpp"

namespace c4s {
namespace {

constexpr int kManyU = 6;   // a thread's ids read together
// Up to two rounds of one workgroup a CU, and a little over, a row that falls to
// its exact replay sets the call, and it takes longer beside another: bf16 rows
// with ties, 309 rows of 5132 ids 143 / 184 us and of 2500 ids 93 / 108, 513 rows
// of 5132 ids 181 / 187. Above, the rounds saved are worth more: 700 rows of 5132
// ids 263 / 203, of 2500 ids 164 / 123, of 8194 ids 108 / 90.
constexpr int kManyRows = 576;

// draw_finish, with the kept masses taken again from the row in LDS.
__device__ __forceinline__ void draw_finish_many(const StepIO& io, const RowCfg& c, const KeptRule& kr, int lo, int n,
                                                 float m, const Scan2& ds, uint32_t n_kept, uint32_t st_path,
                                                 uint32_t st_exact, StepSh& ss, const StepRowSh& rs, uint64_t* kl,
                                                 const float* val) {
  const double rt = 1.0 / (double)c.temp;
  auto z_at = [&](int id) __attribute__((always_inline)) { return c.temp_on ? div_rcp(val[id], rt) : val[id]; };
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
  const uint64_t obw = __ballot(owner);
  if (obw) {
    // the owner's wave: lane j takes the owner's id lo + j and its kept fp32
    // mass (independent loads and tests, one a lane), the running sums in id
    // order by a wave scan in double from the owner's exclusive prefix (its
    // rounding, about 2^-53 relative a step, lies far inside the margin), then
    // the first kept id whose sum reaches r and the sums on both sides of it
    const int ol = __ffsll((unsigned long long)obw) - 1, l = lane_id();
    const int lo_o = (int)readlane_u32((uint32_t)lo, ol);
    const int n_o = (int)readlane_u32((uint32_t)n, ol);
    const float zr = z_at(min(lo_o + l, c.V - 1)), zl = l < n_o ? zr : neg_inf();
    const double ex_o = readlane_f64(ds.ex, ol);
    bool kp;   // lanes past the owner's ids hold -inf: not kept
    const float el = kept_mass32(kr, zl, m, lo_o + l, kp);
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
  if (!__syncthreads_or(owner && !certain)) {
    if (owner) step_out(io, c.V, found, st2, true, st_path, st_exact, 0u, n_kept);
    return;
  }
  // the kept masses in double. The kept test is the one pass's (kept_in): a
  // dense row reaches this draw only without values whose double mass lies
  // near underflow, so `z - m > -745` there is exactly `exp((double)(z - m)) > 0`.
  if (n_kept <= (uint32_t)kWave) {
    // at most 64 kept ids: in id order (thread order, then the thread's own)
    // to one wave, which draws on them in double and replays the sums
    // sequentially when that is too close (lane_draw)
    uint32_t at = ds.uex;
#pragma unroll 1
    for (int j = 0; j < n; ++j) {
      const float zj = z_at(lo + j);
      if (zj != neg_inf() && kept_in(kr, zj, m, lo + j))
        kl[at++] = ((uint64_t)__float_as_uint(zj) << 32) | (uint32_t)(lo + j);
    }
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
#pragma unroll 1
  for (int j = 0; j < n; ++j) {
    const float zj = z_at(lo + j);
    if (zj != neg_inf() && kept_in(kr, zj, m, lo + j)) dk += exp((double)(zj - m));
  }
  const Scan2 d2 = block_scan2(dk, 0.0, 0u, ss.wa, ss.wb, ss.wu);
  const double r2 = u * d2.tot;
  const double m2 = 2.0 * rel_eps(c.V) * d2.tot;
  const bool own2 = (d2.ex < r2 && r2 <= d2.in) || (t == kStepThreads - 1 && r2 > d2.in);
  found = -1;
  certain = false;
  const uint64_t ob = __ballot(own2);
  if (ob) {   // the owner's wave: lane j takes the owner's id lo + j, the prefix by a wave scan
    const int ol = __ffsll((unsigned long long)ob) - 1, l = lane_id();
    const int lo_o = readlane_u32((uint32_t)lo, ol), n_o = readlane_u32((uint32_t)n, ol);
    const float zl = z_at(min(lo_o + l, c.V - 1));
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
  if (!__syncthreads_or(own2 && !certain)) {
    if (own2) step_out(io, c.V, found, st2, true, st_path, st_exact, 1u, n_kept);
    return;
  }
  if (wave_id() == 0) {   // the reference's sequential sums, one wave
    const int tk = draw_replay(rs.io, rs.cfg, kr, m, u);
    if (lane_id() == 0) step_out(io, c.V, tk, st2, true, st_path, st_exact, 2u, n_kept);
  }
}

// sampled_step; PT bounds the ids a thread owns.
template <int PT, int kKind>
__device__ __forceinline__ bool sampled_step_many(const StepIO& io, const RowCfg& c, int lo, int n, float* val, uint32_t* hc,
                                                  unsigned long long* hm, uint64_t* sbuf, uint64_t* list, StepSh& ss,
                                                  StepRowSh& rs) {
  const int t = threadIdx.x, lane = lane_id(), w = wave_id();
  const float ninf = neg_inf();
  // ---- sampled rows: temperature (sampling.cpp:14-17) and the maximum ----
  const double rt = 1.0 / (double)c.temp;   // used only when the temperature applies
  // fn(j, z) for the thread's ids in order, kManyU of them read together; z is
  // -inf past the ids
  auto each = [&](auto&& fn) __attribute__((always_inline)) {
#pragma unroll 1
    for (int j0 = 0; j0 < n; j0 += kManyU) {
      float yv[kManyU];
#pragma unroll
      for (int u = 0; u < kManyU; ++u) yv[u] = val[min(lo + j0 + u, c.V - 1)];
#pragma unroll
      for (int u = 0; u < kManyU; ++u) fn(j0 + u, j0 + u < n ? (c.temp_on ? div_rcp(yv[u], rt) : yv[u]) : ninf);
    }
  };
  {
    float lm = ninf;
    each([&](int, float zj) __attribute__((always_inline)) { lm = fmaxf(lm, zj); });
    lm = wave_max_dpp(lm);
    if (lane == 0) ss.wmax[w] = lm;
  }
  __syncthreads();
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
    each([&](int j, float zj) __attribute__((always_inline)) {
      const float tt = zj - m;
      if (topk) {
        const int b = bucket_of_diff(-tt);   // the last bucket for -inf
        atomicAdd(b < kNB - 1 ? &hc[w * kNB + b] : reinterpret_cast<uint32_t*>(list) + t, 1u);
      } else {
        // 0 for -inf without a select: below about -150 the fp32 exp2 is 0
        // and mass32 returns +0, so clamping at -1000 changes no mass
        float ej = mass32(fmaxf(tt, -1000.0f));
        if (dense) {
          // p == 1 removes the zero-mass positions: exp((double)tt) == 0 below
          // about -745.13; near that, and for subnormal kept masses, the chain decides
          const bool fin = zj != ninf;
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
    });
    const double s = (double)s32;
    const double er = s * (0x1p-20 + PT * 0x1p-24) + (double)max(n, 0) * 0x1p-125;
    const Scan2 sc = block_scan2(s, er, kc | (flags << 16), ss.wa, ss.wb, ss.wu);
    const uint32_t n_pos = sc.utot & 0xFFFFu;   // dense rows: kept ids with a finite value
    // p == 1 with min_keep above the positive-mass count keeps zero-mass values
    // unmasked (sampling.cpp:67-68): the multi-pass chain handles that
    if ((sc.utot >> 16) || (dense && thr == 0.0 && n_pos < (uint32_t)max(0, c.min_keep))) {
      one_pass = false;
    } else if (dense) {
      // nothing to cut: the draw over the fp32 masses scanned above
      const KeptRule kr{true, thr < 0.0, 0ull};
      if (io.masked)
        each([&](int j, float zj) __attribute__((always_inline)) {
          if (j < n) io.masked[lo + j] = (thr < 0.0 || (zj != ninf && zj - m > -745.0f)) ? zj : ninf;
        });
      draw_finish_many(io, c, kr, lo, n, m, sc, n_pos, 1u | 4u | 16u, 0u, ss, rs, list, val);
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
          each([&](int j, float zj) __attribute__((always_inline)) {
            const int b = bucket_of(zj, m);
            const bool inw = ((int)(b >= lo2) & (int)(b <= bhi)) != 0;
            const int sb = sub_bucket_of(zj, m, lo2, sc2);
            if (topk) {
              atomicAdd(inw ? &hc[w * kNB + sb] : reinterpret_cast<uint32_t*>(list) + t, 1u);
            } else {
              const float ec = mass32(fmaxf(zj - m, -1000.0f));
              atomicAdd(inw ? &hm[w * kNB + sb] : reinterpret_cast<unsigned long long*>(list) + t,
                        (unsigned long long)(uint32_t)(ec * 0x1p31f) + kHistOne);
            }
          });
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
          each([&](int j, float zj) __attribute__((always_inline)) {
            const float q = (m - zj) * kBucketScale;
            xm |= ((int)!(q < qlo) & (int)(last || q < qhi)) ? 1u << j : 0u;
          });
        } else {
          each([&](int j, float zj) __attribute__((always_inline)) { xm |= (side(zj) == 0) ? 1u << j : 0u; });
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
        __syncthreads();
        const int nX = (int)ss.nx;
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
            if (t == 0) ss.zx = key_value(v);   // X's largest value (read after the barriers below)
            decide_cut<true>(rs.cfg, v, nX, m, thr, S, errS, Ma, eMa, n_above, list, ss);
          } else if (w == 0) {
            v = lane < nX ? list[lane] : 0ull;
            v = sort_desc_wave(v, P2);
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
            const float zx = ss.zx;
            each([&](int, float zj) __attribute__((always_inline)) {
              const double ed = exp((double)(zj - m));
              se += ed;
              sa += (nX > 0 ? zj > zx : side(zj) < 0) ? ed : 0.0;
            });
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
    each([&](int j, float zj) __attribute__((always_inline)) {   // z is -inf past the thread's ids: never kept with a mass
      bool kp;
      const float ej = kept_mass32(kr, zj, m, lo + j, kp);
      const bool kf = kp && zj != ninf;
      kc += kf ? 1u : 0u;
      ks32 += ej;
    });
    // subnormal kept masses (libm implementations may disagree): the smallest
    // kept value is the last kept key's (a -inf there also sends the row on)
    flags = (t == 0 && key_value(kthr) - m < -690.0f) ? 1u : 0u;
    if (io.masked)
      each([&](int j, float zj) __attribute__((always_inline)) {
        bool kp;
        kept_mass32(kr, zj, m, lo + j, kp);
        if (j < n) io.masked[lo + j] = kp ? zj : ninf;
      });
    const double ks = (double)ks32;
    const double ek = ks * (0x1p-20 + PT * 0x1p-24) + (double)kc * 0x1p-125;
    const Scan2 ds = block_scan2(ks, ek, kc | (flags << 16), ss.wa, ss.wb, ss.wu);
    if ((ds.utot >> 16) == 0u) {
      draw_finish_many(io, c, kr, lo, n, m, ds, ds.utot & 0xFFFFu, 1u | (topk ? 2u : 0u) | 4u | 16u, tp_exact ? 1u : 0u, ss,
                       rs, list, val);
      return true;
    }
  }
  return false;
}

// The chain on a row that one pass leaves: its LDS has no room for the chain's
// masses, so the row is read again from HBM on every pass, with LDS for the exact
// top_p's keys alone (rare). Calls of nothing but such rows, 8194 ids, 600 / 1000
// rows (k_rows_step with its chain in LDS): top_p 0 411 / 490 us (517 / 695), with
// min_keep 0 as well 740 / 1076 (1190 / 2032), values below the draw's floor 953 /
// 1040 (1367 / 1826), bf16 top_k 30 and top_p 0 239 / 282 (215 / 288), bf16 top_p 1
// with min_keep above the masses that count 153 / 184 (138 / 189).
__device__ __forceinline__ void chain_fallback_global(const StepIO& io, const RowCfg& c, unsigned char* lds, uint32_t bytes,
                                                   StepScratch& sh, bool tp_exact_first) {
  GlobalRow src;
  src.xf = io.xf;
  src.xb = io.xb;
  src.V = c.V;
  src.bitmap = io.bitmap ? io.bitmap : io.hbits;
  src.pen_on = c.pen_on;
  src.pen = c.pen;
  src.temp_on = false;
  src.temp = 1.0f;
  src.thr_key = 0u;
  src.topk_on = false;
  src.sortbuf = reinterpret_cast<uint32_t*>(lds);
  src.sortcap = bytes;
  uint64_t rng = *io.rng;
  const int tok = run_chain<kStepWaves, GlobalRow, true>(src, sh, c, rng, io.masked, sh.step_stats, tp_exact_first);
  if (threadIdx.x == 0) {
    const uint32_t* sp = sh.step_stats;
    step_out(io, c.V, tok, rng, true, sp[0], sp[1], sp[2], sp[3]);
  }
}

// k_rows_step for many more rows than CUs.
template <int PT>
__global__ __launch_bounds__(kStepThreads) __attribute__((amdgpu_waves_per_eu(4))) void k_rows_step_many(RowsArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ StepScratch sh;
  __shared__ StepSh ss;
  __shared__ StepRowSh rs;
  const int row = blockIdx.x;
  const int V = a.vocab;
  const int t = threadIdx.x;
  // Every read that depends on no other goes out first: the row's flags and
  // parameters, its history offsets, then the row itself (fp32 rows into
  // registers here, stored to LDS below); nothing waits on them before the
  // row's loads are in flight, so the step pays one memory round trip up front
  // instead of one per dependent read.
  const int64_t roff = (int64_t)row * a.ld;
  const float* xf_row = a.dtype == 0 ? static_cast<const float*>(a.logits) + roff : nullptr;
  StepFetch f;
  if (xf_row) step_fetch(xf_row, V, f);
  const bool act = a.row_active ? flag_byte(a.row_active, row) : true;
  const bool sample = a.do_sample ? flag_byte(a.do_sample, row) : true;
  const float pv = a.pen ? a.pen[row] : 1.0f, tv = a.temp ? a.temp[row] : 1.0f;
  const int32_t kv = a.top_k ? a.top_k[row] : 0, mv = a.min_keep ? a.min_keep[row] : 1;
  const float ppv = a.top_p ? a.top_p[row] : 1.0f;
  const bool csr_arg = a.hist_off && !a.hist_bits;
  int64_t h0 = 0, h1 = 0;
  if (csr_arg) {
    h0 = a.hist_off[row];
    h1 = a.hist_off[row + 1];
  }
  if (!act) {
    if (t == 0) a.out_tok[row] = -1;
    return;
  }
  const RowCfg c = make_cfg_vals(0u, V, pv, tv, kv, ppv, mv, sample);
  C4S_PHASE(0);
  unsigned char* work = smem;
  float* vbuf = reinterpret_cast<float*>(smem + kStepWorkBytes);
  uint32_t* bitmap = reinterpret_cast<uint32_t*>(vbuf + vpad(V) + 4);
  uint32_t* hc = reinterpret_cast<uint32_t*>(work);   // [waves][kNB] bucket counts
  unsigned long long* hm = reinterpret_cast<unsigned long long*>(work + kHistBytes);   // [waves][kNB] masses, 2^-32 units
  uint64_t* sbuf = reinterpret_cast<uint64_t*>(work + 3 * kHistBytes);
  uint64_t* list = sbuf + 2 * kSortCap;
  const int P = odd_chunk<kStepThreads>(V);
  const int lo = min(V, t * P), n = min(V, lo + P) - lo;
  const bool csr = c.pen_on && !a.hist_bits;
  StepIO io;
  io.xf = xf_row;
  io.xb = a.dtype == 1 ? static_cast<const uint16_t*>(a.logits) + roff : nullptr;
  io.bitmap = csr ? bitmap : nullptr;
  io.hbits = (c.pen_on && a.hist_bits) ? a.hist_bits + (int64_t)row * hist_words(V) : nullptr;
  io.out_tok = a.out_tok + row;
  io.rng = a.rng ? a.rng + row : nullptr;
  io.masked = a.out_masked ? a.out_masked + (int64_t)row * V : nullptr;
  io.stats = a.stats ? a.stats + 4 * (int64_t)row : nullptr;
  io.join = a.hist_bits ? a.hist_bits + (int64_t)row * hist_words(V) : nullptr;
  io.stop_token = a.stop_token;
  if (t == 0) {   // read only after the barrier below
    rs.cfg = c;
    rs.io = io;
    rs.tp_exact_first = 0u;
  }
  const float ninf = neg_inf();

  // The history's first two ids of this thread (or this thread's words of the
  // history set) go out behind the row's loads, before anything waits for the
  // row: storing the row to LDS waits for the row alone.
  if (!csr) h0 = h1 = 0;
  const int hid = (csr && h0 + t < h1) ? a.hist_ids[h0 + t] : -1;
  const int hid2 = (csr && h0 + t + kStepThreads < h1) ? a.hist_ids[h0 + t + kStepThreads] : -1;
  // penalty bits of this thread's ids: words lo/32 and lo/32 + 1 (up to 33 ids
  // from bit lo % 32 span at most two words)
  static_assert(PT <= 33, "a thread's ids span at most two bitmap words");
  uint32_t pw[2] = {0u, 0u};
  if (io.hbits) {
    // every load unconditional (index clamped), so nothing waits for them here:
    // the penalty below keeps only the bits of ids lo .. lo + n - 1, and a
    // clamped word past the set would stand for ids at or above V
    const int w0 = lo >> 5, hwn = hist_words(V);
#pragma unroll
    for (int q = 0; q < 2; ++q) pw[q] = io.hbits[min(w0 + q, hwn - 1)];
  }
  // the row into LDS (fp32: its loads went out above)
  float* val;
  if (io.xf) {
    val = step_store(io.xf, V, f, vbuf);
  } else {
    val = stage_row_bf16(io.xb, V, vbuf);
  }
  // LDS: the history bitmap and the histograms start at zero
  const int nw = bitmap_words(V);
  if (csr)
    for (int i = t; i < nw; i += kStepThreads) bitmap[i] = 0u;
  if (!c.greedy)
    for (int i = t; i < (int)(3 * kHistBytes / 4); i += kStepThreads) hc[i] = 0u;
  __syncthreads();
  if (csr) {
    if (hid >= 0 && hid < V) atomicOr(&bitmap[hid >> 5], 1u << (hid & 31));   // sampling.cpp:24
    if (hid2 >= 0 && hid2 < V) atomicOr(&bitmap[hid2 >> 5], 1u << (hid2 & 31));
    for (int64_t j = h0 + t + 2 * kStepThreads; j < h1; j += kStepThreads) {
      const int id = a.hist_ids[j];
      if (id >= 0 && id < V) atomicOr(&bitmap[id >> 5], 1u << (id & 31));
    }
    __syncthreads();
    // unconditional reads (index clamped, as for the caller's set above)
    const int w0 = lo >> 5;
#pragma unroll
    for (int q = 0; q < 2; ++q) pw[q] = bitmap[min(w0 + q, nw - 1)];
  }
  C4S_PHASE(1);
  if (c.pen_on) {
    // sampling.cpp:19-28 on this thread's ids in LDS, one set bit at a time
    // (each distinct id once); the row in LDS is the penalised row from here on
    // (dividing only the set bits: every value of the thread through the
    // double reciprocal costs more than this loop)
    const double rp = 1.0 / (double)c.pen;
    uint32_t pm = (uint32_t)(((((uint64_t)pw[1] << 32) | pw[0]) >> (lo & 31))) & ((1u << n) - 1u);
    while (pm) {
      const int i = lo + __ffs(pm) - 1;
      pm &= pm - 1;
      const float x = val[i];
      val[i] = (x < 0) ? x * c.pen : div_rcp(x, rp);   // sampling.cpp:26
    }
  }
  C4S_PHASE(14);
  // this thread's ids (odd stride: no LDS bank conflicts), every read
  // unconditional (index clamped) and the padding selected afterwards
  float y[PT];
  read_row(val, lo, n, V, y);
  if (n < PT) {
#pragma unroll
    for (int j = 0; j < PT; ++j) y[j] = j < n ? y[j] : ninf;
  }
  C4S_PHASE(29);

  if (c.greedy) {   // text2semantic.cpp:144-145: argmax of the penalised row, first maximum
    float bv = ninf;
    int bi = INT_MAX;
#pragma unroll
    for (int j = 0; j < PT; ++j)
      if (j < n) argmax_merge(bv, bi, y[j], lo + j);
    block_argmax<kStepThreads>(bv, bi, sh.redf, sh.redi);
    if (io.masked)
#pragma unroll
      for (int j = 0; j < PT; ++j)
        if (j < n) io.masked[lo + j] = y[j];
    if (t == 0) step_out(io, V, bi, 0ull, false, 8u | 16u, 0u, 0u, (uint32_t)V);
    return;
  }

  // top-k rows with k <= 64: on a candidate list when it settles the step
  if (c.draw && c.topk_on && c.k <= kWave && c.p > 0.0f && !io.masked) {
    if (list_fast<PT>(io, c, V, y, lo, n, val, *reinterpret_cast<FastSh*>(work))) return;
    for (int i = t; i < (int)(3 * kHistBytes / 4); i += kStepThreads) hc[i] = 0u;
    __syncthreads();
  }

  bool done;
  if (c.topk_on) done = sampled_step_many<PT, kKindTopK>(io, c, lo, n, val, hc, hm, sbuf, list, ss, rs);
  else if (c.p >= 1.0f) done = sampled_step_many<PT, kKindDense>(io, c, lo, n, val, hc, hm, sbuf, list, ss, rs);
  else done = sampled_step_many<PT, kKindTopP>(io, c, lo, n, val, hc, hm, sbuf, list, ss, rs);
  if (done) return;
  __syncthreads();   // every thread is done with the work area
  chain_fallback_global(rs.io, rs.cfg, work, (uint32_t)(kStepWorkBytes + 4 * (size_t)vpad(V)), sh,
                        rs.tp_exact_first != 0u);
}

// LDS of one row: the one pass's work area, the row, the bitmap.
size_t many_lds_bytes(int V) { return kStepWorkBytes + 4 * ((size_t)vpad(V) + 4) + 4 * (size_t)bitmap_words(V); }

}  // namespace

// More than 2.25 rows a CU (kManyRows), two of them in a CU's LDS (static part included: up to
// about 9200 ids), the exact top_p's keys (a power of two) within one row's.
bool rows_step_many_fits(const RowsArgs& a) {
  constexpr size_t kStatic = sizeof(StepScratch) + sizeof(StepSh) + sizeof(StepRowSh) + 256;
  size_t keys = 1;
  while (keys < (size_t)a.vocab) keys <<= 1;
  return a.n_rows > kManyRows && 2 * (many_lds_bytes(a.vocab) + kStatic) <= 160 * 1024 &&
         kStepWorkBytes + 4 * (size_t)vpad(a.vocab) >= 4 * keys;
}

hipError_t launch_rows_step_many(const RowsArgs& a, hipStream_t s) {
  const size_t lds = many_lds_bytes(a.vocab);
  const int P = ((a.vocab + kStepThreads - 1) / kStepThreads) | 1;   // ids a thread owns (odd_chunk)
  const dim3 g(a.n_rows), b(kStepThreads);
  if (P <= 9) hipLaunchKernelGGL(k_rows_step_many<9>, g, b, lds, s, a);
  else if (P <= 17) hipLaunchKernelGGL(k_rows_step_many<17>, g, b, lds, s, a);
  else hipLaunchKernelGGL(k_rows_step_many<25>, g, b, lds, s, a);
  return hipGetLastError();
}

}  // namespace c4s
