// One AR step at vocabularies too large for LDS, by slices of a row.
//
// A row is cut into slices of kSlice ids and decided in three phases, each of
// which reads a slice with coalesced 16-byte loads and keeps it in registers:
//
//  A (per slice)  penalty (and, for sampled rows, temperature); greedy rows:
//     the slice's first maximum; top-k rows (k <= kBigMaxK): every value that
//     can be among the row's k largest; rows without top_k: the slice's
//     maximum m_s and a histogram of fp32 masses exp(z - m_s) over buckets of
//     1/32 below it, on a grid of absolute values.
//  B (rows without top_k) the slices' histograms merged to one over the row
//     give the window of buckets X in which the nucleus boundary lies; then per
//     slice, with the reference's masses exp((double)fl(z - m)): their sum, the
//     sum above X by chunk of ids, and X's entries as a list.
//  C (per row)    greedy: the largest of the slices' maxima; top-k: the slices'
//     candidates sorted, then topk_finish; else X sorted by (value desc, id
//     asc), the cut at mass (1 - p) S (sampling.cpp:60-65), the draw's chunk
//     from the chunk sums and the token from that chunk's ids read again
//     (text2semantic.cpp:150-165).
//
// Sums are formed in parallel in double; a decision within rel_eps of its
// boundary, or any other case the phases do not cover, sends the row to the
// general path (rows_global_row) before its RNG or any output changes.
//
// Either each phase is a launch of one workgroup per (slice, row), so a handful
// of rows spreads over the chip, or one workgroup walks its row through all
// phases (big_by_phase has the rule). On the multi-pass chain a nucleus row was
// bound by one CU's radix passes, each with a double exp and two LDS atomics a
// value: 32 bf16 rows of 151936 took 823 us, 48 us here (12 A, 20 B, 13 C).
// What bounds the phases now: B's double masses (about 40 instructions a value)
// and, in C, a chain of short steps between barriers.

#pragma once

#include "c4s_step.hpp"

namespace c4s {
namespace {

constexpr int kSlice = 16384;              // ids per slice
constexpr int kBigNB = 1024;               // histogram buckets of 1 / kBigScale below the maximum
constexpr float kBigScale = 32.0f;
constexpr int kBigListCap = 2048;          // entries a slice may list
constexpr int kBigRowCap = 6144;           // entries a row's lists may hold
constexpr int kBigSortCap = 4096;          // boundary entries one row may sort
constexpr int kBigMaxChunks = 1056;
// top-k rows: the slice's bound is taken from its threads' two largest keys;
// a wave that holds any of the row has its 64 lanes filled first, so 128 keys
// stand behind a bound for up to 121 (k + 1)
constexpr int kBigMaxK = 120;

// What a slice reports (one per slice in the row's workspace).
struct BigHdr {
  unsigned long long best;   // greedy: key of the first maximum (value key, ~id)
  double S;                  // sum of the slice's masses (relative to the row maximum)
  double Sab;                // the same above X
  float ms;                  // largest z of the slice
  uint32_t n;                // entries listed (may exceed the list: the row is not settled here)
  uint32_t nab;              // values above X (dense rows: finite values)
  uint32_t tout;             // top-k: largest key below the listed candidates
  uint32_t flags;            // 1: masses near underflow
  uint32_t pad;
  float wm;                  // the first slice's: the row's window (phase B, for phase C)
  int wxlo, wxhi;
};
static_assert(sizeof(BigHdr) == 64, "header layout");

// A row's workspace: headers, histograms, lists, chunk sums.
struct BigWs {
  BigHdr* hdr;               // [nsl]
  float* hist;               // [nsl][kBigNB]
  unsigned long long* list;  // [nsl][kBigListCap]
  double* chunk;             // [nsl * chunks a slice]
};
__host__ __device__ __forceinline__ int big_slices(int V) { return (V + 7 + kSlice - 1) / kSlice; }
constexpr size_t kBigSliceBytes = 64 + 4 * (size_t)kBigNB + 8 * (size_t)kBigListCap + 16 * 8;
// the sort workspace of a row (4 bytes times the power of two at or above V) holds it
static_assert(kBigSliceBytes <= 2 * 4 * (size_t)kSlice, "a slice's workspace within its share");
__device__ __forceinline__ BigWs big_ws(const RowsArgs& a, int row, int nsl) {
  unsigned char* p = reinterpret_cast<unsigned char*>(a.sort_ws + (int64_t)row * a.sort_ws_stride);
  BigWs w;
  w.hdr = reinterpret_cast<BigHdr*>(p);
  w.chunk = reinterpret_cast<double*>(p + (size_t)nsl * 64);
  w.list = reinterpret_cast<unsigned long long*>(p + (size_t)nsl * (64 + 128));
  w.hist = reinterpret_cast<float*>(p + (size_t)nsl * (64 + 128 + 8 * (size_t)kBigListCap));
  return w;
}

// The row as the slices see it: element position p stands for id p - off, so
// that 16-byte loads at multiples of 16 bytes are aligned whatever the row's
// first address.
struct BigGeo {
  const void* base;   // the row's first element
  int dtype, V, off;
};
__device__ __forceinline__ BigGeo big_geo(const RowsArgs& a, int row) {
  BigGeo g;
  const int es = a.dtype == 0 ? 4 : 2;
  g.base = static_cast<const unsigned char*>(a.logits) + (int64_t)row * a.ld * es;
  g.dtype = a.dtype;
  g.V = a.vocab;
  g.off = (int)((reinterpret_cast<uintptr_t>(g.base) & 15u) / (unsigned)es);
  return g;
}
struct BigRow {
  bool pen_on, temp_on;
  float pen;
  double rpen, rtemp;
  __device__ __forceinline__ float z(float y) const { return temp_on ? div_rcp(y, rtemp) : y; }
};
__device__ __forceinline__ BigRow big_row(const RowCfg& c) {
  BigRow r;
  r.pen_on = c.pen_on;
  r.temp_on = c.temp_on;
  r.pen = c.pen;
  r.rpen = 1.0 / (double)c.pen;
  r.rtemp = 1.0 / (double)c.temp;
  return r;
}

// A row's history as a thread holds it: its first kBigPre ids (CSR), loaded
// ahead of their use.
constexpr int kBigPre = 4;
struct BigHist {
  int64_t h0, h1;
  int id[kBigPre];
};
template <int NTH>
__device__ __forceinline__ BigHist big_hist(const RowsArgs& a, int64_t h0, int64_t h1) {
  BigHist h;
  h.h0 = h0;
  h.h1 = h1;
#pragma unroll
  for (int i = 0; i < kBigPre; ++i) {
    const int64_t j = h.h0 + threadIdx.x + NTH * i;
    h.id[i] = j < h.h1 ? a.hist_ids[j] : -1;
  }
  return h;
}
// The history's bits for ids id0 .. id0 + 32 nw - 1 (id0 may be negative)
// into bm[0 .. nw - 1]: from the kept set (its words shifted), or cleared and
// then set from the CSR ids, with a barrier after each.
template <int NTH>
__device__ __forceinline__ void big_bits_clear(const RowsArgs& a, int row, int id0, int nw, uint32_t* bm) {
  for (int i = threadIdx.x; i < nw; i += NTH) {
    uint32_t v = 0u;
    if (a.hist_bits) {
      const uint32_t* hb = a.hist_bits + (int64_t)row * hist_words(a.vocab);
      const int w = (id0 >> 5) + i, hw = hist_words(a.vocab);
      v = __funnelshift_r(w >= 0 && w < hw ? hb[w] : 0u, w + 1 >= 0 && w + 1 < hw ? hb[w + 1] : 0u, id0 & 31);
    }
    bm[i] = v;
  }
}
template <int NTH>
__device__ __forceinline__ void big_bits_set(const RowsArgs& a, const BigHist& h, int id0, int nw, uint32_t* bm) {
  auto set = [&](int id) {
    const int64_t d = (int64_t)id - id0;
    if (id >= 0 && id < a.vocab && d >= 0 && d < 32 * (int64_t)nw) atomicOr(&bm[d >> 5], 1u << (d & 31));   // sampling.cpp:24
  };
#pragma unroll
  for (int i = 0; i < kBigPre; ++i) set(h.id[i]);
  for (int64_t j = h.h0 + threadIdx.x + (int64_t)NTH * kBigPre; j < h.h1; j += NTH) set(a.hist_ids[j]);
}

// A thread's VPT values of slice s, penalised: wave w of the slice holds the
// 64 VPT positions from s kSlice + 64 VPT w on, load j of lane l the EPV
// positions from 64 EPV j + EPV l on. -inf outside the row.
template <int VPT, int EPV>
__device__ __forceinline__ int big_id(int s, int i, int off) {
  return s * kSlice + wave_id() * (kWave * VPT) + (i / EPV) * (kWave * EPV) + lane_id() * EPV + (i % EPV) - off;
}
template <int VPT, int EPV>
struct BigFetch {
  uint4 q[VPT / EPV];
};
__device__ __forceinline__ bool big_inside(const BigGeo& g, int s) {   // uniform: the slice lies in the row
  return s * kSlice - g.off >= 0 && (s + 1) * kSlice - g.off <= g.V;
}
template <int VPT, int EPV>
__device__ __forceinline__ void big_fetch(const BigGeo& g, int s, BigFetch<VPT, EPV>& f) {
  const int id0 = big_id<VPT, EPV>(s, 0, g.off);
  const uint4* p = reinterpret_cast<const uint4*>(static_cast<const unsigned char*>(g.base) + (int64_t)id0 * (16 / EPV));
  if (big_inside(g, s)) {
#pragma unroll
    for (int j = 0; j < VPT / EPV; ++j) f.q[j] = p[kWave * j];
  } else {
#pragma unroll
    for (int j = 0; j < VPT / EPV; ++j) {
      const int i0 = id0 + kWave * EPV * j;
      if (i0 >= 0 && i0 + EPV <= g.V) f.q[j] = p[kWave * j];
    }
  }
}
template <int VPT, int EPV>
__device__ __forceinline__ void big_take(const BigGeo& g, int s, const BigFetch<VPT, EPV>& f, float (&y)[VPT]) {
  const int id0 = big_id<VPT, EPV>(s, 0, g.off);
  const bool inside = big_inside(g, s);
  const float ninf = neg_inf();
#pragma unroll
  for (int j = 0; j < VPT / EPV; ++j) {
    const int i0 = id0 + kWave * EPV * j;
    if (inside || (i0 >= 0 && i0 + EPV <= g.V)) {
      if constexpr (EPV == 4) {
        y[4 * j] = __uint_as_float(f.q[j].x);
        y[4 * j + 1] = __uint_as_float(f.q[j].y);
        y[4 * j + 2] = __uint_as_float(f.q[j].z);
        y[4 * j + 3] = __uint_as_float(f.q[j].w);
      } else {
        const uint32_t v[4] = {f.q[j].x, f.q[j].y, f.q[j].z, f.q[j].w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          y[8 * j + 2 * e] = __uint_as_float(v[e] << 16);
          y[8 * j + 2 * e + 1] = __uint_as_float(v[e] & 0xFFFF0000u);
        }
      }
    } else {   // the row's first and last elements, one at a time
#pragma unroll
      for (int e = 0; e < EPV; ++e) {
        const int id = i0 + e;
        float x = ninf;
        if (id >= 0 && id < g.V) {
          if constexpr (EPV == 4) x = static_cast<const float*>(g.base)[id];
          else x = __uint_as_float((uint32_t)static_cast<const uint16_t*>(g.base)[id] << 16);
        }
        y[EPV * j + e] = x;
      }
    }
  }
}
// sampling.cpp:19-28 on those values: bit p of bm stands for the slice's
// position p, so a load's bits lie in one word.
template <int VPT, int EPV>
__device__ __forceinline__ void big_penalise(const BigRow& r, const uint32_t* bm, float (&y)[VPT]) {
  const int p0 = wave_id() * (kWave * VPT) + lane_id() * EPV;
  uint32_t bits[VPT / EPV];
#pragma unroll
  for (int j = 0; j < VPT / EPV; ++j) bits[j] = bm[(p0 + kWave * EPV * j) >> 5];
#pragma unroll
  for (int j = 0; j < VPT / EPV; ++j) {
    const uint32_t b = (bits[j] >> (p0 & 31)) & ((1u << EPV) - 1u);   // a load's stride is whole words
    if (b) {
#pragma unroll
      for (int e = 0; e < EPV; ++e) {
        const float x = y[EPV * j + e];
        const float px = x < 0 ? x * r.pen : div_rcp(x, r.rpen);
        y[EPV * j + e] = ((b >> e) & 1u) ? px : x;
      }
    }
  }
}
constexpr int kBigBitWords = kSlice / 32;   // a slice's positions

struct BigShA {
  uint32_t bm[kBigBitWords];
  union {
    unsigned long long hist[kBigNB];   // masses, 2^-31 units
    uint32_t kh[2][2048];              // top-k: key prefixes
  };
  float wf[NW];
  uint32_t wu[NW], wv[NW];
  unsigned long long wk[NW];
  uint32_t pick[4];
  uint32_t n;
};

// Bin of hist (2048 bins, from the top) holding the m-th largest counted key,
// and the count above it; false (uniform) when fewer were counted. Either way a
// barrier has passed since the last read of red, so the caller may write it.
template <int NTH>
__device__ __forceinline__ bool big_pick(const uint32_t* hist, uint32_t* red, uint32_t* out, uint32_t m, uint32_t& bin,
                                         uint32_t& above) {
  constexpr int PB = 2048 / NTH;
  const int t = threadIdx.x;
  uint32_t cb[PB], loc = 0;
#pragma unroll
  for (int i = 0; i < PB; ++i) { cb[i] = hist[2047 - PB * t - i]; loc += cb[i]; }
  const uint32_t inc = wave_scan_u32(loc);
  if (lane_id() == kWave - 1) red[wave_id()] = inc;
  __syncthreads();
  uint32_t ex = inc - loc, total = 0;
#pragma unroll
  for (int i = 0; i < NTH / kWave; ++i) {
    const uint32_t x = red[i];
    ex += i < wave_id() ? x : 0u;
    total += x;
  }
  if (total < m) {
    __syncthreads();
    return false;
  }
  if (ex < m && ex + loc >= m) {
    uint32_t run = ex;
#pragma unroll
    for (int i = 0; i < PB; ++i) {
      if (run < m && run + cb[i] >= m) { out[0] = (uint32_t)(2047 - PB * t - i); out[1] = run; }
      run += cb[i];
    }
  }
  __syncthreads();
  bin = out[0];
  above = out[1];
  return true;
}

// The entries of a thread's set bits (VPT <= 32) to the slice's list: one slot
// claim a wave, and stores that wait for nothing.
template <int VPT, class Entry>
__device__ __forceinline__ void big_push(uint32_t cm, unsigned long long* list, uint32_t& n, Entry&& entry) {
  static_assert(VPT <= 32, "a thread's values as one mask");
  const uint32_t c = (uint32_t)__popc(cm), inc = wave_scan_u32(c);
  uint32_t base = 0;
  if (lane_id() == kWave - 1 && inc) base = atomicAdd(&n, inc);
  uint32_t slot = readlane_u32(base, kWave - 1) + inc - c;
#pragma unroll
  for (int i = 0; i < VPT; ++i)
    if ((cm >> i) & 1u) {
      if (slot < (uint32_t)kBigListCap) list[slot] = entry(i);
      ++slot;
    }
}

// Phase A of slice s. Every thread of the workgroup; a barrier between calls.
template <int NTH, int EPV>
__device__ __forceinline__ void big_phase_a(const RowsArgs& a, int row, const RowCfg& c, const BigGeo& g, const BigRow& r,
                                            const BigHist& hs, const BigFetch<kSlice / NTH, EPV>& f, const BigWs& ws,
                                            int s, BigShA& sh) {
  constexpr int VPT = kSlice / NTH;
  const int t = threadIdx.x, lane = lane_id(), w = wave_id();
  const float ninf = neg_inf();
  float y[VPT];
  const int b0 = s * kSlice - g.off;   // the first position's id
  C4S_PHASE(2);
  const bool topk = c.topk_on, nuc = !c.greedy && !c.topk_on;
  if (c.pen_on) big_bits_clear<NTH>(a, row, b0, kBigBitWords, sh.bm);
  if (nuc) {
    for (int i = t; i < kBigNB; i += NTH) sh.hist[i] = 0ull;
  } else if (topk) {
    for (int i = t; i < 2 * 2048; i += NTH) (&sh.kh[0][0])[i] = 0u;
    if (t == 0) sh.n = 0u;
  }
  __syncthreads();
  if (c.pen_on) {
    big_bits_set<NTH>(a, hs, b0, kBigBitWords, sh.bm);
    __syncthreads();
  }
  C4S_PHASE(3);
  big_take<VPT, EPV>(g, s, f, y);
  if (c.pen_on) big_penalise<VPT, EPV>(r, sh.bm, y);
  C4S_PHASE(4);
  BigHdr* h = ws.hdr + s;
  if (c.greedy) {
    float bv = ninf;
    int bi = 0;
#pragma unroll
    for (int i = 0; i < VPT; ++i)
      if (y[i] > bv) { bv = y[i]; bi = i; }
    // index -> id: load j = i / EPV
    const int id = s * kSlice + w * (kWave * VPT) + (bi / EPV) * (kWave * EPV) + lane * EPV + (bi % EPV) - g.off;
    unsigned long long k = bv == ninf ? 0ull : (((unsigned long long)fkey(bv) << 32) | (uint32_t)~(uint32_t)id);
    k = wave_max_u64_dpp(k);
    if (lane == 0) sh.wk[w] = k;
    __syncthreads();
    if (t == 0) {
      unsigned long long b = 0ull;
      for (int i = 0; i < NTH / kWave; ++i) b = b > sh.wk[i] ? b : sh.wk[i];
      h->best = b;
    }
    C4S_PHASE(5);
    return;
  }
  if (topk) {
    // L0: at least k + 1 of the slice's values (all, where it holds fewer)
    // have a key at or above it (two 11-bit passes over the threads' two
    // largest keys); -inf and what lies outside the row is no candidate
    uint32_t t1 = 0, t2 = 0;
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const uint32_t k = fkey(y[i]);
      t2 = max(t2, min(t1, k));
      t1 = max(t1, k);
    }
    C4S_PHASE(22);
    if (t1 > kKeyNegInf) atomicAdd(&sh.kh[0][t1 >> 21], 1u);
    if (t2 > kKeyNegInf) atomicAdd(&sh.kh[0][t2 >> 21], 1u);
    __syncthreads();
    const uint32_t msel = (uint32_t)c.k + 1u;
    uint32_t L0 = 0, bin, ab;
    if (big_pick<NTH>(sh.kh[0], sh.wu, sh.pick, msel, bin, ab)) {
      L0 = bin << 21;
      if (ab + sh.kh[0][bin] > 64u) {   // uniform
        if (t1 > kKeyNegInf && (t1 >> 21) == bin) atomicAdd(&sh.kh[1][(t1 >> 10) & 2047u], 1u);
        if (t2 > kKeyNegInf && (t2 >> 21) == bin) atomicAdd(&sh.kh[1][(t2 >> 10) & 2047u], 1u);
        __syncthreads();
        uint32_t b2, a2;
        big_pick<NTH>(sh.kh[1], sh.wv, sh.pick + 2, msel - ab, b2, a2);
        L0 |= b2 << 10;
      }
    }
    L0 = max(L0, kKeyNegInf + 1u);
    C4S_PHASE(23);
    uint32_t below = 0, cm = 0;
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const uint32_t k = fkey(y[i]);
      cm |= k >= L0 ? 1u << i : 0u;
      below = max(below, k < L0 ? k : 0u);
    }
    big_push<VPT>(cm, ws.list + (size_t)s * kBigListCap, sh.n, [&](int i) {
      return ((unsigned long long)fkey(r.z(y[i])) << 32) | (uint32_t)~(uint32_t)big_id<VPT, EPV>(s, i, g.off);
    });
    below = wave_max_u32_dpp(below);
    if (lane == 0) sh.wu[w] = below;
    __syncthreads();
    if (t == 0) {
      uint32_t b = 0;
      for (int i = 0; i < NTH / kWave; ++i) b = max(b, sh.wu[i]);
      h->tout = b > kKeyNegInf ? fkey(r.z(kfloat(b))) : 0u;
      h->n = sh.n;
    }
    C4S_PHASE(24);
    return;
  }
  // rows without top_k: z, the slice maximum and the histogram below it
  float lm = ninf;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    y[i] = r.z(y[i]);
    lm = fmaxf(lm, y[i]);
  }
  lm = wave_max_dpp(lm);
  if (lane == 0) sh.wf[w] = lm;
  __syncthreads();
  float ms = ninf;
#pragma unroll
  for (int i = 0; i < NTH / kWave; ++i) ms = fmaxf(ms, sh.wf[i]);
  if (t == 0) h->ms = ms;
  C4S_PHASE(25);
  // Dense rows (p >= 1) have no boundary to find. The bound on ms takes in every
  // slice that big_window counts: a row's maximum below 2^18 in magnitude and
  // slices within 32 of it (the grid's differences are exact up to 2^19).
  if (!(c.p < 1.0f) || !(fabsf(ms) < 0x1p19f)) return;   // uniform
  const float fqs = floorf(ms * kBigScale);
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const float fq = floorf(y[i] * kBigScale);
    if (fqs - fq < (float)(kBigNB - 1)) {   // +inf for -inf
      const float e = mass32(y[i] - ms);
      atomicAdd(&sh.hist[(int)fq & (kBigNB - 1)], (unsigned long long)(uint32_t)(e * 0x1p31f));
    }
  }
  __syncthreads();
  float* hist = ws.hist + (size_t)s * kBigNB;
  C4S_PHASE(5);
  for (int i = t; i < kBigNB; i += NTH) hist[i] = (float)((double)sh.hist[i] * 0x1p-31);
  C4S_PHASE(6);
}

struct BigShB {
  uint32_t bm[kBigBitWords];
  float ms[kBigNB];
  double wd[NW], we[NW];
  uint32_t wu[NW], wv[NW];
  uint32_t n;
};

// The row's window from the slices' histograms: X holds the values z with
// xlo <= fQ - floor(32 z) <= xhi (fQ = floor(32 m)), values above it are kept
// whatever the exact sums are. Dense rows: everything is above. False
// (uniform) when the phases do not cover the row.
// A slice's histogram holds the mass of grid value q = floor(32 z) at q mod
// kBigNB, so that its loads need no slice's maximum: they go out together with
// the headers', kBigFly slices at a time, ahead of the row's own loads.
struct BigWin {
  float m, fQ;
  int xlo, xhi;
};
constexpr int kBigFly = 12;
template <int NTH>
struct BigMerge {
  static constexpr int PB = kBigNB / NTH;
  float hm[2];              // the slices' maxima, one or two a lane
  float v[kBigFly][PB];     // the first slices' masses at places PB t + i
};
template <int NTH>
__device__ __forceinline__ void big_merge_fetch(const BigWs& ws, int nsl, int s0, BigMerge<NTH>& f) {
#pragma unroll
  for (int q = 0; q < kBigFly; ++q)
#pragma unroll
    for (int i = 0; i < BigMerge<NTH>::PB; ++i)
      f.v[q][i] = ws.hist[(size_t)min(s0 + q, nsl - 1) * kBigNB + BigMerge<NTH>::PB * threadIdx.x + i];
}
template <int NTH>
__device__ __forceinline__ void big_window_fetch(const BigWs& ws, int nsl, BigMerge<NTH>& f) {
  static_assert((kMaxVocab + 7) / kSlice + 1 <= 2 * kWave, "two headers a lane");
#pragma unroll
  for (int q = 0; q < 2; ++q) f.hm[q] = q * kWave + lane_id() < nsl ? ws.hdr[q * kWave + lane_id()].ms : neg_inf();
  big_merge_fetch<NTH>(ws, nsl, 0, f);
}
template <int NTH>
__device__ __forceinline__ bool big_window(const RowCfg& c, const BigWs& ws, int nsl, BigShB& sh, BigMerge<NTH>& f,
                                           BigWin& win) {
  constexpr int PB = BigMerge<NTH>::PB;
  const int t = threadIdx.x, lane = lane_id(), w = wave_id();
  const float m = wave_max_dpp(fmaxf(f.hm[0], f.hm[1]));
  win.m = m;
  win.fQ = floorf(m * kBigScale);
  win.xlo = kBigNB;
  win.xhi = -1;
  // grid differences are exact below 2^18; the draw's maximum starts at -1e30
  if (!(fabsf(m) < 0x1p18f) || !(c.p > 0.0f)) return false;
  if (!(c.p < 1.0f)) {
    win.xlo = INT_MAX;
    return true;
  }
  C4S_PHASE(26);
  const int Q = (int)win.fQ;
  float ms[PB];
#pragma unroll
  for (int i = 0; i < PB; ++i) ms[i] = 0.0f;
  for (int s0 = 0; s0 < nsl; s0 += kBigFly) {
    if (s0 > 0) big_merge_fetch<NTH>(ws, nsl, s0, f);
#pragma unroll
    for (int q = 0; q < kBigFly; ++q) {
      const int s = min(s0 + q, nsl - 1);
      const float mss = readlane_f32(s < kWave ? f.hm[0] : f.hm[1], s & (kWave - 1));
      const float sf = win.fQ - floorf(mss * kBigScale);   // +inf for an empty slice
      const bool on = s0 + q < nsl && sf < (float)kBigNB;
      const int qs = on ? Q - (int)sf : 0;                  // the slice's largest grid value
      const float sc = on ? mass32(mss - m) : 0.0f;
#pragma unroll
      for (int i = 0; i < PB; ++i) {
        // place r holds the grid value qs - ((qs - r) mod kBigNB); the slice's
        // values kBigNB or more below Q belong to no bucket
        const int below = (qs - (PB * t + i)) & (kBigNB - 1);
        ms[i] = on && Q - qs + below < kBigNB ? __builtin_fmaf(f.v[q][i], sc, ms[i]) : ms[i];
      }
    }
  }
  C4S_PHASE(27);
  // to bucket order: place r is bucket (Q - r) mod kBigNB
#pragma unroll
  for (int i = 0; i < PB; ++i) sh.ms[(Q - (PB * t + i)) & (kBigNB - 1)] = ms[i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < PB; ++i) ms[i] = sh.ms[PB * t + i];
  C4S_PHASE(28);
  double loc = 0.0;
#pragma unroll
  for (int i = 0; i < PB; ++i) loc += (double)ms[i];
  const double inc = wave_scan_f64(loc);
  if (lane == kWave - 1) sh.wd[w] = inc;
  __syncthreads();
  double ex = inc - loc, tot = 0.0;
#pragma unroll
  for (int i = 0; i < NTH / kWave; ++i) {
    const double x = sh.wd[i];
    ex += i < w ? x : 0.0;
    tot += x;
  }
  // the histogram's error against the exact masses: fp32 masses, scalings and
  // sums (2^-18 relative), truncation (2^-31 a value) and the values more than
  // 32 below their slice's maximum (e^-31 a value)
  const double err = tot * 0x1p-17 + (double)c.V * 0x1p-30;
  const double B = tot - (1.0 - (double)c.p) * tot;
  const double Blo = B - err, Bhi = B + err;
  double run = ex;
  int lo = kBigNB, hi = kBigNB;
#pragma unroll
  for (int i = 0; i < PB; ++i) {
    run += (double)ms[i];
    if (lo == kBigNB && run >= Blo) lo = PB * t + i;
    if (hi == kBigNB && run >= Bhi) hi = PB * t + i;
  }
  // the first of each wave (an atomic minimum over the lanes would be a loop
  // over them), then of the workgroup
  const uint64_t bl = __ballot(lo < kBigNB), bh = __ballot(hi < kBigNB);
  const int wl = bl ? (int)readlane_u32((uint32_t)lo, __ffsll((unsigned long long)bl) - 1) : kBigNB;
  const int wh = bh ? (int)readlane_u32((uint32_t)hi, __ffsll((unsigned long long)bh) - 1) : kBigNB;
  if (lane == 0) { sh.wu[w] = (uint32_t)wl; sh.wv[w] = (uint32_t)wh; }
  __syncthreads();
  win.xhi = kBigNB;
#pragma unroll
  for (int i = 0; i < NTH / kWave; ++i) {
    win.xlo = min(win.xlo, (int)sh.wu[i]);
    win.xhi = min(win.xhi, (int)sh.wv[i]);
  }
  __syncthreads();
  return win.xhi < kBigNB - 1;   // not in the open bucket below the last
}

// Phase B of slice s.
template <int NTH, int EPV>
__device__ __forceinline__ void big_phase_b(const RowsArgs& a, int row, const RowCfg& c, const BigGeo& g, const BigRow& r,
                                            const BigHist& hs, const BigFetch<kSlice / NTH, EPV>& f, const BigWs& ws,
                                            int s, const BigWin& win, BigShB& sh) {
  constexpr int VPT = kSlice / NTH, NWV = NTH / kWave;
  const int t = threadIdx.x, lane = lane_id(), w = wave_id();
  float y[VPT];
  const int b0 = s * kSlice - g.off;   // the first position's id
  if (c.pen_on) big_bits_clear<NTH>(a, row, b0, kBigBitWords, sh.bm);
  if (t == 0) sh.n = 0u;
  __syncthreads();
  if (c.pen_on) {
    big_bits_set<NTH>(a, hs, b0, kBigBitWords, sh.bm);
    __syncthreads();
  }
  big_take<VPT, EPV>(g, s, f, y);
  if (c.pen_on) big_penalise<VPT, EPV>(r, sh.bm, y);
  C4S_PHASE(9);
  const float flo = (float)win.xlo, fhi = (float)win.xhi;   // INT_MAX: above every difference that counts
  double S = 0.0, Sab = 0.0;
  uint32_t nab = 0, flags = 0;
  uint32_t cm = 0;   // X
  const bool dense = !(c.p < 1.0f);
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const float z = r.z(y[i]);
    const float tt = z - win.m;
    const double e = exp_neg((double)tt);   // 0 for -inf
    const float d = win.fQ - floorf(z * kBigScale);
    const bool ab = dense ? z != neg_inf() : d < flo;
    S += e;
    Sab += ab ? e : 0.0;
    nab += ab ? 1u : 0u;
    if (dense && ab && tt < -690.0f) flags = 1u;   // subnormal masses: libm implementations may disagree
    cm |= !ab && d <= fhi ? 1u << i : 0u;
  }
  big_push<VPT>(cm, ws.list + (size_t)s * kBigListCap, sh.n,
                [&](int i) { return key64(r.z(y[i]), big_id<VPT, EPV>(s, i, g.off)); });
  C4S_PHASE(10);
  S = wave_sum_dpp(S);
  Sab = wave_sum_dpp(Sab);
  nab = wave_scan_u32(nab);
  flags = __ballot(flags != 0u) ? 1u : 0u;
  if (lane == kWave - 1) {
    ws.chunk[s * NWV + w] = Sab;
    sh.wd[w] = S;
    sh.we[w] = Sab;
    sh.wu[w] = nab;
    sh.wv[w] = flags;
  }
  __syncthreads();
  if (t == 0) {
    double s1 = 0.0, s2 = 0.0;
    uint32_t n = 0, f = 0;
    for (int i = 0; i < NWV; ++i) { s1 += sh.wd[i]; s2 += sh.we[i]; n += sh.wu[i]; f |= sh.wv[i]; }
    BigHdr* h = ws.hdr + s;
    h->S = s1;
    h->Sab = s2;
    h->nab = n;
    h->n = sh.n;
    h->flags = f;
  }
  C4S_PHASE(11);
}

constexpr int kBigSub = 256;   // sub-buckets of the boundary window

struct BigShC {
  unsigned long long x[kBigRowCap];      // the slices' lists
  unsigned long long list[kBigSortCap];  // the entries at the boundary
  double chunk[kBigMaxChunks];
  unsigned long long list2[kBigSub];     // the same, narrowed by id
  double sm[kBigSub];
  uint32_t sn[kBigSub];
  uint32_t kmin, kmax;
  uint32_t bm[kBigBitWords];
  double wd[NW];
  uint32_t wu[NW], wv[NW];
  uint32_t pre[80];        // slices' list offsets
  unsigned long long kthr;
  double mab, cex;
  uint32_t n, nabx;
  int slo, shi;
  int chunk_of;
  int tok, verdict;
};

// Workgroup scan (thread order) of a double and a count over NT threads:
// exclusive prefixes and totals; two barriers.
struct BigScan {
  double ex, in, tot;
  uint32_t utot;
};
__device__ __forceinline__ BigScan big_scan(double v, uint32_t u, BigShC& sh) {
  const int w = wave_id();
  const double inc = wave_scan_f64(v);
  const uint32_t uinc = wave_scan_u32(u);
  __syncthreads();
  if (lane_id() == kWave - 1) { sh.wd[w] = inc; sh.wu[w] = uinc; }
  __syncthreads();
  BigScan r;
  double base = 0.0, run = 0.0;
  uint32_t ut = 0;
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    if (i == w) base = run;
    run += sh.wd[i];
    ut += sh.wu[i];
  }
  r.ex = base + wave_shr1_f64(inc, 0.0);
  r.in = base + inc;
  r.tot = run;
  r.utot = ut;
  return r;
}

__device__ __forceinline__ void big_out(const RowsArgs& a, int row, int tok, bool draw, uint64_t st2, uint32_t s0,
                                        uint32_t kept) {
  a.out_tok[row] = tok;
  if (draw && a.rng) a.rng[row] = st2;
  join_history(a, row, tok);
  if (a.stats) {
    uint32_t* st = a.stats + 4 * (int64_t)row;
    st[0] = s0;
    st[1] = 0u;
    st[2] = 0u;
    st[3] = kept;
  }
}

// Phase C of a row without top_k (NT threads): true when the row is finished.
// VPT: values a thread of phase B held (a chunk of ids is 64 VPT positions).
// X (up to kBigRowCap entries) goes to LDS; a histogram of its exact
// masses over kBigSub sub-buckets finds the few entries at the boundary, and
// only those are sorted (sorting all of X, about 900 entries on the 151936-id
// rows, took 33k of the phase's 72k cycles).
template <int VPT>
__device__ __forceinline__ bool big_phase_c(const RowsArgs& a, int row, const RowCfg& c, const BigGeo& g, const BigRow& r,
                                            const BigHist& hs, const BigWs& ws, int nsl, const BigWin& win, BigShC& sh) {
  constexpr int kChunkPos = kWave * VPT;
  const int t = threadIdx.x, lane = lane_id(), w = wave_id();
  const bool dense = !(c.p < 1.0f);
  const int nch = nsl * (kSlice / kChunkPos);
  // headers: nsl <= 65, one or two a lane, by every wave alike
  double S = 0.0, Ma = 0.0;
  uint32_t nab = 0, nx = 0, bad = 0;
  for (int b = 0; b < nsl; b += kWave) {
    const int i = b + lane;
    const bool in = i < nsl;
    const BigHdr h = ws.hdr[in ? i : 0];
    const uint32_t n = in ? h.n : 0u;
    const uint32_t inc = wave_scan_u32(n);
    if (in && w == 0) sh.pre[i] = nx + inc - n;
    S += wave_sum_dpp(in ? h.S : 0.0);
    Ma += wave_sum_dpp(in ? h.Sab : 0.0);
    nab += readlane_u32(wave_scan_u32(in ? h.nab : 0u), kWave - 1);
    nx += readlane_u32(inc, kWave - 1);
    bad |= __ballot(in && (h.flags != 0u || h.n > (uint32_t)kBigListCap)) ? 1u : 0u;
  }
  const int nX = (int)nx;
  C4S_PHASE(13);
  C4S_PHASE_VAL(30, nX);
  if (bad || nX > kBigRowCap) return false;   // uniform
  const double thr = 1.0 - (double)c.p;   // sampling.cpp:64 removes while cum <= 1 - p
  const int mk = max(0, c.min_keep);
  uint32_t kept = nab;
  for (int i = t; i < nch; i += NT) sh.chunk[i] = ws.chunk[i];
  if (t < kChunkPos / 32) sh.bm[t] = 0u;
  if (dense) {
    // p == 1 with min_keep above the positive masses keeps zero-mass values (sampling.cpp:67-68)
    if (thr == 0.0 && nab < (uint32_t)mk) return false;
  } else {
    if (t < kBigSub) {
      sh.sm[t] = 0.0;
      sh.sn[t] = 0u;
    }
    if (t == 0) { sh.n = 0u; sh.slo = kBigSub; sh.shi = kBigSub; sh.kmin = ~0u; sh.kmax = 0u; }
    __syncthreads();
    // the slices' lists: consecutive entries of one after another
    for (int j = t, q = 0; j < nX; j += NT) {
      while (q + 1 < nsl && (int)sh.pre[q + 1] <= j) ++q;
      sh.x[j] = ws.list[(size_t)q * kBigListCap + (j - (int)sh.pre[q])];
    }
    // sub-buckets of equal width over the window, monotone in z
    const float nbk = (float)(win.xhi + 1 - win.xlo), ssc = (float)kBigSub / nbk;
    const float top = win.fQ + 1.0f - (float)win.xlo;   // exact: below 2^24
    auto sub_of = [&](float z) { return min(kBigSub - 1, max(0, (int)((top - z * kBigScale) * ssc))); };
    for (int j = t; j < nX; j += NT) {   // the thread's own entries
      const float z = key_value(sh.x[j]);
      const int b = sub_of(z);
      atomicAdd(&sh.sm[b], exp_neg((double)(z - win.m)));
      atomicAdd(&sh.sn[b], 1u);
    }
    __syncthreads();
    C4S_PHASE(14);
    // entry j is removed iff the mass at or below it in ascending order,
    // M = S - (mass above it), is <= thr S (sampling.cpp:60-65)
    const double A = thr * S, mg = rel_eps(c.V) * S, B = S - A;
    // what lies above X is kept unseen: only where its exact mass falls short of
    // the boundary, whatever the histograms said
    if (!(Ma < B - 2.0 * mg)) return false;   // uniform
    // where the kept set ends among the sub-buckets, from mass m0 and n0 entries before them
    auto sub_scan = [&](double m0, uint32_t n0) {
      if (w == 0) {
        constexpr int PS = kBigSub / kWave;
        double m4[PS], lm = 0.0;
        uint32_t n4[PS], ln = 0;
#pragma unroll
        for (int q = 0; q < PS; ++q) {
          m4[q] = sh.sm[PS * lane + q];
          n4[q] = sh.sn[PS * lane + q];
          lm += m4[q];
          ln += n4[q];
        }
        double run = m0 + (wave_scan_f64(lm) - lm);
        uint32_t nr = n0 + wave_scan_u32(ln) - ln;
        int lo = kBigSub, hi = kBigSub;
        double mlo = 0.0;
        uint32_t nlo = 0;
#pragma unroll
        for (int q = 0; q < PS; ++q) {
          const double nxm = run + m4[q];
          if (lo == kBigSub && nxm >= B - 2.0 * mg) { lo = PS * lane + q; mlo = run; nlo = nr; }
          if (hi == kBigSub && nxm >= B + 2.0 * mg) hi = PS * lane + q;
          run = nxm;
          nr += n4[q];
        }
        const uint64_t bl = __ballot(lo < kBigSub), bh = __ballot(hi < kBigSub);
        if (bl && lane == __ffsll((unsigned long long)bl) - 1) {
          sh.slo = lo;
          sh.mab = mlo;
          sh.nabx = nlo;
        }
        if (bh && lane == __ffsll((unsigned long long)bh) - 1) sh.shi = hi;
      }
      __syncthreads();
    };
    sub_scan(Ma, nab);
    int slo = sh.slo, shi = sh.shi;
    if (slo >= kBigSub || shi >= kBigSub) return false;   // uniform
    uint32_t kmin = ~0u, kmax = 0u;
    for (int j = t; j < nX; j += NT) {
      const uint64_t e = sh.x[j];
      const int b = sub_of(key_value(e));
      if (b >= slo && b <= shi) {
        const uint32_t slot = atomicAdd(&sh.n, 1u);
        if (slot < (uint32_t)kBigSortCap) sh.list[slot] = e;
        kmin = min(kmin, (uint32_t)(e >> 32));
        kmax = max(kmax, (uint32_t)(e >> 32));
      }
    }
    kmin = wave_min_u32_dpp(kmin);
    kmax = wave_max_u32_dpp(kmax);
    if (lane == 0 && kmax) {
      atomicMin(&sh.kmin, kmin);
      atomicMax(&sh.kmax, kmax);
    }
    __syncthreads();
    int nB = (int)sh.n;
    if (nB > kBigSortCap) return false;   // uniform
    double Mb = sh.mab;
    uint32_t nbx = sh.nabx;
    unsigned long long* list = sh.list;
    if (nB > kWave && sh.kmin == sh.kmax) {
      // many entries of one value (logits of few bits): in id order, so the
      // same again over ranges of ids
      const double e1 = exp_neg((double)(kfloat(sh.kmin) - win.m));
      const int iw = (c.V + kBigSub - 1) / kBigSub;
      __syncthreads();   // the scan's results and n have been read
      if (t < kBigSub) {
        sh.sm[t] = 0.0;
        sh.sn[t] = 0u;
      }
      if (t == 0) { sh.n = 0u; sh.slo = kBigSub; sh.shi = kBigSub; }
      __syncthreads();
      for (int j = t; j < nB; j += NT) {
        const int b = (int)~(uint32_t)sh.list[j] / iw;
        atomicAdd(&sh.sm[b], e1);
        atomicAdd(&sh.sn[b], 1u);
      }
      __syncthreads();
      sub_scan(Mb, nbx);
      slo = sh.slo;
      shi = sh.shi;
      if (slo >= kBigSub || shi >= kBigSub) return false;   // uniform
      for (int j = t; j < nB; j += NT) {
        const int b = (int)~(uint32_t)sh.list[j] / iw;
        if (b >= slo && b <= shi) {
          const uint32_t slot = atomicAdd(&sh.n, 1u);
          if (slot < (uint32_t)kBigSub) sh.list2[slot] = sh.list[j];
        }
      }
      __syncthreads();
      nB = (int)sh.n;
      if (nB > kBigSub) return false;   // uniform
      Mb = sh.mab;
      nbx = sh.nabx;
      list = sh.list2;
    }
    C4S_PHASE_VAL(31, nB);
    int P = 1;
    while (P < nB) P <<= 1;
    if (nB <= kWave) {
      if (w == 0) {
        const uint64_t v = sort_desc_wave(lane < nB ? (uint64_t)list[lane] : 0ull, P);
        if (lane < nB) list[lane] = v;
      }
      __syncthreads();
    } else {
      for (int i = nB + t; i < P; i += NT) list[i] = 0ull;
      __syncthreads();
      bitonic_desc_u64(reinterpret_cast<uint64_t*>(list), P);
    }
    const int per = (P + NT - 1) / NT, j0 = t * per;
    double loc = 0.0;
    for (int i = 0; i < per; ++i)
      if (j0 + i < nB) loc += exp_neg((double)(key_value(list[j0 + i]) - win.m));
    const BigScan sc = big_scan(loc, 0u, sh);
    double ab = Mb + sc.ex;
    uint32_t nk = 0, unsure = 0;
    for (int i = 0; i < per; ++i)
      if (j0 + i < nB) {
        const double M = S - ab;
        nk += M > A ? 1u : 0u;
        if (!(fabs(M - A) > mg) && nbx + (uint32_t)(j0 + i) >= (uint32_t)mk) unsure = 1u;
        ab += exp_neg((double)(key_value(list[j0 + i]) - win.m));
      }
    const BigScan cn = big_scan(0.0, nk | (unsure << 20), sh);
    if (cn.utot >> 20) return false;   // uniform
    nk = cn.utot;
    // min_tokens_to_keep (sampling.cpp:67-68): the top min_keep positions stay
    if (nbx + nk < (uint32_t)mk) {
      if ((uint32_t)mk > nbx + (uint32_t)nB) return false;
      nk = (uint32_t)mk - nbx;
    }
    kept = nbx + nk;
    if (kept == 0u || nB == 0) return false;
    // the last kept entry; with none kept here, everything above the list
    const uint64_t kthr = nk > 0u ? list[nk - 1u] : list[0] + 1ull;
    // subnormal kept masses: the smallest kept value decides
    if (key_value(kthr) - win.m < -690.0f) return false;
    if (t == 0) sh.kthr = kthr;
    C4S_PHASE(15);
    // the kept entries of X join their chunks' masses
    for (int j = t; j < nX; j += NT) {
      const unsigned long long e = sh.x[j];
      if (e >= kthr)
        atomicAdd(&sh.chunk[((int)~(uint32_t)e + g.off) / kChunkPos], exp_neg((double)(key_value(e) - win.m)));
    }
  }
  __syncthreads();
  C4S_PHASE(16);
  static_assert(kBigMaxChunks <= 2 * NT, "two chunks a thread");
  const double c0 = 2 * t < nch ? sh.chunk[2 * t] : 0.0, c1 = 2 * t + 1 < nch ? sh.chunk[2 * t + 1] : 0.0;
  const BigScan cs = big_scan(c0 + c1, 0u, sh);
  const double K = cs.tot;
  const uint64_t st2 = xorshift64(a.rng[row]);
  const double rr = unit_from_state(st2) * K;
  const uint32_t s0 = 1u | 4u | 16u;
  if (!(rr > 0.0)) {   // the first id satisfies r <= acc (text2semantic.cpp:161-162)
    if (t == 0) big_out(a, row, 0, true, st2, s0, kept);
    return true;
  }
  if (t == 0) sh.chunk_of = -1;
  __syncthreads();
  if ((cs.ex < rr && rr <= cs.in)) {
    const bool second = rr > cs.ex + c0;
    sh.chunk_of = 2 * t + (second ? 1 : 0);
    sh.cex = second ? cs.ex + c0 : cs.ex;
  }
  __syncthreads();
  const int ch = sh.chunk_of;
  if (ch < 0) return false;   // r past the rounded total (uniform)
  const double cex = sh.cex;
  const uint64_t kthr = dense ? 0ull : sh.kthr;
  C4S_PHASE(17);
  // that chunk's ids again, kChunkPos / NT consecutive ones a thread
  constexpr int kPer = kChunkPos / NT;
  const int first = ch * kChunkPos - g.off;
  float xv[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int id = min(max(first + t * kPer + i, 0), g.V - 1);
    xv[i] = g.dtype == 0 ? static_cast<const float*>(g.base)[id]
                         : __uint_as_float((uint32_t)static_cast<const uint16_t*>(g.base)[id] << 16);
  }
  if (c.pen_on) {   // a CSR history's bits were cleared at the start
    if (a.hist_bits) big_bits_clear<NT>(a, row, first, kChunkPos / 32, sh.bm);
    else big_bits_set<NT>(a, hs, first, kChunkPos / 32, sh.bm);
    __syncthreads();
  }
  double e[kPer], sum = 0.0;
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int id = first + t * kPer + i;
    e[i] = 0.0;
    if (id >= 0 && id < g.V) {
      const int q = t * kPer + i;
      float x = xv[i];
      if (c.pen_on && ((sh.bm[q >> 5] >> (q & 31)) & 1u)) x = x < 0 ? x * r.pen : div_rcp(x, r.rpen);
      const float z = r.z(x);
      const float d = win.fQ - floorf(z * kBigScale);
      const bool kp = dense ? z != neg_inf() : (d < (float)win.xlo || (d <= (float)win.xhi && key64(z, id) >= kthr));
      if (kp) e[i] = exp_neg((double)(z - win.m));
    }
    sum += e[i];
  }
  const BigScan ds = big_scan(sum, 0u, sh);
  if (t == 0) sh.verdict = 0;
  __syncthreads();
  const double mg = 2.0 * rel_eps(c.V) * K;
  double run = cex + ds.ex;
  const double end = cex + ds.in;
  if (sum > 0.0 && run < rr && rr <= end) {
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const double nx2 = i == kPer - 1 ? end : run + e[i];
      if (e[i] > 0.0 && run < rr && rr <= nx2) {
        sh.tok = first + t * kPer + i;
        sh.verdict = (nx2 - rr > mg && rr - run > mg) ? 1 : 0;
      }
      run = nx2;
    }
  }
  __syncthreads();
  if (!sh.verdict) return false;
  if (t == 0) big_out(a, row, sh.tok, true, st2, s0, kept);
  C4S_PHASE(18);
  return true;
}

struct BigShT {
  unsigned long long x[kBigRowCap];   // the slices' candidates
  uint32_t pre[80];
};

// Phase C of a top-k row: the slices' candidates sorted, then topk_finish.
__device__ __forceinline__ bool big_phase_c_topk(const RowsArgs& a, int row, const RowCfg& c, const BigWs& ws, int nsl,
                                                 T2Sh& ts, BigShT& sh) {
  const int t = threadIdx.x, lane = lane_id(), w = wave_id();
  uint32_t n = 0, tout = 0, bad = 0;
  for (int b = 0; b < nsl; b += kWave) {
    const int i = b + lane;
    const bool in = i < nsl;
    const BigHdr h = ws.hdr[in ? i : 0];
    const uint32_t hn = in ? h.n : 0u, inc = wave_scan_u32(hn);
    if (in && w == 0) sh.pre[i] = n + inc - hn;
    n += readlane_u32(inc, kWave - 1);
    tout = max(tout, wave_max_u32_dpp(in ? h.tout : 0u));
    bad |= __ballot(in && h.n > (uint32_t)kBigListCap) ? 1u : 0u;
  }
  const uint32_t k = (uint32_t)c.k;
  if (bad || n > (uint32_t)kBigRowCap || n < k) return false;   // uniform
  // the candidates by their distance below the largest, as topk_one_read bins
  // them; those from the k-th largest's bin up are sorted
  for (int i = t; i < kT2Buckets; i += NT) ts.hist[0][i] = 0u;
  if (t == 0) ts.n = 0u;
  __syncthreads();
  uint32_t mx = 0;
  for (int j = t, q = 0; j < (int)n; j += NT) {
    while (q + 1 < nsl && (int)sh.pre[q + 1] <= j) ++q;
    const unsigned long long e = ws.list[(size_t)q * kBigListCap + (j - (int)sh.pre[q])];
    sh.x[j] = e;
    mx = max(mx, (uint32_t)(e >> 32));
  }
  mx = wave_max_u32_dpp(mx);
  if (lane == 0) ts.wm4[w] = mx;
  __syncthreads();
  uint32_t M = 0u;
#pragma unroll
  for (int i = 0; i < NW; ++i) M = max(M, ts.wm4[i]);
  auto bin_of = [&](unsigned long long e) {   // one_pick scans from the highest bin: the bins nearest M
    return (uint32_t)(kT2Buckets - 1) - min((uint32_t)(kT2Buckets - 1), (M - (uint32_t)(e >> 32)) >> kOneBinShift);
  };
  for (int j = t; j < (int)n; j += NT) atomicAdd(&ts.hist[0][bin_of(sh.x[j])], 1u);   // the thread's own entries
  __syncthreads();
  if (!one_pick<kT2Buckets>(ts.hist[0], k, ts)) return false;
  const uint32_t bk = ts.pick[0];
  if (ts.pick[1] + ts.hist[0][bk] > (uint32_t)kT2Cap) return false;   // uniform
  for (int j = t; j < (int)n; j += NT)
    if (bin_of(sh.x[j]) >= bk) ts.list[atomicAdd(&ts.n, 1u)] = sh.x[j];
  __syncthreads();
  n = ts.n;
  uint64_t* list = ts.list;
  if (n <= (uint32_t)kRankSortMax) {
    rank_sort_desc_u64(ts.list, ts.sorted, (int)n);
    list = ts.sorted;
  } else {
    int P = 1;
    while (P < (int)n) P <<= 1;
    for (int i = (int)n + t; i < P; i += NT) ts.list[i] = 0ull;
    __syncthreads();
    bitonic_desc_u64(ts.list, P);
  }
  // no value outside the lists ties the k-th
  if (!(tout < (uint32_t)(list[k - 1] >> 32))) return false;
  T2Row src{};
  return topk_finish(a, row, c, src, ts, list, 16u);
}

// Which rows the phases take: the chain's greedy rows and sampled rows whose
// top_k is off or at most kBigMaxK, without the masked-row output.
__device__ __forceinline__ bool big_covers(const RowsArgs& a, const RowCfg& c) {
  return a.mode == 0u && !a.out_masked && (c.greedy || (c.draw && a.rng && (!c.topk_on || c.k <= kBigMaxK)));
}

__device__ __forceinline__ void big_greedy_out(const RowsArgs& a, int row, const BigWs& ws, int nsl) {
  unsigned long long best = 0ull;
  for (int i = lane_id(); i < nsl; i += kWave) best = best > ws.hdr[i].best ? best : ws.hdr[i].best;
  best = wave_max_u64_dpp(best);
  // an all -inf row: the first id
  if (threadIdx.x == 0) big_out(a, row, best ? (int)~(uint32_t)best : 0, false, 0ull, 8u | 16u, (uint32_t)a.vocab);
}

// The phases C of any row; a barrier has passed since the last use of smem.
template <int VPT>
__device__ __forceinline__ bool big_finish(const RowsArgs& a, int row, const RowCfg& c, const BigGeo& g, const BigRow& r,
                                           const BigHist& hs, const BigWs& ws, int nsl, const BigWin& win,
                                           unsigned char* smem) {
  if (c.greedy) {
    big_greedy_out(a, row, ws, nsl);
    return true;
  }
  if (c.topk_on)   // ts, then the offsets
    return big_phase_c_topk(a, row, c, ws, nsl, *reinterpret_cast<T2Sh*>(smem),
                            *reinterpret_cast<BigShT*>(smem + ((sizeof(T2Sh) + 15) & ~(size_t)15)));
  return big_phase_c<VPT>(a, row, c, g, r, hs, ws, nsl, win, *reinterpret_cast<BigShC*>(smem));
}
constexpr size_t kBigTopkBytes = ((sizeof(T2Sh) + 15) & ~(size_t)15) + sizeof(BigShT);
constexpr size_t kBigFinishBytes = kBigTopkBytes > sizeof(BigShC) ? kBigTopkBytes : sizeof(BigShC);
static_assert(sizeof(BigShA) <= kBigFinishBytes && sizeof(BigShB) <= kBigFinishBytes, "one area for every phase");

// One workgroup (NT threads) walks its row through the phases.
template <int EPV>
__device__ __forceinline__ bool big_single(const RowsArgs& a, int row, const RowCfg& c, int64_t h0, int64_t h1,
                                           unsigned char* smem) {
  constexpr int VPT = kSlice / NT;
  const BigGeo g = big_geo(a, row);
  const BigRow r = big_row(c);
  const BigHist hs = big_hist<NT>(a, h0, h1);
  const int nsl = big_slices(c.V);
  const BigWs ws = big_ws(a, row, nsl);
  BigWin win{};
  BigFetch<VPT, EPV> f;
  for (int s = 0; s < nsl; ++s) {
    big_fetch<VPT, EPV>(g, s, f);
    big_phase_a<NT, EPV>(a, row, c, g, r, hs, f, ws, s, *reinterpret_cast<BigShA*>(smem));
    __syncthreads();
  }
  if (!c.greedy && !c.topk_on) {
    BigShB& sb = *reinterpret_cast<BigShB*>(smem);
    BigMerge<NT> mf;
    big_window_fetch<NT>(ws, nsl, mf);
    if (!big_window<NT>(c, ws, nsl, sb, mf, win)) return false;
    for (int s = 0; s < nsl; ++s) {
      big_fetch<VPT, EPV>(g, s, f);
      big_phase_b<NT, EPV>(a, row, c, g, r, hs, f, ws, s, win, sb);
      __syncthreads();
    }
  }
  return big_finish<VPT>(a, row, c, g, r, hs, ws, nsl, win, smem);
}

}  // namespace
}  // namespace c4s
