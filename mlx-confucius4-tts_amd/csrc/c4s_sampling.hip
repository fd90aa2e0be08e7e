// gfx950 kernels for the c4tts Text2Semantic token-sampling path.
//
// One workgroup (1024 threads = 16 wave64) owns one row. The chain follows the
// reference order (src/t2s/text2semantic.cpp:142-166):
//   repetition penalty -> greedy ? argmax : temperature -> top_k -> top_p -> draw
// with the per-processor semantics of src/t2s/sampling.cpp:14-76 and the
// xorshift64 inverse-CDF draw of text2semantic.cpp:150-165.
//
// Exactness. Penalty, temperature and top-k are single IEEE fp32 operations or
// comparisons and are reproduced bit for bit. top_p and the draw accumulate
// double sums sequentially in the reference (ascending value order, resp. id
// order). Here those sums are formed in parallel; every decision taken from
// them (does the nucleus cut remove this position, does r <= acc hold at this
// id) is accepted only when its margin exceeds a bound on the difference
// between any sequential and any parallel evaluation (relative
// (4n+64)*2^-53 + 2^-48, which also covers a few ulp of exp(double) between
// libm implementations). Otherwise the row re-runs that step as an exact
// sequential emulation in reference order. Selections use radix passes over
// order-preserving 32-bit keys (no sort); the top_p tie order is the declared
// one: within a tie group cut by the nucleus the lower ids survive.
//
// Rows with vocab <= kLdsVocabMax are staged in LDS (values + cached double
// masses); larger rows are re-read from HBM on every pass (penalty via an LDS
// bitmap, temperature re-applied on the fly).


#include "c4s_list.hpp"
#include "c4s_step.hpp"

namespace c4s {
namespace {

// ---- kernels -------------------------------------------------------------------

// The drawn token joins the row's kept history set unless it is the stop token
// (text2semantic.cpp:333-334: a finished row appends nothing).
__device__ __forceinline__ void join_history(const RowsArgs& a, int row, int tok) {
  if (a.hist_bits && tok >= 0 && tok < a.vocab && tok != a.stop_token)
    atomicOr(&a.hist_bits[(int64_t)row * hist_words(a.vocab) + (tok >> 5)], 1u << (tok & 31));
}

__global__ __launch_bounds__(NT) void k_rows_lds(RowsArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ Scratch sh;
  const int row = blockIdx.x;
  const int V = a.vocab;
  if (a.row_active && !a.row_active[row]) {
    if (threadIdx.x == 0) a.out_tok[row] = -1;
    return;
  }
  const RowCfg c = make_cfg(a.mode, V, row, a.temp, a.top_k, a.top_p, a.pen, a.min_keep,
                            a.do_sample);
  LdsLayout L = lds_layout(smem, V);
  const int64_t roff = (int64_t)row * a.ld;
  if (a.dtype == 0) {
    RowFetch f;
    const float* p = static_cast<const float*>(a.logits) + roff;
    fetch_row(p, V, f);
    L.val = store_row(p, V, f, L.val);
  } else {
    for (int i = threadIdx.x; i < V; i += NT) L.val[i] = load_logit(a.logits, a.dtype, roff + i);
  }
  if (c.pen_on) {
    const int nw = bitmap_words(V);
    if (a.hist_bits) {   // the history set kept across steps
      const uint32_t* hb = a.hist_bits + (int64_t)row * hist_words(V);
      for (int w = threadIdx.x; w < nw; w += NT) L.bitmap[w] = w < hist_words(V) ? hb[w] : 0u;
    } else {
      for (int w = threadIdx.x; w < nw; w += NT) L.bitmap[w] = 0u;
      __syncthreads();
      const int64_t h0 = a.hist_off[row], h1 = a.hist_off[row + 1];
      for (int64_t j = h0 + threadIdx.x; j < h1; j += NT) {
        const int id = a.hist_ids[j];
        if (id < 0 || id >= V) continue;   // sampling.cpp:24
        atomicOr(&L.bitmap[id >> 5], 1u << (id & 31));
      }
    }
    __syncthreads();
    penalise_chunk(L.val, L.bitmap, V, c.pen);
  }
  __syncthreads();
  LdsRow src{L.val, L.E, V, 0u, false};
  uint64_t rng = a.rng ? a.rng[row] : 0ull;
  float* masked = a.out_masked ? a.out_masked + (int64_t)row * V : nullptr;
  uint32_t* st = a.stats ? a.stats + 4 * (int64_t)row : nullptr;
  int tok = 0;
  if (!(fast_topk_applies(c, V) &&
        fast_topk_any(L.val, V, c, sh, reinterpret_cast<unsigned char*>(L.E), rng, tok, masked, st)))
    tok = run_chain(src, sh, c, rng, masked, st);
  if (threadIdx.x == 0) {
    a.out_tok[row] = tok;
    if (c.draw && a.rng) a.rng[row] = rng;
    join_history(a, row, tok);
  }
}

// ---- large vocabularies: top_k in two passes -----------------------------------------
//
// A sampled row with top_k in [1, kT2MaxK] (e.g. 256 rows x V = 151936, k = 50)
// does not need the whole row after top_k: every entry below the k-th largest
// value is -inf from there on (sampling.cpp:30-40), so top_p (sampling.cpp:
// 42-71) and the draw (text2semantic.cpp:150-165) only see the survivors.
// Pass 1 reads the row once (penalty, temperature) for its maximum and a
// histogram of the top kT2Bits bits of the order-preserving value keys, which
// locates the bucket b* of the k-th largest value; pass 2 reads it again and
// collects every entry of b* and above (at most kT2Cap) with its id. Sorted,
// their first k give the threshold (ties kept). Wave 0 then replays top_p and
// the draw on the survivors sequentially in double, in the reference's order
// (top_p ascending by value, equal values higher id first; the draw in id
// order), so the sums are the reference's own: the -inf positions add 0.
constexpr int kT2Bits = 11;
constexpr int kT2Buckets = 1 << kT2Bits;
constexpr int kT2Copies = 4;        // histogram copies (by wave) to spread the LDS atomics
constexpr int kT2Cap = 2 * NT;      // candidates the sort takes
constexpr int kT2MaxK = NT;
constexpr int kT2MaxV = 1 << 19;    // above: the LDS holds the history bitmap only

struct T2Sh {
  uint32_t hist[kT2Copies][kT2Buckets];
  uint64_t list[kT2Cap];
  uint64_t sorted[256];             // the rank sort's result (list itself after the bitonic network)
  double e[kT2Cap];                 // the draw's masses in id order
  uint32_t wsum[NW];
  float wmax[NW];
  uint32_t wm4[NW];                 // one read: per-wave largest candidate key
  uint32_t n;
  int bstar;
  uint32_t nge, nkeep;
  int tok;
  uint32_t dex;                     // the draw replayed sequentially (1) or not
  uint32_t pick[2];                 // one read: the picked candidate's bin and the candidates above it
  uint32_t nq;                      // one read: gathered entries whose penalised key reaches the bound
};

__host__ __device__ __forceinline__ size_t t2_offset(int V) { return ((size_t)4 * ((V + 31) / 32) + 15) & ~(size_t)15; }

constexpr int kRankSortMax = 256;   // above: the bitonic network
// Descending sort of n <= kRankSortMax distinct 64-bit keys by rank counting
// (each key's place is the count of keys above it) into `out`; one barrier. The
// four lanes of a quad share a key and count over every fourth entry each (a
// thread a key: 3.6k cycles for the 80 entries of a top_k 50 row).
__device__ __forceinline__ void rank_sort_desc_u64(const uint64_t* buf, uint64_t* out, int n) {
  static_assert(4 * kRankSortMax == NT, "a quad a key");
  const int t = threadIdx.x, nS = __builtin_amdgcn_readfirstlane(n), q = t & 3, i = t >> 2;
  if (__builtin_amdgcn_readfirstlane(i & ~15) < nS) {   // waves whose keys all lie past n
    const uint64_t mine = buf[min(i, nS - 1)];
    uint32_t r = 0;
    int j = 0;
    for (; j + 16 <= nS; j += 16) {
      uint64_t o[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) o[u] = buf[j + 4 * u + q];
#pragma unroll
      for (int u = 0; u < 4; ++u) r += o[u] > mine ? 1u : 0u;
    }
    for (; j < nS; j += 4)
      if (j + q < nS) r += buf[j + q] > mine ? 1u : 0u;
    r += xor_lane_u32<1>(r);
    r += xor_lane_u32<2>(r);
    if (q == 0 && i < nS) out[r] = mine;
  }
  __syncthreads();
}

// In-buffer descending bitonic sort of P (a power of two) 64-bit keys by the
// NT threads of the workgroup.
__device__ void bitonic_desc_u64(uint64_t* buf, int P) {
  for (int k = 2; k <= P; k <<= 1) {
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int t = threadIdx.x; t < (P >> 1); t += NT) {
        const int i = (t / j) * 2 * j + (t % j);
        const int pi = i + j;
        const uint64_t x = buf[i], y = buf[pi];
        const bool down = (i & k) == 0;
        if ((x < y) == down) { buf[i] = y; buf[pi] = x; }
      }
      __syncthreads();
    }
  }
}

// The row's value at id i after penalty and temperature (sampling.cpp:19-28,
// 14-17), as the multi-pass chain computes it.
struct T2Row {
  const float* xf;
  const uint16_t* xb;
  const uint32_t* bitmap;
  bool pen_on, temp_on;
  float pen, temp;
  double rpen, rtemp;   // fl64(1 / pen), fl64(1 / temp)
  __device__ __forceinline__ float z(int i, float x) const {
    if (pen_on && ((bitmap[i >> 5] >> (i & 31)) & 1u)) x = (x < 0) ? x * pen : div_rcp(x, rpen);
    return temp_on ? div_rcp(x, rtemp) : x;
  }
  // f(i, z) for every id, each by one thread: 16-byte loads over the aligned body
  template <class F>
  __device__ __forceinline__ void each(int V, F&& f) const {
    const int t = threadIdx.x;
    if (xf) {
      const RowShape rs = row_shape(xf, V);
      const float4* p4 = reinterpret_cast<const float4*>(xf + rs.head);
      for (int q = t; q < rs.nq; q += NT) {
        const float4 v = p4[q];
        const int i = rs.head + 4 * q;
        f(i, z(i, v.x));
        f(i + 1, z(i + 1, v.y));
        f(i + 2, z(i + 2, v.z));
        f(i + 3, z(i + 3, v.w));
      }
      if (t < rs.head) f(t, z(t, xf[t]));
      else if (t < rs.head + rs.tail) {
        const int i = rs.head + 4 * rs.nq + (t - rs.head);
        f(i, z(i, xf[i]));
      }
    } else {
      for (int i = t; i < V; i += NT) f(i, z(i, __uint_as_float((uint32_t)xb[i] << 16)));
    }
  }
};

// ---- one read of the row (fp32 rows, penalty >= 1) ----
//
// Each thread streams its ids once (16-byte loads, U of them in flight) and
// keeps its four largest entries as packed keys: the top 23 bits of the
// order-preserving key of the raw value x, then a 9-bit index of the entry
// in the thread's stream (3 v_med3 and 1 v_max a value, no LDS atomics). The
// penalty only lowers a value (penalty >= 1, sampling.cpp:26) and fl(y / T) is
// monotone in y, so the raw keys bound the penalised and divided ones from
// above. One pick over the 4 NT candidates, binned by their distance below
// the largest, gives Q, the 23-bit prefix of the lowest key in the bin of the
// (k + kOneSlack)-th largest candidate (the slack leaves room for entries the
// penalty takes below Q). Every entry whose raw prefix reaches Q is gathered:
// from the four of a thread whose fourth lies below Q, else from its stream
// read again by its wave; each is read again (a few cache lines), penalised
// and divided exactly, and goes to ts.list. The rest of the row stays out of
// the top k when at least k gathered entries still reach Q after their
// penalty (then the k-th largest value is at or above Q's smallest key, and
// every entry at or above it was gathered; otherwise the pick is taken again
// deeper down) and no value below Q can tie the k-th quotient (checked once
// the list is sorted). Returns false, with nothing but the work area written,
// when a check fails: the two passes over the row decide then.
constexpr int kOneIdxBits = 9;
constexpr uint32_t kOneEdge = (1u << kOneIdxBits) - 1;   // index of the thread's unaligned head / tail entry
constexpr int kOneUnroll = 8;
constexpr uint32_t kOneSlack = 16;
constexpr int kOneBinShift = 15;   // candidate bins of 2^15 packed keys: 1/256 of a binade
// 16-byte loads a thread; the unrolled loop rounds them up to kOneUnroll, and
// every index it makes (padding past the row included) stays below kOneEdge
constexpr int kOneMaxIters = 120;
static_assert(kOneMaxIters % kOneUnroll == 0 && 4 * kOneMaxIters - 1 < (int)kOneEdge, "indices below the edge's");
constexpr int kOneMaxV = 4 * NT * kOneMaxIters;

__device__ __forceinline__ uint32_t one_pack(float x, uint32_t idx) {
  return (fkey(x) & ~kOneEdge) | idx;
}
// The median of three (v_med3_u32): max(lo, min(hi, e)) when lo <= hi, which
// the compiler cannot know here.
__device__ __forceinline__ uint32_t med3_u32(uint32_t a, uint32_t b, uint32_t c) {
  uint32_t r;
  asm("v_med3_u32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
// t0 >= t1 >= t2 >= t3 keeps the four largest (the order holds from the start, all zero)
__device__ __forceinline__ void one_insert(uint32_t& t0, uint32_t& t1, uint32_t& t2, uint32_t& t3, uint32_t e) {
  t3 = med3_u32(t3, t2, e);
  t2 = med3_u32(t2, t1, e);
  t1 = med3_u32(t1, t0, e);
  t0 = max(t0, e);
}

// Bin of `hist` (nb bins scanned from the top, nb / NT a thread) holding the
// m-th largest counted key, and the count above it, into ts.pick; false when
// fewer than m keys were counted. Two barriers.
template <int NB>
__device__ __forceinline__ bool one_pick(const uint32_t* hist, uint32_t m, T2Sh& ts) {
  constexpr int PB = NB / NT;
  const int t = threadIdx.x, lane = lane_id(), w = wave_id();
  uint32_t cb[PB], loc = 0;
#pragma unroll
  for (int i = 0; i < PB; ++i) { cb[i] = hist[NB - 1 - PB * t - i]; loc += cb[i]; }
  const uint32_t inc = wave_scan_u32(loc);
  if (lane == kWave - 1) ts.wsum[w] = inc;
  __syncthreads();
  uint32_t ex = inc - loc, total = 0;
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    const uint32_t x = ts.wsum[i];
    ex += (i < w) ? x : 0u;
    total += x;
  }
  if (total < m) return false;   // uniform
  if (ex < m && ex + loc >= m) {
    uint32_t run = ex;
#pragma unroll
    for (int i = 0; i < PB; ++i) {
      if (run < m && run + cb[i] >= m) { ts.pick[0] = (uint32_t)(NB - 1 - PB * t - i); ts.pick[1] = run; }
      run += cb[i];
    }
  }
  __syncthreads();
  return true;
}

// Buffer resource of `bytes` bytes from p (raw: byte offsets; a load past
// the end returns zeros without an access). Loads through one issue on every
// path, so that the waits of later loads count them exactly.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t raw_rsrc(const void* p, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, bytes, 0x00020000);
}
__device__ __forceinline__ float4 rsrc_load16(__amdgpu_buffer_rsrc_t r, int off) {
  return __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}

// The first kOneUnroll 16-byte loads of this thread's stream of an f32 row
// (the layout of topk_one_read), issued before the row's set-up so that they
// are in flight meanwhile; with `on` false nothing is read (xf need only be
// a pointer).
struct OneFirst {
  float4 v[kOneUnroll];
};
__device__ __forceinline__ void one_first(const float* xf, int V, bool on, OneFirst& f) {
  const RowShape rs = row_shape(xf, V);
  const __amdgpu_buffer_rsrc_t r = raw_rsrc(xf + rs.head, on ? 16 * rs.nq : 0);
  const float ninf = neg_inf();
#pragma unroll
  for (int u = 0; u < kOneUnroll; ++u) {
    const int q = threadIdx.x + NT * u;
    const float4 v = rsrc_load16(r, 16 * q);
    f.v[u] = (q < rs.nq) ? v : make_float4(ninf, ninf, ninf, ninf);
  }
}

__device__ __forceinline__ bool topk_one_read(const RowsArgs& a, const RowCfg& c, const float* xf, const uint32_t* bitmap,
                              T2Sh& ts, uint32_t& qkey, const OneFirst& first) {
  const int V = c.V, t = threadIdx.x, w = wave_id(), lane = lane_id();
  const RowShape rs = row_shape(xf, V);
  const float4* p4 = reinterpret_cast<const float4*>(xf + rs.head);
  const float ninf = neg_inf();
  uint32_t t0 = 0u, t1 = 0u, t2 = 0u, t3 = 0u;   // 0: below every packed key
  const int iters = (rs.nq + NT - 1) / NT;
  auto take = [&](const float4 (&v)[kOneUnroll], int j0) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kOneUnroll; ++u) {
      const uint32_t i0 = 4u * (uint32_t)(j0 + u);
      one_insert(t0, t1, t2, t3, one_pack(v[u].x, i0));
      one_insert(t0, t1, t2, t3, one_pack(v[u].y, i0 + 1u));
      one_insert(t0, t1, t2, t3, one_pack(v[u].z, i0 + 2u));
      one_insert(t0, t1, t2, t3, one_pack(v[u].w, i0 + 3u));
    }
  };
  take(first.v, 0);   // loads 0 .. kOneUnroll - 1 (past the row: -inf)
  for (int j0 = kOneUnroll; j0 < iters; j0 += kOneUnroll) {
    float4 v[kOneUnroll];
#pragma unroll
    for (int u = 0; u < kOneUnroll; ++u) {
      const int q = t + NT * (j0 + u);
      v[u] = (q < rs.nq) ? p4[q] : make_float4(ninf, ninf, ninf, ninf);
    }
    take(v, j0);
  }
  const int edge = (t < rs.head) ? t : ((t < rs.head + rs.tail) ? rs.head + 4 * rs.nq + (t - rs.head) : -1);
  if (edge >= 0) one_insert(t0, t1, t2, t3, one_pack(xf[edge], kOneEdge));
  C4S_PHASE(8);
  auto id_of = [&](uint32_t e) -> int {
    const uint32_t ix = e & kOneEdge;
    if (ix == kOneEdge) return edge;
    return rs.head + 4 * (t + NT * (int)(ix >> 2)) + (int)(ix & 3u);
  };
  auto valid = [&](uint32_t e) {   // a real entry of the row (not padding past it)
    const uint32_t ix = e & kOneEdge;
    return e != 0u && (ix == kOneEdge ? edge >= 0 : t + NT * (int)(ix >> 2) < rs.nq);
  };
  // The candidates by their distance below the largest, M: bin b (from the
  // top) holds the packed keys in (M - (b + 1) 2^S, M - b 2^S], 1/256 of a
  // binade, the last bin everything farther down (the LDS atomics spread over
  // many bins where a histogram of the keys' top bits had a few).
  for (int i = t; i < kT2Buckets; i += NT) ts.hist[0][i] = 0u;
  {
    const uint32_t m0 = wave_max_u32(t0);
    if (lane == 0) ts.wm4[w] = m0;
    if (t == 0) { ts.n = 0u; ts.nq = 0u; }
  }
  __syncthreads();
  uint32_t M = 0u;
#pragma unroll
  for (int i = 0; i < NW; ++i) M = max(M, ts.wm4[i]);
  const uint32_t tk[4] = {t0, t1, t2, t3};
  uint32_t* h1 = ts.hist[0];
#pragma unroll
  for (int i = 0; i < 4; ++i)   // one_pick scans from the highest bin: the bins nearest M
    if (tk[i]) atomicAdd(&h1[(kT2Buckets - 1) - min((uint32_t)(kT2Buckets - 1), (M - tk[i]) >> kOneBinShift)], 1u);
  __syncthreads();
  C4S_PHASE(1);
  const uint32_t k = (uint32_t)c.k;
  uint32_t kb = k + kOneSlack;
  for (int attempt = 0;; ++attempt) {
    if (!one_pick<kT2Buckets>(h1, kb, ts)) return false;   // fewer candidates than that (uniform)
    const uint32_t bfar = (kT2Buckets - 1) - ts.pick[0];   // bins below M
    const int64_t lo = (int64_t)M - ((int64_t)(bfar + 1) << kOneBinShift) + 1;
    // the bound: the prefix of the lowest key of that bin, above -inf's
    if (bfar >= (uint32_t)(kT2Buckets - 1) || lo <= (int64_t)kKeyNegInf) return false;
    const uint32_t Q = (uint32_t)lo >> kOneIdxBits;
    const uint32_t kq = Q << kOneIdxBits;   // smallest key with prefix Q
    C4S_PHASE(2);
    // every entry whose raw prefix reaches Q, with its penalised
    // (sampling.cpp:26) and divided (:16) value
    uint32_t reach = 0u;
    auto push = [&](int id, float x) {
      float y = x;
      if (c.pen_on && ((bitmap[id >> 5] >> (id & 31)) & 1u)) y = (y < 0) ? y * c.pen : y / c.pen;
      reach += fkey(y) >= kq ? 1u : 0u;
      const float z = c.temp_on ? y / c.temp : y;
      const uint32_t slot = atomicAdd(&ts.n, 1u);
      if (slot < (uint32_t)kT2Cap) ts.list[slot] = ((uint64_t)fkey(z) << 32) | (uint32_t)~(uint32_t)id;
    };
    // A thread whose fourth candidate lies below Q holds every such entry of
    // its stream among its four; another may hold more: its wave reads that
    // thread's stream again (16-byte loads, one a lane).
    const bool redo = (t3 >> kOneIdxBits) >= Q;
    if (!redo) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (valid(tk[i]) && (tk[i] >> kOneIdxBits) >= Q) {
          const int id = id_of(tk[i]);
          push(id, xf[id]);
        }
    }
    for (uint64_t rm = __ballot(redo); rm; rm &= rm - 1) {
      const int tf = w * kWave + (__ffsll((unsigned long long)rm) - 1);
      for (int j = lane; j < iters; j += kWave) {
        const int q = tf + NT * j;
        if (q < rs.nq) {
          const float4 v = p4[q];
          const int i0 = rs.head + 4 * q;
          if ((fkey(v.x) >> kOneIdxBits) >= Q) push(i0, v.x);
          if ((fkey(v.y) >> kOneIdxBits) >= Q) push(i0 + 1, v.y);
          if ((fkey(v.z) >> kOneIdxBits) >= Q) push(i0 + 2, v.z);
          if ((fkey(v.w) >> kOneIdxBits) >= Q) push(i0 + 3, v.w);
        }
      }
      const int ef = (tf < rs.head) ? tf : ((tf < rs.head + rs.tail) ? rs.head + 4 * rs.nq + (tf - rs.head) : -1);
      if (lane == 0 && ef >= 0 && (fkey(xf[ef]) >> kOneIdxBits) >= Q) push(ef, xf[ef]);
    }
    reach = wave_sum_u32(reach);
    if (lane == 0 && reach) atomicAdd(&ts.nq, reach);
    __syncthreads();
    C4S_PHASE(3);
    const uint32_t n = ts.n, nq = ts.nq;
    if (n > (uint32_t)kT2Cap) return false;   // uniform
    if (nq >= k) {
      qkey = kq;
      return true;
    }
    // fewer than k reach Q after their penalty: a bound further down
    if (attempt == 2) return false;
    __syncthreads();   // every thread has read ts.n and ts.nq
    if (t == 0) { ts.n = 0u; ts.nq = 0u; }
    __syncthreads();
    kb *= 4u;
  }
}

// top_k, top_p and the draw on the sorted candidates list[0, ts.n) (every
// entry at or above the k-th largest value among them); returns true.
__device__ __forceinline__ bool topk_finish(const RowsArgs& a, int row, const RowCfg& c, const T2Row& src, T2Sh& ts,
                            uint64_t* list, uint32_t stat_bits) {
  const int V = c.V, t = threadIdx.x, w = wave_id(), lane = lane_id();
  const float ninf = neg_inf();
  const uint32_t k = (uint32_t)c.k;
  const int n = (int)ts.n;
  // top_k: every entry with the k-th largest value or above survives
  const uint32_t kkey = (uint32_t)(list[k - 1] >> 32);
  if (w == 0) {
    int ns = (int)k;
    for (int more = kWave; more == kWave && ns < n; ns += more)   // a run of ties ends the survivors
      more = __popcll(__ballot(ns + lane < n && (uint32_t)(list[min(ns + lane, n - 1)] >> 32) >= kkey));
    const float vmax = kfloat((uint32_t)(list[0] >> 32));
    int nkeep = ns, tok = -2;   // -2: not decided here
    uint32_t dex = 0u;
    if (ns <= kWave) {
      // At most 64 survivors, one a lane in value order: top_p and the draw
      // with sums formed in parallel, each decision farther than rel_eps from
      // its boundary or taken by the sequential sums below (top_p) or the
      // sequential replay of lane_draw (the draw), as the candidate-list step
      // does. Survivor j's mass is exp(z_j - vmax), vmax the first survivor's.
      const bool sv = lane < ns;
      const uint64_t ent = list[sv ? lane : 0];
      const float zs = sv ? kfloat((uint32_t)(ent >> 32)) : ninf;
      const int ids = (int)~(uint32_t)ent;
      const double e = sv ? exp((double)(zs - vmax)) : 0.0;
      // the sequential path for subnormal masses and below the draw's -1e30 floor
      bool ok = !__ballot(sv && e < 0x1p-1000) && !(vmax < -1e30f);
      const double thr = 1.0 - (double)c.p;
      if (ok && c.topp_on && thr >= 0.0) {
        // entry j removed iff the mass at or below it in ascending order,
        // M = S - (mass above it), is <= thr S (sampling.cpp:60-65)
        const double S = wave_sum_dpp(e);
        const double M = S - (wave_scan_f64(e) - e);
        bool rem, unsure = false;
        if (thr == 0.0) {
          rem = sv && M == 0.0;
        } else {
          const double A = thr * S;
          rem = sv && M <= A;
          unsure = sv && lane >= c.min_keep && !(fabs(M - A) > rel_eps(V) * fmax(M, A));
        }
        if (__ballot(unsure)) {
          ok = false;
        } else {
          nkeep = ns - __popcll(__ballot(rem));
          const int mk = min(max(0, c.min_keep), ns);   // sampling.cpp:67-68
          if (nkeep < mk) nkeep = mk;
        }
      }
      if (ok) {   // text2semantic.cpp:150-165 over the kept survivors in id order
        const uint64_t st2 = xorshift64(a.rng[row]);
        tok = lane_draw<19>(sv && lane < nkeep, ids, ids, e, unit_from_state(st2), V, dex);
      } else {
        nkeep = ns;
      }
    }
    if (tok == -2 && c.topp_on) {
      // sampling.cpp:52-65 in ascending order (list position ns - 1 - j)
      double total = 0.0;
      for (int base = 0; base < ns; base += kWave) {
        const int j = base + lane;
        const double e = j < ns ? exp((double)(kfloat((uint32_t)(list[ns - 1 - j] >> 32)) - vmax)) : 0.0;
        total = seq_sum_lanes(total, e, min(kWave, ns - base));
      }
      const double thr = 1.0 - (double)c.p;
      double cum = 0.0;
      int removed = 0;
      bool stop = false;
      for (int base = 0; base < ns && !stop; base += kWave) {
        const int j = base + lane;
        const double q = j < ns ? exp((double)(kfloat((uint32_t)(list[ns - 1 - j] >> 32)) - vmax)) / total : 0.0;
        removed = base + seq_cut_lanes(cum, q, min(kWave, ns - base), thr, stop);
      }
      nkeep = ns - removed;
      const int mk = min(max(0, c.min_keep), ns);   // sampling.cpp:67-68
      if (nkeep < mk) nkeep = mk;
    }
    if (lane == 0) {
      ts.nkeep = (uint32_t)nkeep;
      ts.tok = tok;
      ts.dex = dex;
    }
  }
  __syncthreads();
  const int nkeep = (int)ts.nkeep;
  C4S_PHASE(5);
  // the state before the draw: kept values, -inf elsewhere
  if (a.out_masked) {
    float* mrow = a.out_masked + (int64_t)row * V;
    for (int i = t; i < V; i += NT) mrow[i] = ninf;
    __syncthreads();
    for (int j = t; j < nkeep; j += NT) {   // the row's own value (the key folds -0 onto +0)
      const int i = (int)~(uint32_t)list[j];
      mrow[i] = src.z(i, src.xf ? src.xf[i] : __uint_as_float((uint32_t)src.xb[i] << 16));
    }
  }
  if (ts.tok != -2) {   // drawn above
    if (t == 0) {
      const int tok = ts.tok;
      a.out_tok[row] = tok;
      a.rng[row] = xorshift64(a.rng[row]);
      join_history(a, row, tok);
      if (a.stats) {
        uint32_t* st = a.stats + 4 * (int64_t)row;
        st[0] = 1u | 2u | 4u | 32u | stat_bits;
        st[1] = 0u;
        st[2] = ts.dex;
        st[3] = (uint32_t)nkeep;
      }
    }
    return true;
  }
  // the kept entries in id order: (~id) as the high half sorts descending by it
  int Pk = 1;
  while (Pk < nkeep) Pk <<= 1;
  __syncthreads();
  const int Ps = nkeep <= kRankSortMax ? nkeep : Pk;
  for (int j = t; j < Ps; j += NT) {
    const uint64_t v = j < nkeep ? list[j] : 0ull;
    list[j] = j < nkeep ? (((uint64_t)(uint32_t)v << 32) | (v >> 32)) : 0ull;
  }
  __syncthreads();
  if (nkeep <= kRankSortMax) {
    uint64_t* out = list == ts.list ? ts.sorted : ts.list;
    rank_sort_desc_u64(list, out, nkeep);
    list = out;
  } else {
    bitonic_desc_u64(list, Pk);
  }
  C4S_PHASE(6);
  if (w == 0) {
    // text2semantic.cpp:150-165 over the kept entries in id order (the maximum
    // starts from -1e30f; -inf positions add 0)
    float m = -1e30f;
    for (int j = lane; j < nkeep; j += kWave) m = fmaxf(m, kfloat((uint32_t)list[j]));
    m = wave_max_f32(m);
    double total = 0.0;
    for (int base = 0; base < nkeep; base += kWave) {
      const int j = base + lane;
      const float zj = j < nkeep ? kfloat((uint32_t)list[j]) : ninf;
      const double e = (j < nkeep && zj != ninf) ? exp((double)(zj - m)) : 0.0;
      if (j < nkeep) ts.e[j] = e;
      total = seq_sum_lanes(total, e, min(kWave, nkeep - base));
    }
    const uint64_t st2 = xorshift64(a.rng[row]);
    const double r = unit_from_state(st2) * total;
    int tok = V - 1;   // no id reached r (text2semantic.cpp:160)
    double acc = 0.0;
    bool done = false;
    for (int base = 0; base < nkeep && !done; base += kWave) {
      const int j = base + lane;
      const double e = j < nkeep ? ts.e[j] : 0.0;
      const int q = seq_find_lanes(acc, e, min(kWave, nkeep - base), r);
      if (q >= 0) {
        tok = (int)~(uint32_t)(list[base + q] >> 32);
        done = true;
      }
    }
    if (lane == 0) {
      a.out_tok[row] = tok;
      a.rng[row] = st2;
      join_history(a, row, tok);
      if (a.stats) {
        uint32_t* st = a.stats + 4 * (int64_t)row;
        st[0] = 1u | 2u | 4u | 32u | stat_bits;
        st[1] = 0u;
        st[2] = 0u;
        st[3] = (uint32_t)nkeep;
      }
    }
  }
  C4S_PHASE(7);
  return true;
}

// Returns false (nothing written) when the survivors' bucket holds more than
// the sort takes; the multi-pass chain decides the row then.
__device__ __forceinline__ bool topk_two_pass(const RowsArgs& a, int row, const RowCfg& c, const T2Row& src, T2Sh& ts,
                                              const OneFirst& first) {
  const int V = c.V, t = threadIdx.x, w = wave_id(), lane = lane_id();
  const float ninf = neg_inf();
  const uint32_t k = (uint32_t)c.k;
  // one read of the row when its checks pass
  uint32_t qkey = 0u;
  bool one = src.xf && V <= kOneMaxV && (!c.pen_on || c.pen >= 1.0f) &&
             topk_one_read(a, c, src.xf, src.bitmap, ts, qkey, first);
  uint64_t* list = ts.list;
  if (one) {
    const int n = (int)ts.n;
    if (n <= kRankSortMax) {
      rank_sort_desc_u64(ts.list, ts.sorted, n);
      list = ts.sorted;
    } else {
      int P = 1;
      while (P < n) P <<= 1;
      for (int i = n + t; i < P; i += NT) ts.list[i] = 0ull;
      __syncthreads();
      bitonic_desc_u64(ts.list, P);
    }
    C4S_PHASE(4);
    // no value below the bound ties the k-th quotient (the largest of them, divided)
    if (c.temp_on && !(fkey(kfloat(qkey - 1u) / c.temp) < (uint32_t)(list[k - 1] >> 32))) one = false;
  }
  if (one) return topk_finish(a, row, c, src, ts, list, 64u);
  __syncthreads();   // the work area is free again
  for (int i = t; i < kT2Copies * kT2Buckets; i += NT) (&ts.hist[0][0])[i] = 0u;
  if (t == 0) ts.n = 0u;
  __syncthreads();
  // pass 1: maximum and histogram
  uint32_t* hist = ts.hist[w % kT2Copies];
  float lmax = ninf;
  src.each(V, [&](int, float zi) {
    lmax = fmaxf(lmax, zi);
    atomicAdd(&hist[fkey(zi) >> (32 - kT2Bits)], 1u);
  });
  lmax = wave_max_f32(lmax);
  if (lane == 0) ts.wmax[w] = lmax;
  __syncthreads();
  // b*: thread t takes buckets 2047 - 2t (higher) and 2046 - 2t; counts from the top
  const int bh = kT2Buckets - 1 - 2 * t, bl = bh - 1;
  uint32_t ch = 0, cl = 0;
#pragma unroll
  for (int q = 0; q < kT2Copies; ++q) { ch += ts.hist[q][bh]; cl += ts.hist[q][bl]; }
  const uint32_t inc = wave_scan_u32(ch + cl);
  if (lane == kWave - 1) ts.wsum[w] = inc;
  __syncthreads();
  uint32_t ex = inc - (ch + cl);
  for (int i = 0; i < w; ++i) ex += ts.wsum[i];
  if (ex < k && k <= ex + ch) { ts.bstar = bh; ts.nge = ex + ch; }
  else if (ex + ch < k && k <= ex + ch + cl) { ts.bstar = bl; ts.nge = ex + ch + cl; }
  __syncthreads();
  const int bstar = ts.bstar;
  const uint32_t nge = ts.nge;
  if (nge > (uint32_t)kT2Cap) return false;   // uniform
  // pass 2: the candidates (bucket >= b*)
  src.each(V, [&](int i, float zi) {
    const uint32_t key = fkey(zi);
    if ((int)(key >> (32 - kT2Bits)) >= bstar) {
      const uint32_t slot = atomicAdd(&ts.n, 1u);
      ts.list[slot] = ((uint64_t)key << 32) | (uint32_t)~(uint32_t)i;
    }
  });
  __syncthreads();
  const int n = (int)ts.n;   // == nge
  int P = 1;
  while (P < n) P <<= 1;
  for (int i = n + t; i < P; i += NT) ts.list[i] = 0ull;
  __syncthreads();
  bitonic_desc_u64(ts.list, P);
  return topk_finish(a, row, c, src, ts, ts.list, 0u);
}

}  // namespace
}  // namespace c4s

#include "c4s_big.hpp"

namespace c4s {
namespace {

// A row's flags, parameters and history offsets by scalar loads, all issued
// before any waits for them (a byte flag read as its aligned word: flag_byte);
// false for an inactive row.
__device__ __forceinline__ bool global_cfg(const RowsArgs& a, int row, RowCfg& c, int64_t& h0, int64_t& h1) {
  h0 = h1 = 0;
  if (a.hist_off && !a.hist_bits) {
    h0 = a.hist_off[row];
    h1 = a.hist_off[row + 1];
  }
  const bool act = a.row_active ? flag_byte(a.row_active, row) : true;
  const bool sample = a.do_sample ? flag_byte(a.do_sample, row) : true;
  const float pv = a.pen ? a.pen[row] : 1.0f, tv = a.temp ? a.temp[row] : 1.0f;
  const int32_t kv = a.top_k ? a.top_k[row] : 0, mv = a.min_keep ? a.min_keep[row] : 1;
  const float ppv = a.top_p ? a.top_p[row] : 1.0f;
  c = make_cfg_vals(a.mode, a.vocab, pv, tv, kv, ppv, mv, (a.mode & kCustom) || sample);
  if (!c.pen_on) h0 = h1 = 0;
  return act;
}

// The general path of one row (the whole workgroup): the top-k reads where
// they apply, else the multi-pass chain re-reading the row.
__device__ __forceinline__ void rows_global_row(const RowsArgs& a, int row, const RowCfg& c, int64_t h0, int64_t h1,
                                                unsigned char* smem, Scratch& sh) {
  const int V = a.vocab;
  const int64_t roff = (int64_t)row * a.ld;
  // The history's first ids (four a thread), then, for a row that the top-k
  // read takes, that read's first loads: in flight during the set-up (loads
  // complete in issue order, so the ids come first)
  constexpr int kPreIds = 4;
  const bool csr = c.pen_on && !a.hist_bits;
  int hid[kPreIds];
  {
    const int nb = (int)min(h1 - h0, (int64_t)NT * kPreIds) * 4;   // the first ids' bytes
    const __amdgpu_buffer_rsrc_t r = raw_rsrc(csr ? a.hist_ids + h0 : a.out_tok, nb);
#pragma unroll
    for (int i = 0; i < kPreIds; ++i) {
      const int jo = threadIdx.x + NT * i;
      const int id = __builtin_amdgcn_raw_buffer_load_b32(r, 4 * jo, 0, 0);
      hid[i] = 4 * jo < nb ? id : -1;
    }
  }
  const bool one_row = c.draw && c.topk_on && c.k <= kT2MaxK && V <= kT2MaxV && a.rng && a.dtype == 0 &&
                       V <= kOneMaxV && (!c.pen_on || c.pen >= 1.0f);
  OneFirst first;
  one_first(static_cast<const float*>(a.logits) + (one_row ? roff : 0), V, one_row, first);
  uint32_t* bitmap = reinterpret_cast<uint32_t*>(smem);
  const int nw = (V + 31) / 32;
  for (int w = threadIdx.x; w < nw; w += NT) bitmap[w] = 0u;
  __syncthreads();
  if (c.pen_on) {
    if (a.hist_bits) {   // the history set kept across steps
      const uint32_t* hb = a.hist_bits + (int64_t)row * hist_words(V);
      for (int w = threadIdx.x; w < nw; w += NT) bitmap[w] = hb[w];
    } else {
#pragma unroll
      for (int i = 0; i < kPreIds; ++i)
        if (hid[i] >= 0 && hid[i] < V) atomicOr(&bitmap[hid[i] >> 5], 1u << (hid[i] & 31));
      for (int64_t j = h0 + threadIdx.x + (int64_t)NT * kPreIds; j < h1; j += NT) {
        const int id = a.hist_ids[j];
        if (id < 0 || id >= V) continue;
        atomicOr(&bitmap[id >> 5], 1u << (id & 31));
      }
    }
    __syncthreads();
  }
  C4S_PHASE(0);
  if (c.draw && c.topk_on && c.k <= kT2MaxK && V <= kT2MaxV && a.rng) {
    T2Row tr;
    tr.xf = a.dtype == 0 ? static_cast<const float*>(a.logits) + roff : nullptr;
    tr.xb = a.dtype == 1 ? static_cast<const uint16_t*>(a.logits) + roff : nullptr;
    tr.bitmap = bitmap;
    tr.pen_on = c.pen_on;
    tr.pen = c.pen;
    tr.temp_on = c.temp_on;
    tr.temp = c.temp;
    tr.rpen = 1.0 / (double)c.pen;
    tr.rtemp = 1.0 / (double)c.temp;
    if (topk_two_pass(a, row, c, tr, *reinterpret_cast<T2Sh*>(smem + t2_offset(V)), first)) return;
    __syncthreads();
  }
  GlobalRow src;
  src.xf = a.dtype == 0 ? static_cast<const float*>(a.logits) + roff : nullptr;
  src.xb = a.dtype == 1 ? static_cast<const uint16_t*>(a.logits) + roff : nullptr;
  src.V = V;
  src.bitmap = bitmap;
  src.pen_on = c.pen_on;
  src.pen = c.pen;
  src.temp_on = false;
  src.temp = 1.0f;
  src.thr_key = 0u;
  src.topk_on = false;
  src.sortbuf = a.sort_ws + (int64_t)row * a.sort_ws_stride;
  src.sortcap = (uint32_t)(a.sort_ws_stride * 4);
  uint64_t rng = a.rng ? a.rng[row] : 0ull;
  float* masked = a.out_masked ? a.out_masked + (int64_t)row * V : nullptr;
  uint32_t* st = a.stats ? a.stats + 4 * (int64_t)row : nullptr;
  const int tok = run_chain(src, sh, c, rng, masked, st);
  if (threadIdx.x == 0) {
    a.out_tok[row] = tok;
    if (c.draw && a.rng) a.rng[row] = rng;
    join_history(a, row, tok);
  }
}
// Whether the top-k read in one pass over the row takes it (fp32, penalty >= 1).
__device__ __forceinline__ bool one_read_applies(const RowsArgs& a, const RowCfg& c) {
  return c.draw && c.topk_on && c.k <= kT2MaxK && a.rng && a.dtype == 0 && c.V <= kOneMaxV &&
         (!c.pen_on || c.pen >= 1.0f);
}

template <int EPV, bool kPhases>
__global__ __launch_bounds__(NT) void k_rows_global(RowsArgs a) {
  C4S_PHASE(14);
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ Scratch sh;
  const int row = blockIdx.x;
  RowCfg c;
  int64_t h0, h1;
  if (!global_cfg(a, row, c, h0, h1)) {
    if (threadIdx.x == 0) a.out_tok[row] = -1;
    return;
  }
  if (kPhases && __builtin_expect(!one_read_applies(a, c) && big_covers(a, c), 0)) {
    if (big_single<EPV>(a, row, c, h0, h1, smem)) return;
    __syncthreads();
  }
  rows_global_row(a, row, c, h0, h1, smem, sh);
}

constexpr int kBigThreads = 512;   // phases A and B by slices

// Whether a call goes a launch a phase (else one workgroup a row). Both forms,
// microseconds a call at V = 151936 (10 slices; top_k / nucleus / greedy):
// fp32, 32 rows 25.6 / 48 / 15.4 against 25.3 / 159 / 37, 48 rows 26.8 / 50 /
// 16 against 25.4 / 161 / 37, 64 rows 33 / 66 / 20 against 25.7 / 163 / 37:
// fp32 top-k rows have the one read, so the launches stop paying where their
// workgroups pass the CUs; bf16, 32 rows 24 / 52 / 15 against 77 / 160 / 35, 256
// rows 68 / 159 / 40 against 79 / 164 / 36. At V = 20000 (2 slices) the
// launches cost more than spreading gives: 64 fp32 rows 20 / 35 / 14 against
// 13 / 45 / 11. The host does not see the rows' parameters, so the fp32 line is
// the top-k rows', and nucleus and greedy rows beyond it pay for that: 64 rows of
// 151936 as above, 50257 ids (4 slices) 17 / 74 / 18 in one workgroup a row where
// bf16 rows by phases take 22 / 38 / 14.
bool big_by_phase(const RowsArgs& a) {
  const int nsl = big_slices(a.vocab);
  return a.dtype == 0 ? nsl >= 8 && (int64_t)nsl * a.n_rows <= 320 : nsl >= 4;
}

// Workgroup -> (row, slice): consecutive workgroups go to the XCDs in turn, so
// workgroup 8 i + x takes slices of rows x, x + 8, ...: a row's slices share
// one XCD's L2, where phase B merges their histograms. The grid is rounded up
// to whole groups of 8 rows; false past the last row.
__device__ __forceinline__ bool big_place(const RowsArgs& a, int& row, int& s) {
  const int nsl = big_slices(a.vocab), i = (int)blockIdx.x >> 3;
  row = 8 * (i / nsl) + ((int)blockIdx.x & 7);
  s = i % nsl;
  return row < a.n_rows;
}

template <int EPV>
__global__ __launch_bounds__(kBigThreads) __attribute__((amdgpu_waves_per_eu(4))) void k_big_a(RowsArgs a) {
  __shared__ BigShA sh;
  C4S_PHASE(0);
  int row, s;
  if (!big_place(a, row, s)) return;
  const BigGeo g = big_geo(a, row);
  BigFetch<kSlice / kBigThreads, EPV> f;
  big_fetch<kSlice / kBigThreads, EPV>(g, s, f);   // in flight while the parameters arrive
  RowCfg c;
  int64_t h0, h1;
  if (!global_cfg(a, row, c, h0, h1) || !big_covers(a, c)) return;
  const BigHist hs = big_hist<kBigThreads>(a, h0, h1);
  const int nsl = big_slices(c.V);
  big_phase_a<kBigThreads, EPV>(a, row, c, g, big_row(c), hs, f, big_ws(a, row, nsl), s, sh);
}

template <int EPV>
__global__ __launch_bounds__(kBigThreads) __attribute__((amdgpu_waves_per_eu(4))) void k_big_b(RowsArgs a) {
  __shared__ BigShB sh;
  C4S_PHASE(7);
  int row, s;
  if (!big_place(a, row, s)) return;
  const BigGeo g = big_geo(a, row);
  const int nsl = big_slices(a.vocab);
  const BigWs ws = big_ws(a, row, nsl);
  // in issue order: the headers and histograms (of a row that has none, what
  // its workspace holds), the slice
  BigMerge<kBigThreads> mf;
  big_window_fetch<kBigThreads>(ws, nsl, mf);
  RowCfg c;
  int64_t h0, h1;
  if (!global_cfg(a, row, c, h0, h1) || !big_covers(a, c) || c.greedy || c.topk_on) return;
  BigFetch<kSlice / kBigThreads, EPV> f;
  big_fetch<kSlice / kBigThreads, EPV>(g, s, f);
  const BigHist hs = big_hist<kBigThreads>(a, h0, h1);
  BigWin win;
  const bool ok = big_window<kBigThreads>(c, ws, nsl, sh, mf, win);
  if (s == 0 && threadIdx.x == 0) {
    ws.hdr->wm = win.m;
    ws.hdr->wxlo = win.xlo;
    ws.hdr->wxhi = ok ? win.xhi : kBigNB;
  }
  if (!ok) return;
  C4S_PHASE(8);
  big_phase_b<kBigThreads, EPV>(a, row, c, g, big_row(c), hs, f, ws, s, win, sh);
}

__global__ __launch_bounds__(NT) void k_big_c(RowsArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ Scratch sh;
  const int row = blockIdx.x;
  C4S_PHASE(20);
  RowCfg c;
  int64_t h0, h1;
  if (!global_cfg(a, row, c, h0, h1)) {
    if (threadIdx.x == 0) a.out_tok[row] = -1;
    return;
  }
  if (big_covers(a, c)) {
    const int nsl = big_slices(c.V);
    const BigWs ws = big_ws(a, row, nsl);
    const BigHist hs = big_hist<NT>(a, h0, c.greedy || c.topk_on ? h0 : h1);
    BigWin win{};
    bool ok = true;
    if (!c.greedy && !c.topk_on) {
      win.m = ws.hdr->wm;
      win.fQ = floorf(win.m * kBigScale);
      win.xlo = ws.hdr->wxlo;
      win.xhi = ws.hdr->wxhi;
      ok = win.xhi < kBigNB;
    }
    C4S_PHASE(12);
    if (ok && big_finish<kSlice / kBigThreads>(a, row, c, big_geo(a, row), big_row(c), hs, ws, nsl, win, smem)) {
      C4S_PHASE(21);
      return;
    }
    __syncthreads();
  }
  rows_global_row(a, row, c, h0, h1, smem, sh);
}

// hist_bits[b] = the ids in [0, V) of row b's CSR history (sampling.cpp:24).
__global__ __launch_bounds__(NT) void k_hist_bits_init(const int32_t* ids, const int64_t* off, int V,
                                                       uint32_t* bits) {
  const int row = blockIdx.x;
  const int W = hist_words(V);
  uint32_t* b = bits + (int64_t)row * W;
  for (int w = threadIdx.x; w < W; w += NT) b[w] = 0u;
  __syncthreads();
  if (!ids) return;
  for (int64_t j = off[row] + threadIdx.x; j < off[row + 1]; j += NT) {
    const int id = ids[j];
    if (id >= 0 && id < V) atomicOr(&b[id >> 5], 1u << (id & 31));
  }
}

// Multi-step AR stream for rows staged in LDS: one persistent workgroup per
// row walks all steps. The row's distinct penalised ids live in an LDS bitmap
// that gains every sampled token that is not the stop token
// (text2semantic.cpp:333-334). While step s runs, the logits of step s+1 are
// already in flight into registers. A stopped row reports -1 afterwards and its
// RNG stays frozen.
__global__ __launch_bounds__(NT) void k_stream_lds(StreamArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ Scratch sh;
  const int row = blockIdx.x;
  const int V = a.vocab;
  const RowCfg c = make_cfg(0u, V, row, a.temp, a.top_k, a.top_p, a.pen, nullptr, a.do_sample);
  LdsLayout L = lds_layout(smem, V);
  const int nw = bitmap_words(V);
  for (int w = threadIdx.x; w < nw; w += NT) L.bitmap[w] = 0u;
  __syncthreads();
  {
    const int64_t h0 = a.hist_off[row], h1 = a.hist_off[row + 1];
    for (int64_t j = h0 + threadIdx.x; j < h1; j += NT) {
      const int id = a.hist_ids[j];
      if (id < 0 || id >= V) continue;
      atomicOr(&L.bitmap[id >> 5], 1u << (id & 31));
    }
  }
  uint64_t rng = a.rng[row];
  bool done = false;
  uint32_t acc_stats[4] = {0, 0, 0, 0};
  const float* base = a.logits + (int64_t)row * a.ld;
  RowFetch pf;
  fetch_row(base, V, pf);
  for (int s = 0; s < a.n_steps; ++s) {
    int32_t* outp = a.out_tok + (int64_t)s * a.n_rows + row;
    if (done) {
      if (threadIdx.x == 0) *outp = -1;
      continue;
    }
    C4S_PHASE(0);
    const float* cur = base + (int64_t)s * a.step_stride;
    float* val = store_row(cur, V, pf, L.val);
    if (s + 1 < a.n_steps) fetch_row(cur + a.step_stride, V, pf);
    __syncthreads();
    if (c.pen_on) {
      penalise_chunk(val, L.bitmap, V, c.pen);
      __syncthreads();
    }
    C4S_PHASE(1);
    LdsRow src{val, L.E, V, 0u, false};
    uint32_t* st = a.stats ? sh.step_stats : nullptr;   // written and read by thread 0 only
    int tok = 0;
    if (!(fast_topk_applies(c, V) &&
          fast_topk_any(val, V, c, sh, reinterpret_cast<unsigned char*>(L.E), rng, tok, nullptr, st)))
      tok = run_chain(src, sh, c, rng, nullptr, st);
    C4S_PHASE(8);
    if (threadIdx.x == 0) {
      *outp = tok;
      if (a.stats) {
        acc_stats[0] |= st[0];
        acc_stats[1] += st[1];
        acc_stats[2] += st[2];
        acc_stats[3] += st[3];
      }
      // Appending a token already in the history changes nothing: the penalty
      // applies once per distinct id (sampling.cpp:22).
      if (tok != a.stop_token && tok >= 0 && tok < V) L.bitmap[tok >> 5] |= 1u << (tok & 31);
    }
    if (tok == a.stop_token) done = true;
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    a.rng[row] = rng;
    if (a.stats) {
      uint32_t* o = a.stats + 4 * (int64_t)row;
      o[0] = acc_stats[0]; o[1] = acc_stats[1]; o[2] = acc_stats[2]; o[3] = acc_stats[3];
    }
  }
}

}  // namespace

size_t rows_lds_bytes(int V) {
  const size_t vp = (size_t)((V + 3) & ~3);
  return 8 * vp + 4 * (vp + 4) + 4 * (size_t)bitmap_words(V);
}

size_t stream_lds_bytes(int V, int) { return rows_lds_bytes(V); }

size_t rows_global_lds_bytes(int V) {
  const size_t own = V <= kT2MaxV ? t2_offset(V) + sizeof(T2Sh) : 4 * (size_t)((V + 31) / 32);
  return own > kBigFinishBytes ? own : kBigFinishBytes;
}

hipError_t launch_hist_bits_init(const int32_t* ids, const int64_t* off, int n_rows, int V, uint32_t* bits,
                                 hipStream_t s) {
  if (n_rows <= 0) return hipSuccess;
  (void)hipGetLastError();
  hipLaunchKernelGGL(k_hist_bits_init, dim3(n_rows), dim3(NT), 0, s, ids, off, V, bits);
  return hipGetLastError();
}

hipError_t launch_rows(const RowsArgs& a, hipStream_t s) {
  if (a.n_rows <= 0) return hipSuccess;
  (void)hipGetLastError();  // report only this launch's status
  if (a.vocab <= kLdsVocabMax && a.mode == 0u) {
    return rows_step_many_fits(a) ? launch_rows_step_many(a, s) : launch_rows_step(a, s);
  } else if (a.vocab <= kLdsVocabMax) {
    const size_t lds = rows_lds_bytes(a.vocab);
    hipLaunchKernelGGL(k_rows_lds, dim3(a.n_rows), dim3(NT), lds, s, a);
  } else {
    const size_t lds = rows_global_lds_bytes(a.vocab);
    if (a.mode == 0u && !a.out_masked && big_by_phase(a)) {
      const dim3 g(8 * big_slices(a.vocab) * ((a.n_rows + 7) / 8));
      if (a.dtype == 0) {
        hipLaunchKernelGGL(k_big_a<4>, g, dim3(kBigThreads), 0, s, a);
        hipLaunchKernelGGL(k_big_b<4>, g, dim3(kBigThreads), 0, s, a);
      } else {
        hipLaunchKernelGGL(k_big_a<8>, g, dim3(kBigThreads), 0, s, a);
        hipLaunchKernelGGL(k_big_b<8>, g, dim3(kBigThreads), 0, s, a);
      }
      hipLaunchKernelGGL(k_big_c, dim3(a.n_rows), dim3(NT), lds, s, a);
    } else {
      if (a.mode != 0u || a.out_masked) hipLaunchKernelGGL((k_rows_global<4, false>), dim3(a.n_rows), dim3(NT), lds, s, a);
      else if (a.dtype == 0) hipLaunchKernelGGL((k_rows_global<4, true>), dim3(a.n_rows), dim3(NT), lds, s, a);
      else hipLaunchKernelGGL((k_rows_global<8, true>), dim3(a.n_rows), dim3(NT), lds, s, a);
    }
  }
  return hipGetLastError();
}

hipError_t launch_stream(const StreamArgs& a, hipStream_t s) {
  if (a.n_rows <= 0 || a.n_steps <= 0) return hipSuccess;
  (void)hipGetLastError();
  const size_t lds = stream_lds_bytes(a.vocab, 0);
  hipLaunchKernelGGL(k_stream_lds, dim3(a.n_rows), dim3(NT), lds, s, a);
  return hipGetLastError();
}

}  // namespace c4s
