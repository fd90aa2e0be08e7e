// One AR step of rows whose vocabulary fits LDS: k_rows_step, one workgroup a row.
// In a file, and so a code object, of its own, the instance of the semantic
// vocabulary first, right behind the helpers that it calls: an instance is about
// 180 KB of code, several times the instruction cache, and the same instructions
// take a different time with where they lie to each other. The head and this
// step, 64 flat rows of 8194 ids: 37.25 us; 37.8 with the instance of fewer ids
// in between; 37.55 to 37.8 in one file with the kernels of other vocabularies,
// as these grew. The instance of fewer ids last: 32 steps of 20 nucleus rows of
// 3000 ids 347.4 us, 349.3 in the middle (the largest last: 10000 ids, 20 rows,
// 508.9 us against 513.0).

#include "c4s_onepass.hpp"

namespace c4s {
namespace {

// One AR step of the reference chain (C4S_MODE_CHAIN) for one row per
// workgroup, in one pass where it can (c4s_step.hpp), else the multi-pass
// chain on the row staged in LDS. PT >= the ids a thread owns.
template <int PT>
__global__ __launch_bounds__(kStepThreads) void k_rows_step(RowsArgs a) {
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
  float* vbuf = reinterpret_cast<float*>(smem + step_work_bytes(V));
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
  float* em = reinterpret_cast<float*>(work + kStepWorkBytes);   // per-id fp32 masses
  if (c.topk_on) done = sampled_step<PT, kKindTopK>(io, c, y, lo, n, val, hc, hm, sbuf, list, em, ss, rs);
  else if (c.p >= 1.0f) done = sampled_step<PT, kKindDense>(io, c, y, lo, n, val, hc, hm, sbuf, list, em, ss, rs);
  else done = sampled_step<PT, kKindTopP>(io, c, y, lo, n, val, hc, hm, sbuf, list, em, ss, rs);
  if (done) return;
  // ---- the multi-pass chain on the row staged in LDS (c4s_chain.hpp) ----
  __syncthreads();   // every thread is done with the work area
  chain_fallback(rs.io, rs.cfg, work, val, sh, rs.tp_exact_first != 0u);
}

// in this order in the code object
template __global__ void k_rows_step<17>(RowsArgs);
template __global__ void k_rows_step<25>(RowsArgs);
template __global__ void k_rows_step<9>(RowsArgs);

}  // namespace

size_t rows_step_lds_bytes(int V) {
  return step_work_bytes(V) + 4 * ((size_t)vpad(V) + 4) + 4 * (size_t)bitmap_words(V);
}

hipError_t launch_rows_step(const RowsArgs& a, hipStream_t s) {
  const size_t lds = rows_step_lds_bytes(a.vocab);
  const int P = ((a.vocab + kStepThreads - 1) / kStepThreads) | 1;   // ids a thread owns (odd_chunk)
  const dim3 g(a.n_rows), b(kStepThreads);
  if (P <= 9) hipLaunchKernelGGL(k_rows_step<9>, g, b, lds, s, a);
  else if (P <= 17) hipLaunchKernelGGL(k_rows_step<17>, g, b, lds, s, a);
  else hipLaunchKernelGGL(k_rows_step<25>, g, b, lds, s, a);
  return hipGetLastError();
}

}  // namespace c4s
