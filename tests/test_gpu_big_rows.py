"""Rows larger than LDS decided by slices: tokens and generator states against
the oracle, bit for bit, where the phases can go wrong -- the ends of a slice
(16384 ids) and of a row at every alignment, empty last slices, the boundary
among ties, rows of -inf, slices far below the maximum, min_tokens_to_keep --
for both storage types, for few rows (a launch a phase) and for many (one
workgroup a row)."""
import numpy as np
import pytest

import c4s_workloads as W
from gpu_util import compare_with_oracle, dev

pytestmark = pytest.mark.gpu

PHASES = 16 | 64   # statistics[0]: decided without the multi-pass chain, by the phases or by the one read


def _batch(seed, n, V, sigma=2.0, hist=300):
    g = np.random.default_rng(seed)
    x = (g.standard_normal((n, V), dtype=np.float32) * np.float32(sigma)).astype(np.float32)
    x[:, g.integers(0, V, 5)] += np.float32(6.0)
    ids, off = W.csr([g.integers(-3, V + 3, size=hist).astype(np.int32) for _ in range(n)])
    kinds = np.arange(n) % 8   # nucleus x3, top-k x2, dense, greedy, nucleus with a temperature of 1
    return W.Batch(logits=x, hist_ids=ids, hist_off=off,
                   temp=np.where(kinds == 7, 1.0, g.uniform(0.6, 1.3, n)).astype(np.float32),
                   top_k=np.choose(kinds, [0, 0, V, 50, 1, 0, 0, 0]).astype(np.int32),
                   top_p=np.choose(kinds, [0.9, 0.5, 0.99, 0.95, 0.8, 1.0, 0.9, 0.8]).astype(np.float32),
                   pen=g.choice(np.array([1.0, 1.2, 10.0, 0.8], np.float32), n),
                   do_sample=(kinds != 6).astype(np.uint8), rng=W.seed_batch(seed, n))


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("V", [12289, 16377, 16384, 16385, 32761, 50257, 131065, 131073, 151936])
def test_slices(orc, gpu_ctx, V, dtype):
    b = _batch(V, 16, V)   # an odd V puts the rows at every alignment
    if dtype == "bf16":
        b.logits = W.f32_to_bf16_bits(b.logits)
    tok, st = compare_with_oracle(orc, gpu_ctx, b, masked=False)
    print(V, dtype, st[:, 0].tolist(), flush=True)
    # the ordinary rows take the phases (a draw close to a boundary may not)
    assert np.count_nonzero(st[:, 0] & PHASES) >= 15


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_many_rows(orc, gpu_ctx, dtype):
    """One workgroup a row, more rows than CUs."""
    b = _batch(7, 260, 16391)
    if dtype == "bf16":
        b.logits = W.f32_to_bf16_bits(b.logits)
    compare_with_oracle(orc, gpu_ctx, b, masked=False)


@pytest.mark.parametrize("rows,V", [(12, 140000), (260, 40000)])
def test_boundaries(orc, gpu_ctx, rows, V):
    """Ties at the cut and at the k-th value, within and past what a slice
    lists; a row of -inf, of one finite value, of equal values; all the mass in
    the last slice; values far below; min_tokens_to_keep past the nucleus."""
    b = _batch(11, rows, V, hist=50)
    x, ninf = b.logits, -np.inf
    b.pen[:] = 1.0
    b.do_sample[:] = 1
    b.temp[:] = 1.0
    b.top_k[:] = 0
    b.top_p[:] = 0.7
    x[0, :] = np.round(x[0] * 4) / 4              # a few hundred ids a value: the cut falls among ties
    x[1, :] = 1.5                                 # every value equal
    x[2, :] = ninf
    x[3, :] = ninf
    x[3, V - 1] = -7.0
    x[4, :30000] -= 300.0                         # the first slice far below the others
    x[5, :] -= 700.0 * (np.arange(V) % 2).astype(np.float32)   # half of the row below the exponent range of the masses
    x[6, 16380:16390] = 30.0                      # the maximum tied across a slice's end
    x[7, :] *= 1000.0                             # one value holds all the mass
    b.top_k[8], x[8, 100:165] = 64, 40.0          # 65 equal values at the k-th
    b.top_k[9], b.temp[9] = 30, 0.0
    x[10, :] += 3e5                               # too large for the grid
    b.top_p[5] = 1.0
    mk = np.ones(rows, np.int32)
    mk[6], mk[7], mk[9], mk[11] = 5000, 3, 40, 0
    compare_with_oracle(orc, gpu_ctx, b, min_keep=mk, masked=False)
    b.logits = W.f32_to_bf16_bits(x)
    compare_with_oracle(orc, gpu_ctx, b, min_keep=mk, masked=False)
    act = (np.arange(rows) % 3 != 1).astype(np.uint8)
    tok, _ = compare_with_oracle(orc, gpu_ctx, b, min_keep=mk, row_active=act, masked=False)
    assert (tok[act == 0] == -1).all()


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("rows,V", [(16, 16385), (16, 65573), (16, 131073), (260, 16385), (30, 151600)])
def test_topk_few_in_a_slice(orc, gpu_ctx, rows, V, dtype):
    """top_k rows whose slices hold fewer than k + 1 values: a last slice of one
    to a few dozen ids, slices of -inf but for none, one, k or k + 1 values."""
    b = _batch(V + rows, rows, V, hist=50)
    k = np.array([1, 2, 7, 49, 50, 63, 64, 120], np.int32)[np.arange(rows) % 8]
    b.top_k, b.do_sample = k, np.ones(rows, np.uint8)
    b.top_p = np.where(np.arange(rows) % 3 == 0, 1.0, 0.9).astype(np.float32)
    b.pen = np.where(np.arange(rows) % 2 == 0, 1.2, 0.8).astype(np.float32)   # below 1: not the one read
    g = np.random.default_rng(rows)
    for r in range(rows):
        for s in range(0, V, 16384):
            m = min(16384, V - s)
            few = [m, 0, 1, int(k[r]), int(k[r]) + 1][(r + s // 16384) % 5]
            if few < m:
                keep = g.choice(m, few, replace=False)
                part = b.logits[r, s:s + m][keep]
                b.logits[r, s:s + m] = -np.inf
                b.logits[r, s + keep] = part
    b.logits[:, 5] = 1.0   # no row without a finite value
    if dtype == "bf16":
        b.logits = W.f32_to_bf16_bits(b.logits)
    compare_with_oracle(orc, gpu_ctx, b, masked=False)


@pytest.mark.parametrize("rows,V", [(9, 140000), (260, 40000)])
def test_maxima_about_the_grids_end(orc, gpu_ctx, rows, V):
    """Nucleus rows with slice maxima on both sides of -2^18 and 2^18, where the
    histograms' grid ends for a row's maximum; each after a call whose rows leave
    other histograms in the same workspace."""
    b = _batch(5, rows, V, sigma=1.0, hist=50)
    b.do_sample[:], b.top_k[:], b.temp[:], b.pen[:] = 1, 0, 1.0, 1.0
    b.top_p = np.choose(np.arange(rows) % 3, [0.5, 0.8, 0.95]).astype(np.float32)
    x = np.clip(b.logits, -8.0, 2.0)
    s = np.arange(V) // 16384
    x_far = x - 8.0 - 2.0 * ((s[None, :] + np.arange(rows)[:, None]) % 4)
    at = (np.arange(rows) * 7919) % V
    for end, top in ((-262144.0, -262143.0), (262144.0, 262143.0)):
        b.logits = np.full_like(x, -10.0)   # its masses at lower grid places than the next rows'
        compare_with_oracle(orc, gpu_ctx, b, masked=False)
        y = (x_far + end).astype(np.float32)
        y[np.arange(rows), at] = np.float32(top)   # the row's maximum
        b.logits = y
        _, st = compare_with_oracle(orc, gpu_ctx, b, masked=False)
        if end < 0:   # settled by the phases, on this row's own histograms
            assert np.count_nonzero(st[:, 0] & 16) >= rows - 2 - rows // 20, st[:, 0].tolist()


@pytest.mark.parametrize("rows,V", [(9, 131077), (200, 20011)])
def test_history_set(orc, gpu_ctx, rows, V):
    """The history kept as a set: three steps, each token joining it."""
    import torch
    b = _batch(23, rows, V, hist=120)
    hist = [b.hist_ids[b.hist_off[i]:b.hist_off[i + 1]].tolist() for i in range(rows)]
    bits = torch.zeros((rows, (V + 31) // 32), dtype=torch.int32, device="cuda")
    gpu_ctx.hist_bits_init(dev(b.hist_ids, torch), dev(b.hist_off, torch), rows, V, bits)
    rng = dev(b.rng, torch)
    want_rng = b.rng
    tok = torch.empty(rows, dtype=torch.int32, device="cuda")
    for _ in range(3):
        gpu_ctx.sample_rows(dev(b.logits, torch), None, None, dev(b.temp, torch), dev(b.top_k, torch),
                            dev(b.top_p, torch), dev(b.pen, torch), rng, tok, do_sample=dev(b.do_sample, torch),
                            hist_bits=bits, stop_token=V - 1)
        ids, off = W.csr([np.asarray(h, np.int32) for h in hist])
        want, want_rng, _ = orc.sample_rows(b.logits, ids, off, b.temp, b.top_k, b.top_p, b.pen, b.do_sample, want_rng,
                                            want_masked=False, n_threads=16)
        got = tok.cpu().numpy()
        assert np.array_equal(got, want)
        assert np.array_equal(rng.cpu().numpy().view(np.uint64), want_rng)
        for i, k in enumerate(want.tolist()):
            if k != V - 1:
                hist[i].append(k)


@pytest.mark.parametrize("n_streams", [2, 10])
def test_streams_of_one_context(gpu_ctx, n_streams):
    """Calls of one context on several streams at once (more of them than the
    context keeps workspaces for, too), of different shapes: the same tokens and
    states as one call after the other."""
    import torch
    bs = [_batch(31 + i, 16, [131073, 151936, 140001][i % 3]) for i in range(n_streams)]
    dv = [{k: dev(getattr(b, k), torch) for k in ("logits", "hist_ids", "hist_off", "temp", "top_k", "top_p", "pen",
                                                  "do_sample")} for b in bs]

    def run(streams):
        rngs = [dev(b.rng, torch) for b in bs]
        toks = [[torch.empty(16, dtype=torch.int32, device="cuda") for _ in range(4)] for _ in bs]
        torch.cuda.synchronize()
        for step in range(4):
            for i, d in enumerate(dv):
                gpu_ctx.sample_rows(d["logits"], d["hist_ids"], d["hist_off"], d["temp"], d["top_k"], d["top_p"],
                                    d["pen"], rngs[i], toks[i][step], do_sample=d["do_sample"], stream=streams[i])
                if streams[0] is None:
                    torch.cuda.synchronize()
        torch.cuda.synchronize()
        return [[t.cpu().numpy() for t in ts] for ts in toks], [r.cpu().numpy() for r in rngs]

    want = run([None] * n_streams)
    got = run([torch.cuda.Stream() for _ in bs])
    for w, g in zip(want[0], got[0]):
        for a, b in zip(w, g):
            assert np.array_equal(a, b)
    for a, b in zip(want[1], got[1]):
        assert np.array_equal(a, b)
