"""Many more rows than CUs: the one-pass step in the form that shares a CU, against
the oracle bit for bit -- vocabularies at the sizes where the ids a thread owns
change and on both sides of the largest one that fits, every row kind, and the
rows that one pass leaves to the chain."""
import numpy as np
import pytest

import c4s_workloads as W
from gpu_util import compare_with_oracle, dev, gpu_rows

pytestmark = pytest.mark.gpu


def _rows(seed, n, V, sigma):
    g = np.random.default_rng(seed)
    x = (g.standard_normal((n, V)) * sigma).astype(np.float32)
    hist = [g.integers(-5, V + 5, size=int(g.integers(0, 300))).astype(np.int32) for _ in range(n)]
    ids, off = W.csr(hist)
    pick = lambda v, t: g.choice(np.array(v, t), n)   # noqa: E731
    return W.Batch(logits=x, hist_ids=ids, hist_off=off, temp=pick([0.7, 1.0, 1.3, 0.0], np.float32),
                   top_k=pick([0, 0, 1, 30, 200, V], np.int32), top_p=pick([0.0, 0.3, 0.8, 0.95, 1.0, 1.2], np.float32),
                   pen=pick([1.0, 1.3, 10.0, 0.5], np.float32), do_sample=(g.random(n) > 0.1).astype(np.uint8),
                   rng=W.seed_batch(seed, n)), pick([1, 1, 1, 0, 2, 40], np.int32)


@pytest.mark.parametrize("masked", [True, False])
@pytest.mark.parametrize("V", [1, 3, 65, 513, 4608, 4609, 8194, 8704, 9000, 9300])
def test_vocab_sizes(orc, gpu_ctx, V, masked):
    b, mk = _rows(V, 600, V, 2.0)
    compare_with_oracle(orc, gpu_ctx, b, min_keep=mk, masked=masked)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("sigma", [0.3, 3.0, 200.0])
def test_kinds(orc, gpu_ctx, sigma, dtype):
    """Flat rows (the refined boundary), peaked ones, and rows wider than the
    masses' exponent range; then rows for the chain: all -inf, one finite value,
    below the draw's floor, every value equal, two values."""
    V, n = 8194, 600
    b, mk = _rows(5, n, V, sigma)
    x = b.logits
    x[0] = -np.inf
    x[1] = -np.inf
    x[1, 17] = 2.0
    x[2] = -1e31
    x[3] = 0.25
    x[4] = np.where(np.arange(V) % 3 == 0, 1.0, 0.0)
    x[5] = np.round(x[5])
    b.do_sample[:6] = 1
    b.pen[:6] = 1.0
    b.temp[:6] = 1.0
    b.top_k[:6] = 0
    b.top_p[:6] = 0.6
    if dtype == "bf16":
        b.logits = W.f32_to_bf16_bits(x)
    act = (np.arange(n) % 7 != 6).astype(np.uint8)
    # p = 0 with min_tokens_to_keep 0 keeps the largest value or nothing, by whether
    # the last sum of the quotients rounds above 1: the last bit of the host's exp
    # decides (the contract in c4s_sampling.h). Nothing kept draws id 0.
    open_ = (b.top_p == 0.0) & (mk == 0) & (b.do_sample == 1) & (act == 1)
    assert open_.sum() >= 8
    tok, rng, _, _ = gpu_rows(gpu_ctx, b, masked=False, min_keep=mk, row_active=act)
    want = [orc.sample_rows(b.logits, b.hist_ids, b.hist_off, b.temp, b.top_k, b.top_p, b.pen, b.do_sample, b.rng,
                            min_keep=m, row_active=act, want_masked=False, n_threads=16)
            for m in (mk, np.maximum(mk, 1))]
    bad = np.flatnonzero((tok != want[0][0]) & ~open_)
    assert bad.size == 0, f"rows {bad[:10].tolist()}: gpu {tok[bad[:10]]} oracle {want[0][0][bad[:10]]}"
    assert ((tok == 0) | (tok == want[1][0]))[open_].all()
    assert np.array_equal(rng, want[0][1])
    assert (tok[act == 0] == -1).all()


def test_history_set(orc, gpu_ctx):
    import torch
    V, n = 4097, 600
    b, _ = _rows(9, n, V, 2.0)
    hist = [b.hist_ids[b.hist_off[i]:b.hist_off[i + 1]].tolist() for i in range(n)]
    bits = torch.zeros((n, (V + 31) // 32), dtype=torch.int32, device="cuda")
    gpu_ctx.hist_bits_init(dev(b.hist_ids, torch), dev(b.hist_off, torch), n, V, bits)
    rng, want_rng = dev(b.rng, torch), b.rng
    tok = torch.empty(n, dtype=torch.int32, device="cuda")
    for _ in range(3):
        gpu_ctx.sample_rows(dev(b.logits, torch), None, None, dev(b.temp, torch), dev(b.top_k, torch),
                            dev(b.top_p, torch), dev(b.pen, torch), rng, tok, do_sample=dev(b.do_sample, torch),
                            hist_bits=bits, stop_token=V - 1)
        ids, off = W.csr([np.asarray(h, np.int32) for h in hist])
        want, want_rng, _ = orc.sample_rows(b.logits, ids, off, b.temp, b.top_k, b.top_p, b.pen, b.do_sample, want_rng,
                                            want_masked=False, n_threads=16)
        assert np.array_equal(tok.cpu().numpy(), want)
        assert np.array_equal(rng.cpu().numpy().view(np.uint64), want_rng)
        for i, k in enumerate(want.tolist()):
            if k != V - 1:
                hist[i].append(k)
