"""Stream rows whose nucleus is wider than the scan's candidate list (flat rows:
more than 512 ids kept): the exact steps inside the speculative chain, token for
token against the oracle."""
import numpy as np
import pytest

import c4s_workloads as W
from gpu_util import dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V,steps,sigma,ties", [(8194, 40, 3.0, False), (8232, 24, 2.0, False), (3001, 24, 0.7, False),
                                                (8194, 24, 3.0, True), (700, 16, 0.2, False), (8194, 300, 3.0, False)])
def test_wide_nucleus(orc, gpu_ctx, V, steps, sigma, ties):
    import torch
    rows = 8
    g = np.random.default_rng(V + steps)
    x = (g.standard_normal((steps, rows, V), dtype=np.float32) * np.float32(sigma)).astype(np.float32)
    if ties:   # a few values only: the cut falls among thousands of equal ones
        x = np.round(x * 2) / 2
    x[0, 0] = -np.inf       # nothing to draw but the last id's fallback
    x[1, 1, 5:] = -np.inf
    ids, off = W.csr([g.integers(0, V, size=int(g.integers(0, 200))).astype(np.int32) for _ in range(rows)])
    temp = g.uniform(1.0, 1.3, rows).astype(np.float32)
    temp[2] = 1.0
    top_p = np.array([0.9, 0.95, 0.99, 0.9, 0.8, 0.97, 0.92, 0.999], np.float32)
    pen = np.array([1.0, 10.0, 1.2, 10.0, 1.0, 1.5, 10.0, 1.0], np.float32)
    top_k = np.zeros(rows, np.int32)
    do = np.ones(rows, np.uint8)
    rng0 = W.seed_batch(77, rows)
    out = torch.empty((steps, rows), dtype=torch.int32, device="cuda")
    stats = torch.zeros((rows, 4), dtype=torch.int32, device="cuda")
    rng = dev(rng0, torch)
    work = torch.cuda.Stream()
    torch.cuda.synchronize()
    gpu_ctx.sample_stream(dev(x, torch), dev(ids, torch), dev(off, torch), dev(temp, torch), dev(top_k, torch),
                          dev(top_p, torch), dev(pen, torch), rng, out, do_sample=dev(do, torch), out_stats=stats,
                          stream=work)
    torch.cuda.synchronize()
    want, want_rng = orc.sample_stream(x, ids, off, temp, top_k, top_p, pen, do, rng0, n_threads=16)
    got = out.cpu().numpy()
    st = stats.cpu().numpy()
    print(V, steps, "exact steps", st[:, 1].tolist(), flush=True)
    assert np.array_equal(got, want), np.argwhere(got != want)[:5].tolist()
    assert np.array_equal(rng.cpu().numpy().view(np.uint64), want_rng)
    assert st[:, 1].sum() > 0   # some steps were wider than the list
