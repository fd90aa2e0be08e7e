"""Graph capture: c4s_sample_rows (no workspace at vocab <= 12288) captured
into a HIP graph gives, on every replay, the tokens and RNG states of the same
call made eagerly; a call whose workspace would grow is refused under capture
and captures once an eager call has sized it, with a workspace that later
eager calls do not touch; calls on other streams are taken while one is
captured; c4s_sample_stream refuses capture with C4S_EINVAL."""
import numpy as np
import pytest

import c4s
import c4s_workloads as W
from gpu_util import dev

pytestmark = pytest.mark.gpu


def _args(torch, b):
    return dict(logits=dev(b.logits, torch), hist_ids=dev(b.hist_ids, torch), hist_off=dev(b.hist_off, torch),
                temp=dev(b.temp, torch), top_k=dev(b.top_k, torch), top_p=dev(b.top_p, torch),
                pen=dev(b.pen, torch), do_sample=dev(b.do_sample, torch))


def test_sample_rows_graph_replays_match_eager(gpu_ctx):
    import torch
    b = W.batch64(seed=77, rows=64)
    a = _args(torch, b)
    s = torch.cuda.Stream()
    n_replays = 4
    # eager: the same call n_replays times in a row (the RNG advances each time)
    rng = dev(b.rng, torch)
    tok = torch.zeros(64, dtype=torch.int32, device="cuda")
    want_tok, want_rng = [], []
    with torch.cuda.stream(s):
        for _ in range(n_replays):
            gpu_ctx.sample_rows(a["logits"], a["hist_ids"], a["hist_off"], a["temp"], a["top_k"], a["top_p"],
                                a["pen"], rng, tok, do_sample=a["do_sample"], stream=s)
            s.synchronize()
            want_tok.append(tok.cpu().numpy().copy())
            want_rng.append(rng.cpu().numpy().copy())
    # captured once, replayed n_replays times from the starting RNG state
    rng0 = dev(b.rng, torch)
    rng.copy_(rng0)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        gpu_ctx.sample_rows(a["logits"], a["hist_ids"], a["hist_off"], a["temp"], a["top_k"], a["top_p"],
                            a["pen"], rng, tok, do_sample=a["do_sample"], stream=s)
    for k in range(n_replays):
        tok.fill_(-5)
        g.replay()
        torch.cuda.synchronize()
        # eager work between replays
        _ = (a["logits"] * 2).sum().item()
        assert np.array_equal(tok.cpu().numpy(), want_tok[k]), k
        assert np.array_equal(rng.cpu().numpy(), want_rng[k]), k


def test_sample_stream_refuses_capture(gpu_ctx):
    import torch
    p = W.batch64_params(seed=3, rows=4, V=100)
    x = dev(W.batch64_logits(4, 3, 4, 100), torch)
    out = torch.zeros((3, 4), dtype=torch.int32, device="cuda")
    rng = dev(p["rng"], torch)
    d = {k: dev(p[k], torch) for k in ("hist_ids", "hist_off", "temp", "top_k", "top_p", "pen", "do_sample")}
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    err = None
    with torch.cuda.graph(g, stream=s):
        try:
            gpu_ctx.sample_stream(x, d["hist_ids"], d["hist_off"], d["temp"], d["top_k"], d["top_p"], d["pen"],
                                  rng, out, do_sample=d["do_sample"], stream=s)
        except c4s.C4SError as e:
            err = str(e)
    assert err is not None and "code 1" in err and "captured" in err


def test_large_vocab_workspace_is_sized_outside_capture():
    """A vocabulary above 12288 needs the context's key workspace: the first
    such call under capture is refused (no allocation inside a capture) and
    queues nothing; once an eager call of that shape has sized the workspace,
    the same call captures, and its replays give the eager call's tokens."""
    import torch
    ctx = c4s.Context(0)   # a fresh context: no workspace yet
    try:
        b = W.batch64(seed=91, rows=4, V=20000)
        a = _args(torch, b)
        s = torch.cuda.Stream()
        tok = torch.full((4,), -5, dtype=torch.int32, device="cuda")
        rng = dev(b.rng, torch)
        torch.cuda.synchronize()

        def call():
            ctx.sample_rows(a["logits"], a["hist_ids"], a["hist_off"], a["temp"], a["top_k"], a["top_p"],
                            a["pen"], rng, tok, do_sample=a["do_sample"], stream=s)

        g0 = torch.cuda.CUDAGraph()
        err = None
        with torch.cuda.graph(g0, stream=s):
            try:
                call()
            except c4s.C4SError as e:
                err = str(e)
        assert err is not None and "code 1" in err and "graph capture" in err
        assert bool((tok == -5).all()), "the refused call queued work"
        # eager: sizes the workspace and gives the reference tokens
        with torch.cuda.stream(s):
            call()
        s.synchronize()
        want_tok, want_rng = tok.cpu().numpy().copy(), rng.cpu().numpy().copy()
        rng.copy_(dev(b.rng, torch))
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            call()
        for k in range(3):
            rng.copy_(dev(b.rng, torch))
            tok.fill_(-5)
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            _ = (a["logits"] * 2).sum().item()   # eager work between replays
            assert np.array_equal(tok.cpu().numpy(), want_tok), k
            assert np.array_equal(rng.cpu().numpy(), want_rng), k
    finally:
        ctx.close()


def _big(torch, seed, rows, V):
    b = W.batch64(seed=seed, rows=rows, V=V)
    return b, _args(torch, b), dev(b.rng, torch), torch.full((rows,), -5, dtype=torch.int32, device="cuda")


def _call(ctx, v, stream):
    _, a, rng, tok = v
    ctx.sample_rows(a["logits"], a["hist_ids"], a["hist_off"], a["temp"], a["top_k"], a["top_p"], a["pen"], rng, tok,
                    do_sample=a["do_sample"], stream=stream)


def test_large_vocab_replays_beside_eager_calls():
    """A graph captured after a warm-up on another stream (as frameworks do it),
    replayed while that stream and others, more of them than the context keeps
    workspaces for, make calls of the same size: every result is the one of the
    same call alone."""
    import torch
    ctx = c4s.Context(0)
    try:
        streams = [torch.cuda.Stream() for _ in range(11)]
        vs = [_big(torch, 40 + i, 16, 151936) for i in range(11)]
        torch.cuda.synchronize()
        want = []
        for v, s in zip(vs, [streams[0]] * 11):   # alone, one after the other
            _call(ctx, v, s)
            torch.cuda.synchronize()
            want.append((v[3].cpu().numpy().copy(), v[2].cpu().numpy().copy()))
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=streams[10]):
            _call(ctx, vs[10], streams[10])
        for k in range(6):
            for v in vs:
                v[2].copy_(dev(v[0].rng, torch))
                v[3].fill_(-5)
            torch.cuda.synchronize()
            with torch.cuda.stream(streams[10]):
                g.replay()
            for i in range(10):
                _call(ctx, vs[(i + k) % 10], streams[i])
            torch.cuda.synchronize()
            for i, (v, w) in enumerate(zip(vs, want)):
                assert np.array_equal(v[3].cpu().numpy(), w[0]), (k, i)
                assert np.array_equal(v[2].cpu().numpy(), w[1]), (k, i)
    finally:
        torch.cuda.synchronize()
        ctx.close()


def test_calls_while_another_stream_is_captured():
    """A call on a stream that has no workspace yet, while another stream of the
    thread is being captured, is taken and leaves the capture whole; so is a
    captured call of a size that only other streams have used."""
    import torch
    ctx = c4s.Context(0)
    try:
        v, u = _big(torch, 71, 8, 131000), _big(torch, 72, 8, 131000)
        s0, s1, s2 = (torch.cuda.Stream() for _ in range(3))
        torch.cuda.synchronize()
        _call(ctx, v, s0)
        _call(ctx, u, s0)
        torch.cuda.synchronize()
        want = [(x[3].cpu().numpy().copy(), x[2].cpu().numpy().copy()) for x in (v, u)]
        for x in (v, u):
            x[2].copy_(dev(x[0].rng, torch))
            x[3].fill_(-5)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s2):
            _call(ctx, v, s2)
            _call(ctx, u, s1)   # not captured: s1 is no part of the graph
        torch.cuda.synchronize()
        assert np.array_equal(u[3].cpu().numpy(), want[1][0])
        assert np.array_equal(u[2].cpu().numpy(), want[1][1])
        assert bool((v[3] == -5).all())
        for k in range(3):
            v[2].copy_(dev(v[0].rng, torch))
            v[3].fill_(-5)
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            _ = (v[1]["logits"] * 2).sum().item()   # eager work between replays
            assert np.array_equal(v[3].cpu().numpy(), want[0][0]), k
            assert np.array_equal(v[2].cpu().numpy(), want[0][1]), k
    finally:
        torch.cuda.synchronize()
        ctx.close()


@pytest.mark.parametrize("V,dim", [(3000, 128), (20000, 128)])
def test_lmhead_sample_on_several_streams(V, dim):
    """c4s_lmhead_sample without a logits buffer on ten streams of one context at
    once: the tokens and states of one call after the other."""
    import torch
    ctx = c4s.Context(0)
    try:
        vs = []
        for i in range(10):
            head, p = W.lmhead(seed=80 + i, M=24, D=dim, V=V)
            d = [dev(x, torch) for x in (head.hidden, head.gamma, head.beta, head.weight, head.bias, p["hist_ids"],
                                         p["hist_off"], p["temp"], p["top_k"], p["top_p"], p["pen"])]
            vs.append((d, p, dev(p["rng"], torch), torch.full((24,), -5, dtype=torch.int32, device="cuda"),
                       dev(p["do_sample"], torch)))

        def run(streams):
            for _, p, rng, tok, _ in vs:
                rng.copy_(dev(p["rng"], torch))
                tok.fill_(-5)
            torch.cuda.synchronize()
            for _ in range(3):
                for (d, _, rng, tok, do), s in zip(vs, streams):
                    ctx.lmhead_sample(*d, rng, tok, do_sample=do, stream=s)
                    if streams[0] is None:
                        torch.cuda.synchronize()
            torch.cuda.synchronize()
            return [(v[3].cpu().numpy().copy(), v[2].cpu().numpy().copy()) for v in vs]

        want = run([None] * 10)
        got = run([torch.cuda.Stream() for _ in vs])
        for i, (a, b) in enumerate(zip(want, got)):
            assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1]), i
    finally:
        torch.cuda.synchronize()
        ctx.close()
