"""LM head at the edges of its tiles' row counts (16, 32, 64 and, past 192 rows and
a round of those tiles, 128 rows with 64 or 128 columns and chunks of 64 inputs),
for the three weight kinds,
against the float64 oracle; the tolerance and its derivation are test_gpu_lmhead's (the same split
of the weights, the same sums)."""
import numpy as np
import pytest

import c4s_workloads as W
from gpu_util import dev
from test_gpu_lmhead import ATOL, _weights

pytestmark = pytest.mark.gpu

CASES = [("bf16", 1, 1280, 8194, 64, 0.0), ("f32", 1, 320, 33, 32, 4.0), ("q8", 16, 288, 1000, 32, 0.0),
         ("bf16", 17, 32, 47, 32, 0.0), ("f32", 32, 1280, 500, 32, 0.0), ("q8", 31, 1280, 300, 128, 4.0),
         ("bf16", 33, 96, 31, 32, 0.0), ("q8", 192, 64, 100, 64, 0.0),
         ("bf16", 193, 32, 1, 32, 0.0), ("bf16", 255, 96, 63, 32, 0.0), ("bf16", 256, 64, 64, 32, 0.0),
         ("bf16", 257, 160, 65, 32, 4.0), ("bf16", 192, 160, 65, 32, 0.0), ("bf16", 300, 1280, 8194, 64, 0.0), ("bf16", 777, 1280, 5000, 64, 0.0),
         ("f32", 193, 96, 129, 32, 0.0), ("f32", 200, 2080, 127, 32, 4.0), ("f32", 520, 256, 8194, 64, 0.0),
         ("q8", 194, 32, 40, 32, 0.0), ("q8", 230, 192, 65, 64, 0.0), ("q8", 257, 256, 130, 128, 4.0),
         ("q8", 600, 1280, 8194, 64, 0.0), ("q8", 1000, 96, 4100, 32, 0.0),
         # past a round of the smaller tiles (512 of 32 columns x 64 rows; bf16 up to 1024 of long K)
         ("bf16", 193, 32, 4096, 32, 0.0), ("bf16", 193, 32, 4097, 32, 0.0), ("bf16", 255, 96, 4159, 32, 0.0),
         ("bf16", 256, 64, 4160, 32, 0.0), ("bf16", 257, 160, 4161, 32, 4.0), ("bf16", 200, 1024, 8193, 64, 0.0),
         ("bf16", 200, 1024, 8192, 64, 0.0), ("f32", 193, 96, 4223, 32, 0.0), ("f32", 200, 224, 4225, 32, 4.0),
         ("f32", 1030, 32, 961, 32, 0.0), ("q8", 194, 32, 4104, 32, 0.0), ("q8", 230, 192, 4161, 64, 0.0),
         ("q8", 257, 256, 4099, 128, 4.0)]


@pytest.mark.parametrize("kind,M,D,V,group,shift", CASES)
def test_lmhead_many_rows(orc, gpu_ctx, kind, M, D, V, group, shift):
    import torch
    head, _ = W.lmhead(seed=M + D, M=M, D=D, V=V)
    if shift:
        head.hidden = W.f32_to_bf16_bits(W.bf16_bits_to_f32(head.hidden) + np.float32(shift))
    wdev, quant, worc, kw = _weights(kind, head, M + D + 1, group)
    ld = V + 3   # rows of the output at every alignment; the columns past V stay as they are
    logits = torch.full((M, ld), 7.0, dtype=torch.float32, device="cuda")
    gpu_ctx.lmhead(dev(head.hidden, torch), dev(head.gamma, torch), dev(head.beta, torch), wdev,
                   dev(head.bias, torch), logits, quant=quant)
    torch.cuda.synchronize()
    got = logits.cpu().numpy()
    assert (got[:, V:] == 7.0).all()
    want = orc.ln_lmhead(head.hidden, head.gamma, head.beta, worc, head.bias, n_threads=16, **kw)
    err = np.abs(got[:, :V].astype(np.float64) - want)
    print(f"{kind} M={M} D={D} V={V}: max abs err {err.max():.3e}  max |logit| {np.abs(want).max():.3f}", flush=True)
    assert np.all(err <= ATOL)


@pytest.mark.parametrize("kind,D,sigmas", [("f32", 1280, 64.0), ("q8", 1280, 64.0), ("f32", 4096, 16.0), ("q8", 4096, 16.0)])
def test_offset_rows(gpu_ctx, kind, D, sigmas):
    """Rows far from mean 0, whose offset cancels between the products, the row
    statistics and c: a call of many rows is as close to 64 bits as a call of few.
    Both take sums of the same lengths, so their errors are draws of one spread;
    of a 2-norm over 192 rows that is off by 1 / sqrt(2 x 192) = 5%: three times
    that. With each sum as one fp32 sum over D the ratios were 2.5 and 1.36
    (1.04 and 1.02 with them in parts joined in double)."""
    import torch
    V, n = 4200, 192
    g = torch.Generator(device="cuda")
    g.manual_seed(D)
    rand = lambda *shape: torch.randn(shape, generator=g, device="cuda")   # noqa: E731
    x = (rand(200, D) + sigmas).to(torch.bfloat16)
    gamma, beta, bias, w = 1.0 + 0.02 * rand(D), 0.02 * rand(D), 0.02 * rand(V), 0.02 * rand(V, D)
    quant, wd = None, w.double()
    if kind == "q8":
        grp = w.view(V, D // 64, 64)
        lo, scale = grp.amin(dim=2), (grp.amax(dim=2) - grp.amin(dim=2)) / 255.0
        q = torch.clamp(torch.round((grp - lo[..., None]) / scale[..., None]), 0, 255)
        wd = (q.double() * scale.double()[..., None] + lo.double()[..., None]).view(V, D)
        w, quant = q.to(torch.uint8).view(V, D), (scale.contiguous(), lo.contiguous(), 64)
    y = x.double() - x.double().mean(dim=1, keepdim=True)
    y = y / (y.square().mean(dim=1, keepdim=True) + 1e-5).sqrt() * gamma.double() + beta.double()
    want = (y @ wd.t() + bias.double())[:n]

    def error(rows):
        logits = torch.empty((rows, V), device="cuda")
        gpu_ctx.lmhead(x[:rows].contiguous(), gamma, beta, w, bias, logits, quant=quant)
        return float((logits[:n].double() - want).norm() / want.norm())

    few, many = error(n), error(200)
    print(f"{kind} D={D} offset {sigmas} sigma: {few:.3e} of {n} rows, {many:.3e} of 200", flush=True)
    assert many <= 1.15 * few
