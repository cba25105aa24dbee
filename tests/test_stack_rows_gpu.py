"""The layer stack at one and two rows, where a layer's norm runs inside its input projections and the out
projection adds into the residual: single layers of each kind at the edges of the norm's row (less than a
workgroup's 2048 elements, exactly that, a ragged second and third piece), against the oracle. Three rows take the separate
norm and give the other side.

Both sides round the normed row (d_model values) and the gated mixer output (512 or 1024) to bf16. The bar
is twice the oracle's own movement when its input moves by 2^-20, plus three values that the oracle's two
runs round alike and the GPU the other way: one step of a value four times the rms, 4 x 2^-8, moves a
product of n such values by 4 x 2^-8 / sqrt(n) of its rms, n the smaller of d_model and 512. (A value is
within 2^-20 of a rounding boundary once in 2^11, so a few of them per row are ordinary.) Sixteen missing
values of 2064 would move it by sqrt(16 / 2064) = 9e-2, forty times the bar."""
import pytest
import torch

import test_stack_gpu as S
from conftest import perturb, rel_err, rms_err
from oracle import mixer_ref as R

from aegist_mixer import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 2, 3])
@pytest.mark.parametrize("d_model", [16, 528, 2048, 2064, 4112, 8192])
@pytest.mark.parametrize("kind", ["delta", "attn"])
def test_single_layer_rows(dev, monkeypatch, kind, d_model, rows):
    cfg = dict(S.CFG, d_model=d_model)
    monkeypatch.setattr(S, "CFG", cfg)
    monkeypatch.setattr(S, "KINDS", [kind])
    layers, dl = S.make_layers(d_model + rows, dev)
    C = 2 * cfg["hk"] * 128 + cfg["hv"] * 128

    def cache():
        n = int(kind == "delta")
        return {"length": 0, "conv": [torch.zeros(rows, C, 3)] * n,
                "state": [torch.zeros(rows, cfg["hv"], 128, 128)] * n,
                "k": [torch.zeros(rows, cfg["n_kv"], 8, 256, dtype=torch.bfloat16)] * (1 - n),
                "v": [torch.zeros(rows, cfg["n_kv"], 8, 256, dtype=torch.bfloat16)] * (1 - n)}
    c0, c1 = cache(), cache()
    stack = ops.HybridStack(cfg, [kind], dl, max_batch=rows, max_tokens=rows, max_context=8)
    g_ = torch.Generator().manual_seed(rows)
    for i in range(2):
        x = torch.randn(rows, 1, d_model, generator=g_)
        ref = R.hybrid_stack_forward(x.clone(), layers, [kind], c0, cfg)
        xp = perturb(x, 7 + i)
        ref_p = R.hybrid_stack_forward(xp.clone(), layers, [kind], c1, cfg)
        xd = x.to(dev)
        stack.forward(xd)
        got, ref, ref_p = xd.cpu() - x, ref - x, ref_p - xp
        flips = 3 * 4 * 2 ** -8 / min(d_model, 512) ** 0.5
        emax, erms = rel_err(got, ref), rms_err(got, ref)
        print(f"{kind} {d_model} x {rows}, step {i}: max {emax:.2e} rms {erms:.2e}", flush=True)
        assert emax < 2 * rel_err(ref_p, ref) + flips and erms < 2 * rms_err(ref_p, ref) + flips
    stack.close()
