"""The gates' and the embedding's wide-load kernels (csrc/mixer_small.hip) at the edges of their forms:
one token a wave below 64 tokens, four from there on, heads in groups of four, rows in pieces of 512
values; widths that are no multiple of eight take the narrow kernels."""
import pytest
import torch

from aegist_mixer import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 3, 63, 64, 66, 129])
@pytest.mark.parametrize("HV,D", [(1, 8), (3, 520), (6, 504), (32, 2048), (5, 12)])
def test_gates_match_exact(dev, T, HV, D):
    g_ = torch.Generator().manual_seed(T * HV + D)
    h = torch.randn(T, D, generator=g_)
    wb, wa = ((torch.randn(HV, D, generator=g_) * D ** -0.5).bfloat16() for _ in range(2))
    a_log, dt = (torch.randn(HV, generator=g_).bfloat16() for _ in range(2))
    gb = ops.engine_delta_gates(*(t.to(dev) for t in (h, wb, wa, a_log, dt))).cpu().double()
    hd, b, a = h.double(), wb.double(), wa.double()
    beta = torch.sigmoid(hd @ b.T)
    g = -a_log.double().exp() * torch.nn.functional.softplus(hd @ a.T + dt.double())
    # fp32 products and sums over D / 64 values a lane and six more levels: an absolute error of at most
    # (D / 64 + 6) 2^-24 sum |h w| in the argument. sigmoid's slope is at most 1/4; softplus's is at most
    # 1, times exp(a_log); expf, log1pf and the last product add 2^-21 of the result, and log1pf(expf(x))
    # at small x 2^-23 of it besides
    depth = (D / 64 + 6) * 2 ** -24
    err_b, err_a = (hd.abs() @ w.abs().T * depth for w in (b, a))
    gg, bb = gb.view(T, 2, HV).unbind(1)
    assert ((bb - beta).abs() <= err_b / 4 + 2 ** -21 * beta).all()
    assert ((gg - g).abs() <= a_log.double().exp() * err_a + 2 ** -20 * g.abs()).all()


@pytest.mark.parametrize("n,D", [(1, 8), (7, 12), (5, 2048), (64, 1032), (3, 4104)])
def test_embed_matches_rows(dev, n, D):
    g_ = torch.Generator().manual_seed(n + D)
    table = torch.randn(50, D, generator=g_).bfloat16()
    ids = torch.randint(0, 50, (n,), generator=g_, dtype=torch.int32)
    ids[0] = 49
    out = ops.embed(table.to(dev), ids.to(dev)).cpu()
    assert torch.equal(out, table[ids.long()].float())
