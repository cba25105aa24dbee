"""The wide-load kernels of the small ops (csrc/mixer_small.hip) at the edges of their forms: gates with
one token a wave, two from 3072 waves on, four from 24576 of short rows, heads in groups of four, rows in pieces of 512 values; norms whose row or head ends inside a thread's pieces; widths that are no multiple of eight or
four take the narrow kernels."""
import pytest
import torch

from aegist_mixer import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 3, 63, 64, 66, 129, 191, 192, 767, 769])
@pytest.mark.parametrize("HV,D", [(1, 8), (3, 520), (6, 504), (32, 2048), (5, 12), (130, 512)])
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


# norms of n values: fp32 squares, sums and one rsqrt, a sum of at most 34 levels (8 x 4 values a thread, the
# wave's 6 and the block's 3, or 2 a lane and 6): (34 + 8) 2^-24 of the result, 2^-18 with room for the last
# products' and the sigmoid's roundings
REL = 2 ** -18


@pytest.mark.parametrize("rows", [1, 5])
@pytest.mark.parametrize("D", [4, 7, 1020, 1024, 1028, 2048, 4100, 8192, 8196])
def test_znorm_matches_exact(dev, rows, D):
    g_ = torch.Generator().manual_seed(rows + D)
    x, w = torch.randn(rows, D, generator=g_), (torch.randn(D, generator=g_) * 0.1).bfloat16()
    ref = x.double() * (x.double().square().mean(-1, keepdim=True) + 1e-6).rsqrt() * (1 + w.double())
    got = ops.engine_znorm(x.to(dev), w.to(dev)).cpu().double()
    assert ((got - ref).abs() <= REL * ref.abs()).all()


@pytest.mark.parametrize("T", [1, 3, 9])
@pytest.mark.parametrize("nq,dk", [(1, 4), (3, 60), (16, 128), (2, 30), (1, 132)])
def test_head_norms_match_exact(dev, T, nq, dk):
    g_ = torch.Generator().manual_seed(T + nq + dk)
    y = torch.randn(T, 3 * nq * dk, generator=g_)
    ref = y.double().clone()
    hd = ref[:, :2 * nq * dk].view(T, 2 * nq, dk)
    hd *= (hd.square().sum(-1, keepdim=True) + 1e-6).rsqrt()
    hd[:, :nq] *= dk ** -0.5
    yd = y.to(dev)
    ops.engine_l2norm_heads(yd, nq, dk, dk ** -0.5)
    assert ((yd.cpu().double() - ref).abs() <= REL * ref.abs()).all()
    o, z = (torch.randn(T, nq, dk, generator=g_) for _ in range(2))
    w = torch.randn(dk, generator=g_).bfloat16()
    od, zd = o.double(), z.double()
    ref = w.double() * od * (od.square().mean(-1, keepdim=True) + 1e-6).rsqrt() * torch.nn.functional.silu(zd)
    got = ops.engine_gated_norm(o.to(dev), z.to(dev), w.to(dev)).cpu().double()
    assert ((got - ref).abs() <= REL * ref.abs()).all()
