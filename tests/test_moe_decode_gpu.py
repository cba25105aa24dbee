"""GPU parity of the experts' decode path (csrc/moe_decode.hip: up to 512 picks, at most two per expert
on average, row lengths 512 / 1024 / 2048) against the fp64 oracle: one pick to the path's largest
batch, experts shared by 1 to 9 picks (workgroups of 1 to 4), out-of-range ids, every row length.
The activations enter as bf16 hi + lo and sums are fp32, as in the larger batches' tiles: bar 5e-5."""
import pytest
import torch

from conftest import rel_err
from oracle import mixer_ref as R
from test_moe_gpu import _experts

from aegist_mixer import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,D,I,E,K,hot,bad", [(1, 2048, 512, 1, 1, 1, False), (1, 2048, 512, 256, 8, 256, False),
                                               (9, 2048, 512, 64, 8, 8, False), (8, 1024, 512, 32, 8, 9, True),
                                               (9, 512, 1024, 40, 8, 12, True), (5, 512, 2048, 24, 3, 24, False),
                                               (16, 2048, 512, 256, 8, 256, True), (64, 512, 512, 256, 8, 200, False),
                                               (32, 1024, 1024, 256, 16, 16, False)])
def test_moe_decode_matches_oracle(dev, T, D, I, E, K, hot, bad):
    print(f"moe decode T={T} D={D} I={I} E={E} K={K} hot={hot} bad={bad}", flush=True)
    g = torch.Generator().manual_seed(T * 31 + D + I)
    rows, h = _experts(E, D, I, T + E), torch.randn(T, D, generator=g)
    idx = torch.stack([torch.randperm(hot, generator=g)[:K] for _ in range(T)]).int()
    if bad:
        idx[::3, 0], idx[1::4, -1] = E + 5, -1
    wts, x0 = torch.rand(T, K, generator=g), torch.randn(T, D, generator=g)
    ysh, wg = torch.randn(T, D, generator=g), (torch.randn(D, generator=g) * 0.05).bfloat16()
    x, hd, rd = x0.to(dev), h.to(dev), rows.to(dev)
    ops.moe_experts(hd, rd, idx.to(dev), wts.to(dev), x, I, ysh=ysh.to(dev), wg=wg.to(dev))
    torch.cuda.synchronize()
    ref = R.moe_experts(h, rows, idx.long(), wts, D, I) + torch.sigmoid(h.double() @ wg.double())[:, None] * ysh.double()
    err = rel_err(x.cpu().double() - x0.double(), ref)
    print(f"  rel err {err:.2e}", flush=True)
    assert err < 5e-5


@pytest.mark.parametrize("T,E,K", [(3, 16, 4), (2, 64, 8), (5, 65, 16), (4, 1000, 8), (2, 2000, 3), (2, 4096, 16)])
def test_router_rounds_take_the_lowest_of_equals(dev, T, E, K):
    """Equal probabilities in lanes and registers of every distance: groups of experts share one weight
    row, so the K picks are the lowest ids of the best groups, in order."""
    g = torch.Generator().manual_seed(E)
    base = torch.randn(5, 256, generator=g).bfloat16()
    W, h = base[torch.randint(0, 5, (E,), generator=g)], torch.randn(T, 256, generator=g)
    idx, _ = ops.router_topk(h.to(dev), W.to(dev), K)
    ref = torch.sort(-(h.double() @ W.double().t()), dim=-1, stable=True).indices[:, :K]
    assert torch.equal(idx.cpu().long(), ref)


@pytest.mark.parametrize("T,D,I,E,K,hot", [(600, 384, 128, 8, 2, 8), (700, 128, 384, 300, 2, 300), (90, 640, 256, 20, 8, 20),
                                           (130, 2048, 128, 8, 4, 5), (33, 256, 2048, 4, 4, 4), (9000, 256, 128, 64, 8, 64),
                                           (65, 1024, 512, 16, 16, 16)])
def test_moe_prefill_tiles_match_oracle(dev, T, D, I, E, K, hot):
    """The prefill tiles (csrc/moe.hip) at 1 to 64 picks a tile, row lengths whose groups are no multiple of
    8 (6, 10, 2), outputs and units that end inside a workgroup, and a grouping of more than 64 blocks; the
    700 tokens of 300 narrow experts take the 64-row workgroups of up to 16 picks."""
    print(f"moe prefill T={T} D={D} I={I} E={E} K={K}", flush=True)
    g = torch.Generator().manual_seed(T + D + I)
    rows, h = _experts(E, D, I, T + E), torch.randn(T, D, generator=g)
    idx = torch.stack([torch.randperm(hot, generator=g)[:K] for _ in range(T)]).int()
    idx[::7, 0] = -1 if K > 1 else idx[::7, 0]
    wts = torch.rand(T, K, generator=g)
    x, hd, rd = torch.zeros(T, D, device=dev), h.to(dev), rows.to(dev)
    ops.moe_experts(hd, rd, idx.to(dev), wts.to(dev), x, I)
    torch.cuda.synchronize()
    err = rel_err(x, R.moe_experts(h, rows, idx.long(), wts, D, I))
    print(f"  rel err {err:.2e}", flush=True)
    assert err < 5e-5


@pytest.mark.parametrize("bad", ["dtype", "size", "stride"])
def test_moe_forward_refuses_bad_shared_scales(dev, bad):
    """The shared expert's gate and up projections go in one launch, under the checks of each alone."""
    D, I = 512, 512
    g = torch.Generator().manual_seed(2)
    w = torch.randint(-127, 128, (I, D), generator=g, dtype=torch.int8).to(dev)
    good = torch.ones(I, dtype=torch.bfloat16, device=dev)
    sc = {"dtype": good.float(), "size": good.repeat(2), "stride": good.repeat(2)[::2]}[bad]
    h, x = torch.randn(2, D, generator=g).to(dev), torch.zeros(2, D, device=dev)
    router = torch.randn(8, D, generator=g).bfloat16().to(dev)
    with pytest.raises(ops.AegistError):
        ops.moe_forward(h, x, router, _experts(8, D, I, 3).to(dev), I, 2, shared=((w, good), (w, sc), (w, good)),
                        shared_gate=torch.zeros(D, dtype=torch.bfloat16, device=dev))


def test_more_picks_of_one_expert_than_tile_products_fit_32_bits(dev):
    """400000 picks of one expert: its tiles' boundaries must not be formed by products of two counts."""
    T, D, I = 400_000, 128, 128
    g = torch.Generator().manual_seed(5)
    rows, h = _experts(1, D, I, 5), torch.randn(T, D, generator=g)
    idx, wts = torch.zeros(T, 1, dtype=torch.int32), torch.rand(T, 1, generator=g)
    x = torch.zeros(T, D, device=dev)
    ops.moe_experts(h.to(dev), rows.to(dev), idx.to(dev), wts.to(dev), x, I)
    assert rel_err(x, R.moe_experts(h, rows, idx.long(), wts, D, I)) < 5e-5


@pytest.mark.parametrize("T,D,I,E,K", [(70, 384, 256, 256, 8), (96, 256, 256, 8, 2), (128, 384, 256, 8, 2), (2048, 256, 256, 4, 2),
                                       (5000, 256, 256, 8, 2), (8000, 256, 256, 8, 2), (1, 256, 768, 64, 8), (9, 512, 512, 8, 2),
                                       (100, 256, 192, 8, 4)])
def test_moe_tile_sizes_match_oracle(dev, T, D, I, E, K):
    """Every size of tile the rule picks (test_moe_tiles.py has it for these batches): prefill tiles of up to
    64 with 1 to 8 picks, 64-row workgroups at 17 to 32 picks, prefill tiles of up to 16, 32, 48 and 64;
    64-row workgroups for one token and few experts, and for units that are no multiple of 128."""
    print(f"moe tiles T={T} D={D} I={I} E={E} K={K}", flush=True)
    g = torch.Generator().manual_seed(T + D + I)
    rows, h = _experts(E, D, I, T + E), torch.randn(T, D, generator=g)
    idx = torch.topk(torch.rand(T, E, generator=g), K, -1).indices.int()
    wts = torch.rand(T, K, generator=g)
    x = torch.zeros(T, D, device=dev)
    ops.moe_experts(h.to(dev), rows.to(dev), idx.to(dev), wts.to(dev), x, I)
    err = rel_err(x, R.moe_experts(h, rows, idx.long(), wts, D, I))
    print(f"  rel err {err:.2e}", flush=True)
    assert err < 5e-5
