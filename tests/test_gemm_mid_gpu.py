"""GPU parity of the projections of one row and more (csrc/gemv.hip, csrc/gemm_mid.hip) against fp64 dot
products of the exact operands, at the edges of their tiles (16 to 128 rows of X, 16 to 256 of W, 64 k
split over 1 to 8 wave groups). bf16 products are exact and summed in fp32: every output is within
K 2^-24 sum |x w s| of the exact one; fp32 X enters as bf16 hi + lo, within another 2^-16 sum |x w s|."""
import pytest
import torch

from aegist_mixer import ops

pytestmark = pytest.mark.gpu


def _operands(M, N, K, w8, xf, seed, dev):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(M, K, generator=g).to(torch.float32 if xf else torch.bfloat16)
    w = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8) if w8 else \
        (torch.randn(N, K, generator=g) * 0.02).to(torch.bfloat16)
    s = (torch.rand(N, generator=g) * 1e-2).to(torch.bfloat16) if w8 else None
    return x.to(dev), w.to(dev), None if s is None else s.to(dev)


def _check(out, y0, x, w, s, K):
    xd, wd = x.double(), w.double() * (1 if s is None else s.double()[:, None])
    ref, mag = xd @ wd.t(), xd.abs() @ wd.abs().t()
    if y0 is not None:
        ref, mag = ref + y0.double(), mag + y0.double().abs()
    bound = ((2.0 ** -16 if x.dtype == torch.float32 else 0) + (K + 2) * 2.0 ** -24) * mag + 1e-30
    worst = ((out.double() - ref).abs() / bound).max().item()
    print(f"  worst error / bound {worst:.3f}", flush=True)
    assert worst <= 1


@pytest.mark.parametrize("w8,xf", [(True, True), (False, False), (False, True), (True, False)])
@pytest.mark.parametrize("M,N,K", [(17, 16, 16), (31, 33, 48), (32, 100, 80), (33, 2048, 512), (64, 2048, 4096),
                                   (65, 1000, 144), (129, 4096, 2048), (300, 8192, 128), (300, 2048, 2064),
                                   (600, 4100, 320), (1030, 8192, 192)])
def test_mid_batch_matches_exact(dev, M, N, K, w8, xf):
    print(f"mid M={M} N={N} K={K} w8={w8} xf={xf}", flush=True)
    x, w, s = _operands(M, N, K, w8, xf, M + N + K, dev)
    _check(ops.linear(x, w, s), None, x, w, s, K)
    y0 = torch.randn(M, N, generator=torch.Generator().manual_seed(1)).to(dev)
    out = ops.linear(x, w, s, out=y0.clone(), accumulate=True)
    _check(out, y0, x, w, s, K)


@pytest.mark.parametrize("w8,xf", [(True, True), (False, False), (False, True), (True, False)])
@pytest.mark.parametrize("M,N,K", [(17, 1, 16), (32, 2048, 512), (33, 1000, 1040), (47, 1365, 1552), (64, 2047, 976),
                                   (100, 2300, 272), (4096, 16, 1024), (4095, 17, 1040),   # 16 rows a tile, one round
                                   (33, 5120, 1536), (24, 8190, 1552), (130, 2100, 1040), (600, 4100, 1552)])  # sized, odd steps
def test_one_round_and_odd_steps(dev, M, N, K, w8, xf):
    print(f"round M={M} N={N} K={K} w8={w8} xf={xf}", flush=True)
    x, w, s = _operands(M, N, K, w8, xf, M + N + K, dev)
    _check(ops.linear(x, w, s), None, x, w, s, K)
    y0 = torch.randn(M, N, generator=torch.Generator().manual_seed(1)).to(dev)
    _check(ops.linear(x, w, s, out=y0.clone(), accumulate=True), y0, x, w, s, K)


@pytest.mark.parametrize("w8,xf", [(True, True), (False, False)])
def test_mid_batch_segments_and_strides(dev, w8, xf):
    """Four weights in one launch (sizes that end inside a tile), X rows inside wider rows and
    outputs whose rows are not 16-byte aligned."""
    M, K, Ns = 50, 256, (300, 32, 7, 130)
    ws = [_operands(M, N, K, w8, xf, N, dev) for N in Ns]
    x = _operands(M, 1, K + 64, w8, xf, 3, dev)[0][:, :K]
    outs = [torch.full((M, N + 3), 7.0, device=dev)[:, :N] for N in Ns]
    ops.linear_multi(x, [w[1] for w in ws], [w[2] for w in ws] if w8 else None, outs=outs)
    for (_, w, s), o in zip(ws, outs):
        _check(o, None, x, w, s, K)
        assert (o.as_strided((M, 3), (o.stride(0), 1), o.shape[1]) == 7).all()


@pytest.mark.parametrize("w8,xf", [(True, True), (False, False), (False, True), (True, False)])
@pytest.mark.parametrize("M,N,K", [(1, 1, 16), (1, 5, 48), (2, 515, 1040), (1, 1030, 2064), (2, 2049, 512), (1, 4099, 528),
                                   (1, 7, 1552), (2, 1029, 3088), (1, 4097, 4112), (2, 3, 8192),
                                   (2, 8200, 32), (1, 8192, 2048), (3, 33, 16), (5, 100, 1040), (16, 2048, 2064),
                                   (7, 6150, 64), (16, 8192, 512), (11, 9000, 256), (9, 16500, 80)])
def test_small_batch_matches_exact(dev, M, N, K, w8, xf):
    """One and two rows (csrc/gemv.hip: rows and pieces that end inside a wave's) and 3 to 16 (the small
    forms of gemm_mid.hip, the streamed weights)."""
    print(f"small M={M} N={N} K={K} w8={w8} xf={xf}", flush=True)
    x, w, s = _operands(M, N, K, w8, xf, M + N + K, dev)
    _check(ops.linear(x, w, s), None, x, w, s, K)
    y0 = torch.randn(M, N, generator=torch.Generator().manual_seed(1)).to(dev)
    _check(ops.linear(x, w, s, out=y0.clone(), accumulate=True), y0, x, w, s, K)


@pytest.mark.parametrize("M", [1, 2, 6])
@pytest.mark.parametrize("w8,xf", [(True, True), (False, False)])
def test_small_batch_segments_and_strides(dev, M, w8, xf):
    K, Ns = 272, (300, 32, 7, 130)
    ws = [_operands(M, N, K, w8, xf, N, dev) for N in Ns]
    x = _operands(M, 1, K + 64, w8, xf, 3, dev)[0][:, :K]
    outs = [torch.full((M, N + 3), 7.0, device=dev)[:, :N] for N in Ns]
    ops.linear_multi(x, [w[1] for w in ws], [w[2] for w in ws] if w8 else None, outs=outs)
    for (_, w, s), o in zip(ws, outs):
        _check(o, None, x, w, s, K)
        assert (o.as_strided((M, 3), (o.stride(0), 1), o.shape[1]) == 7).all()


@pytest.mark.parametrize("M", [1, 2])
@pytest.mark.parametrize("K", [48, 1552, 2064])
def test_one_infinite_weight_is_one_infinite_output(dev, M, K):
    """The loads past a row's end repeat its first values, which must not turn Inf into NaN."""
    x, w, _ = _operands(M, 9, K, False, True, K, dev)
    w[3, 0] = float("inf")
    y = ops.linear(x, w)
    assert torch.isinf(y[:, 3]).all() and torch.equal(y[:, 3] > 0, x[:, 0] > 0)
    assert torch.isfinite(y[:, :3]).all() and torch.isfinite(y[:, 4:]).all()


@pytest.mark.parametrize("w8,M,N,K,bar", [
    (False, 3, 8192, 2048, 1.02e-7), (False, 16, 8192, 2048, 1.03e-7), (False, 16, 2048, 4096, 1.17e-7),
    (False, 16, 512, 2048, 0.98e-7), (False, 48, 8192, 2048, 1.03e-7), (False, 64, 12352, 2048, 1.03e-7),
    (False, 17, 32768, 2048, 1.33e-7), (True, 16, 8192, 2048, 0.73e-7), (True, 64, 12352, 2048, 0.74e-7),
    (True, 300, 8192, 2048, 0.79e-7), (True, 600, 4096, 8192, 1.61e-7)])
def test_exact_operands_are_summed_in_short_chains(dev, w8, M, N, K, bar):
    """bf16 X: the products are exact, and the error is that of the fp32 sums, which grows with the length of
    the chains that are added one product after the other. As a 2-norm over 8192 outputs and more of these very
    operands it is stable, and may not exceed what chains of 128 to 512 products left (the bars: the error
    of the row-tile kernel that these tiles replaced, measured on the same operands, and 1%). One chain of a
    K group each left 1.31e-7, 1.30e-7, 1.37e-7, 1.03e-7, 1.32e-7, 1.86e-7, 1.87e-7 with bf16 W, 0.77e-7,
    1.03e-7, 1.53e-7 and 3.85e-7 with int8."""
    x, w, _ = _operands(M, N, K, w8, False, M + N, dev)
    ref = x.double() @ w.double().t()
    err = ((ops.linear(x, w).double() - ref).norm() / ref.norm()).item()
    print(f"  {M} x {N} x {K} w8={w8}: {err:.3e}, bar {bar:.3e}", flush=True)
    assert err < bar
