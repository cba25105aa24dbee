"""Projections whose operands pass 2 GiB, which csrc/proj.hip cuts into blocks of rows for kernels that address
through 31-bit byte offsets: a weight, an activation matrix, rows so long or so far apart that one at a time is
taken. Operands are small integers and every sum stays below 2^24, so results are exact: a block at a wrong
offset shows in any output."""
import pytest
import torch

from aegist_mixer import ops

pytestmark = pytest.mark.gpu
LIM = 2 ** 31 - 16


def _ints(dev, *shape, dtype, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    t = torch.empty(shape, dtype=dtype, device=dev)
    for part in t.view(-1).split(1 << 28):  # (no 8-byte integers of the whole)
        part.copy_(torch.randint(-1, 2, part.shape, generator=g, device=dev, dtype=torch.int8))
    return t


def _exact(x, w):
    """x w^T in fp64: products over pieces of W's rows, or, for few long rows (where a matrix product would leave
    the whole length to one workgroup), sums of elementwise products over pieces of the length."""
    M, N, K = x.shape[0], w.shape[0], w.shape[1]
    if K < 1 << 20:
        return torch.cat([x.double() @ p.double().t() for p in w.split((1 << 26) // K)], 1)
    out = torch.zeros(M, N, dtype=torch.float64, device=x.device)
    for m in range(M):
        for n in range(N):
            for k in range(0, K, 1 << 26):
                out[m, n] += (x[m, k:k + (1 << 26)].float() * w[n, k:k + (1 << 26)].float()).sum(dtype=torch.float64)
    return out


@pytest.mark.parametrize("M", [1, 3, 20])
@pytest.mark.parametrize("wt,xt,K", [(torch.bfloat16, torch.bfloat16, 1024), (torch.int8, torch.float32, 2048)])
def test_weight_past_2_gib(dev, wt, xt, K, M):
    N = LIM // (K * wt.itemsize) + 700
    print(f"weight {N} x {K} {wt}, {M} rows", flush=True)
    w, x = _ints(dev, N, K, dtype=wt, seed=1), _ints(dev, M, K, dtype=xt, seed=2)
    y0 = _ints(dev, M, N, dtype=torch.float32, seed=3)
    y = ops.linear(x, w, out=y0.clone(), accumulate=True)
    assert torch.equal(y.double(), _exact(x, w) + y0.double())


@pytest.mark.parametrize("wt,xt", [(torch.bfloat16, torch.bfloat16), (torch.int8, torch.float32)])
def test_activations_past_2_gib(dev, wt, xt):
    K, Ns = 512, (64, 40)
    M = LIM // (K * xt.itemsize) + 300
    print(f"activations {M} x {K} {xt}", flush=True)
    ws, x = [_ints(dev, n, K, dtype=wt, seed=n) for n in Ns], _ints(dev, M, K, dtype=xt, seed=2)
    for y, w in zip(ops.linear_multi(x, ws), ws):
        for m in range(0, M, 1 << 18):
            assert torch.equal(y[m:m + (1 << 18)].double(), _exact(x[m:m + (1 << 18)], w))


@pytest.mark.parametrize("wt,xt,K,M", [(torch.bfloat16, torch.bfloat16, 2 ** 27, 2), (torch.int8, torch.float32, 2 ** 28, 1)])
def test_rows_of_2_gib_in_eight(dev, wt, xt, K, M):
    """Eight rows of W pass the limit: one row of X at a time."""
    print(f"9 rows of {K} {wt}, {M} rows of X", flush=True)
    w, x = _ints(dev, 9, K, dtype=wt, seed=1), _ints(dev, M, K, dtype=xt, seed=2)
    assert torch.equal(ops.linear(x, w).double(), _exact(x, w))


def test_rows_of_x_far_apart(dev):
    """Three rows of X reach past the limit through their stride alone."""
    K, ld = 512, LIM // 8
    w, rows = _ints(dev, 100, K, dtype=torch.int8, seed=1), _ints(dev, 4, K, dtype=torch.float32, seed=2)
    ld -= ld % 4
    x = torch.zeros(3 * ld + K, device=dev).as_strided((4, K), (ld, 1))
    x.copy_(rows)
    assert torch.equal(ops.linear(x, w).double(), _exact(rows, w))
