"""Operands that are not on a GPU are refused before any launch: a kernel given a host address faults."""
import pytest
import torch

from aegist_mixer import ops


class _OnGpu(torch.Tensor):
    is_cuda = property(lambda self: True)


def _t(*shape, dtype=torch.bfloat16):
    return torch.zeros(*shape, dtype=dtype).as_subclass(_OnGpu)


@pytest.fixture
def launches(monkeypatch):
    seen = []
    monkeypatch.setattr(ops, "call", lambda name, *args: seen.append(name))
    monkeypatch.setattr(ops, "_stream", lambda device=None: 0)
    return seen


@pytest.mark.parametrize("host", [None, "x", "weight", "scale", "out"])
def test_linear_multi_refuses_host_operands(launches, host):
    def on(what, t):
        return t.as_subclass(torch.Tensor) if what == host else t
    x = on("x", _t(2, 32))
    w = [_t(16, 32, dtype=torch.int8), on("weight", _t(8, 32, dtype=torch.int8))]
    s = [_t(16), on("scale", _t(8))]
    o = [_t(2, 16, dtype=torch.float32), on("out", _t(2, 8, dtype=torch.float32))]
    if host is None:
        ops.linear_multi(x, w, s, outs=o)
        assert launches == ["aegist_linear_multi"]
        return
    with pytest.raises(ops.AegistError, match="not on a GPU"):
        ops.linear_multi(x, w, s, outs=o)
    assert not launches


@pytest.mark.gpu
@pytest.mark.parametrize("host", ["gate", "up", "scale"])
def test_moe_forward_refuses_host_shared_operands(dev, launches, host):
    """The shared expert's gate and up projections, with every launch replaced by a record of its name."""
    D = I = 512
    w, s = torch.zeros(I, D, dtype=torch.int8, device=dev), torch.ones(I, dtype=torch.bfloat16, device=dev)
    shared = ((w.cpu() if host == "gate" else w, s), (w.cpu() if host == "up" else w, s.cpu() if host == "scale" else s), (w, s))
    h = torch.zeros(2, D, device=dev)
    with pytest.raises(ops.AegistError, match="not on a GPU"):
        ops.moe_forward(h, h.clone(), torch.zeros(8, D, dtype=torch.bfloat16, device=dev), None, I, 2, shared=shared,
                        shared_gate=torch.zeros(D, dtype=torch.bfloat16, device=dev))
    assert launches == ["aegist_router_topk_ws"]
