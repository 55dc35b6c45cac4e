"""SwitchGLU's own kernels (row gather, activation, un-sort) against the torch
expressions they stand for, and where the layer keeps those."""

import pytest
import torch

from titan_amd import ops, switch_layers
from titan_amd.switch_layers import QuantizedSwitchLinear, SwiGLU, SwitchGLU, swiglu

pytestmark = pytest.mark.gpu


def _quant(g, lead, K, dev):
    w = torch.randint(-2 ** 31, 2 ** 31, (*lead, K // 8), dtype=torch.int32, device=dev, generator=g)
    s = (0.004 + 0.004 * torch.rand(*lead, K // 64, device=dev, generator=g)).to(torch.bfloat16)
    return w, s, (-7.5 * s.float()).to(torch.bfloat16)


@pytest.mark.parametrize("n,R,D,div", [(1, 1, 8, 1), (65, 7, 24, 10), (640, 64, 2048, 10), (1000, 1000, 520, 1)])
def test_gather_rows(dev, n, R, D, div):
    g = torch.Generator(device=dev).manual_seed(n + D)
    x = torch.randn(R, D, device=dev, generator=g).to(torch.bfloat16)
    rows = torch.randint(0, R * div, (n,), dtype=torch.int32, device=dev, generator=g)
    assert torch.equal(ops.gather_rows(x, rows, div), x[(rows // div).long()])


@pytest.mark.parametrize("R,I", [(1, 8), (3, 40), (513, 512), (70, 768)])
def test_swiglu_kernel(dev, R, I):
    """Within the fp32 error of exp and the division of the torch expression,
    before the same rounding: at most one bf16 ULP, and rarely."""
    g = torch.Generator(device=dev).manual_seed(R + I)
    gu = (4 * torch.randn(R, 1, 2 * I, device=dev, generator=g)).to(torch.bfloat16)
    gu[0, 0, :4] = torch.tensor([0.0, -0.0, 88.0, -100.0], dtype=torch.bfloat16)
    h = ops.swiglu(gu)
    a, u = gu.chunk(2, dim=-1)
    ref = swiglu(a, u)
    assert h.shape == ref.shape
    ulp = (h.view(torch.int16).int() - ref.view(torch.int16).int()).abs()
    assert int(ulp.max()) <= 1 and float((ulp != 0).float().mean()) < 1e-3
    exact = a.double() * torch.sigmoid(a.double()) * u.double()
    assert bool(((h.double() - exact).abs() <= 2.0 ** -8 * exact.abs() * 1.001 + 1e-38).all())


@pytest.mark.parametrize("T", [3, 7, 90])
@pytest.mark.parametrize("how", ["default", "module of its own", "separate projections", "odd stride", "needs grad"])
def test_layer_over_its_kernels_and_without(dev, T, how, monkeypatch):
    """The layer's result over every route equals the one with its kernels off
    (the activation's rounding apart)."""
    g = torch.Generator(device=dev).manual_seed(T)
    E, K, I, k = 16, 512, 256, 10
    gate, up = _quant(g, (E, I), K, dev), _quant(g, (E, I), K, dev)
    down = QuantizedSwitchLinear(*_quant(g, (E, K), I, dev))
    if how == "separate projections":
        layer = SwitchGLU(down, gate_proj=QuantizedSwitchLinear(*gate), up_proj=QuantizedSwitchLinear(*up))
    else:
        fused = QuantizedSwitchLinear(*(torch.cat(p, dim=1) for p in zip(gate, up)))

        class Mine(SwiGLU):
            pass

        layer = SwitchGLU(down, gate_up_proj=fused, activation=Mine() if how == "module of its own" else None)
    x = torch.randn(T, K, device=dev, generator=g).to(torch.bfloat16)
    if how == "odd stride":
        x = torch.cat([x, x], dim=1)[:, :K]
    idx = torch.rand(T, E, device=dev, generator=g).topk(k, dim=-1)[1].to(torch.int32)
    if how == "needs grad":
        x.requires_grad_(True)
    y = layer(x, idx)
    monkeypatch.setattr(switch_layers, "_plain", lambda t, width: False)
    ref = layer(x, idx)
    assert y.shape == ref.shape == (T, k, K)
    y, ref = y.detach(), ref.detach()
    err = (y.double() - ref.double()).norm() / ref.double().norm()
    assert float(err) < 2.0 ** -9  # single ULPs of h, seldom


@pytest.mark.parametrize("rows", [1, 63])
def test_ids_of_more_rows_than_x_has_are_refused(dev, rows):
    g = torch.Generator(device=dev).manual_seed(rows)
    E, K, I, k = 16, 512, 256, 2
    layer = SwitchGLU(QuantizedSwitchLinear(*_quant(g, (E, K), I, dev)),
                      gate_up_proj=QuantizedSwitchLinear(*_quant(g, (E, 2 * I), K, dev)))
    x = torch.randn(64, K, device=dev, generator=g).to(torch.bfloat16)
    idx = torch.randint(0, E, (64, k), dtype=torch.int32, device=dev, generator=g)
    with pytest.raises(IndexError, match="rows"):
        layer(x[:rows], idx)
    # more rows than ids are ignored, as indexing by the ids' rows does
    assert torch.equal(layer(x, idx[:40]), layer(x[:40], idx[:40]))


@pytest.mark.parametrize("T", [3, 90])
@pytest.mark.parametrize("what", ["function", "call"])
def test_a_replaced_default_activation_runs(dev, T, what, monkeypatch):
    """swiglu and SwiGLU.__call__ put in the place of the module's own."""
    g = torch.Generator(device=dev).manual_seed(T)
    E, K, I, k = 16, 512, 256, 4
    layer = SwitchGLU(QuantizedSwitchLinear(*_quant(g, (E, K), I, dev)),
                      gate_up_proj=QuantizedSwitchLinear(*_quant(g, (E, 2 * I), K, dev)))
    x = torch.randn(T, K, device=dev, generator=g).to(torch.bfloat16)
    idx = torch.randint(0, E, (T, k), dtype=torch.int32, device=dev, generator=g)
    calls = []

    def mine(gate, x):
        calls.append(tuple(gate.shape))
        return x - gate

    if what == "function":
        monkeypatch.setattr(switch_layers, "swiglu", mine)
    else:
        monkeypatch.setattr(SwiGLU, "__call__", lambda self, x, gate: mine(gate, x))
    y = layer(x, idx)
    assert len(calls) == 1
    monkeypatch.undo()
    layer.activation = lambda x, gate: x - gate
    assert torch.equal(y, layer(x, idx))


def test_plain_tensors_only(dev, monkeypatch):
    """What keeps a tensor from the layer's own kernels."""
    from torch.autograd import forward_ad

    plain = switch_layers._plain
    t = torch.zeros(4, 64, dtype=torch.bfloat16, device=dev)
    assert plain(t, 64) and plain(t[2:], 64) and plain(torch.zeros(0, 64, dtype=torch.bfloat16, device=dev), 64)
    assert not plain(t.cpu(), 64)
    assert not plain(t.float(), 64)
    assert not plain(t[:, :32], 32)                      # a stride
    assert not plain(t.reshape(-1)[4:68].reshape(1, 64), 64)  # 8-byte alignment
    assert not plain(torch.zeros(4, 60, dtype=torch.bfloat16, device=dev), 60)

    class Sub(torch.Tensor):
        pass

    assert not plain(t.as_subclass(Sub), 64)
    p = t.clone().requires_grad_(True)
    assert not plain(p, 64)
    with torch.no_grad():
        assert plain(p, 64)
    with forward_ad.dual_level():
        assert not plain(t, 64)
        assert not plain(forward_ad.make_dual(t, t), 64)
    seen = []
    torch.func.vmap(lambda r: seen.append(plain(r, 64)) or r)(t)
    torch.func.grad(lambda r: seen.append(plain(r, 64)) or r.float().sum())(t)
    torch.func.jvp(lambda r: seen.append(plain(r, 64)) or r * 2, (t,), (t,))
    torch.func.functionalize(lambda r: seen.append(plain(r, 64)) or r * 2)(t)
    torch.jit.trace(lambda r: seen.append(plain(r, 64)) or r * 2, (t,), check_trace=False)
    assert len(seen) == 5 and not any(seen)
    monkeypatch.setattr(torch.compiler, "is_compiling", lambda: True)
    assert not plain(t, 64)
