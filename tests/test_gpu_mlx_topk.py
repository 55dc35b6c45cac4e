"""The MLX-layout decode gate_up that selects its experts, against the router
top-k and the kernel that takes ids."""

import pytest
import torch

from titan_amd import ops
from titan_amd.moe_block import SharedExpert, SparseMoeBlock

pytestmark = pytest.mark.gpu


def _quant(g, lead, K, dev):
    w = torch.randint(-2 ** 31, 2 ** 31, (*lead, K // 8), dtype=torch.int32, device=dev, generator=g)
    s = (0.004 + 0.004 * torch.rand(*lead, K // 64, device=dev, generator=g)).to(torch.bfloat16)
    return w, s, (-7.5 * s.float()).to(torch.bfloat16)


def _deq64(q):
    w, s, b = q
    shifts = torch.arange(0, 32, 4, device=w.device, dtype=torch.int32)
    c = ((w.unsqueeze(-1) >> shifts) & 15).reshape(*w.shape[:-1], -1).double()
    return c * s.double().repeat_interleave(64, -1) + b.double().repeat_interleave(64, -1)


@pytest.mark.parametrize("norm", [True, False])
@pytest.mark.parametrize("T,k,E,K,I", [(1, 8, 128, 2048, 768), (3, 1, 1, 2048, 6), (16, 64, 64, 2048, 33),
                                       (2, 10, 600, 4096, 64), (5, 20, 256, 4096, 12)])
def test_gate_up_topk_over_mlx_weights(dev, T, k, E, K, I, norm):
    print(f"[case] MLX gate_up with top-k T={T} k={k} E={E} K={K} I={I} norm={norm}", flush=True)
    g = torch.Generator(device=dev).manual_seed(T + k + E)
    w = _quant(g, (E, 2 * I), K, dev)
    x = torch.randn(T, K, device=dev, generator=g).to(torch.bfloat16)
    lg = torch.randn(T, E, device=dev, generator=g)
    lg[:, ::3] = lg[:, ::3].round()  # ties among them
    h, idx, sc = ops.gate_up_silu_topk(x, *w, lg, k, norm)
    idx0, sc0 = ops.router_topk(lg, k, norm)
    assert torch.equal(idx, idx0) and torch.equal(sc, sc0)
    assert torch.equal(h, ops.gate_up_silu(x, *w, idx0))


@pytest.mark.parametrize("T", [1, 3, 7])
@pytest.mark.parametrize("resident,I,shared", [("tiles", 768, False), ("both", 512, False), ("tiles", 768, True),
                                               ("both", 512, True)])
def test_block_decode_over_mlx_weights(dev, T, resident, I, shared):
    print(f"[case] MLX-layout block decode T={T} {resident} I={I} shared={shared}", flush=True)
    g = torch.Generator(device=dev).manual_seed(T + I)
    E, H, k = 24, 2048, 8
    gu, dn = _quant(g, (E, 2 * I), H, dev), _quant(g, (E, H), I, dev)
    sgu, sdn = _quant(g, (1, 2 * I), H, dev), _quant(g, (1, H), I, dev)
    gate = (torch.randn(1, H, device=dev, generator=g) * H ** -0.5).to(torch.bfloat16)
    router = (torch.randn(E, H, device=dev, generator=g) * H ** -0.5).to(torch.bfloat16)
    x = torch.randn(T, H, device=dev, generator=g).to(torch.bfloat16)
    block = SparseMoeBlock(router, gu, dn, k, resident=resident, shared=SharedExpert(sgu, sdn, gate) if shared else None)
    y = block(x)
    idx, sc = block.route(x)
    ref = block.experts(x, idx, sc)
    if not shared:
        assert torch.equal(y, ref)
    else:  # the routed part's rounding, h's and the sum's, against the shared expert in 64 bits
        a, u = (x.double() @ _deq64(sgu)[0].t()).chunk(2, dim=-1)
        mlp = (torch.nn.functional.silu(a) * u) @ _deq64(sdn)[0].t()
        both = ref.double() + torch.sigmoid(x.double() @ gate.double().t()) * mlp
        assert bool(((y.double() - both).abs() <= 2.0 ** -7 * both.abs().max()).all())


# both sides of the lines between the selecting gate_up and a top-k launch: up to
# 256 experts top-32 and 63 pairs, up to 512 top-4 and 64 pairs x top-k, above
# top-16 and 24 pairs
@pytest.mark.parametrize("E,k,T,selects", [
    (256, 10, 6, True), (256, 32, 1, True), (256, 33, 1, False), (64, 21, 3, True), (64, 8, 8, False),
    (257, 4, 4, True), (257, 4, 5, False), (512, 5, 1, False), (512, 10, 1, False), (512, 1, 16, True),
    (513, 16, 1, True), (513, 17, 1, False), (1024, 8, 3, True), (1024, 5, 5, False)])
def test_block_decode_over_mlx_weights_selects_where_it_pays(dev, E, k, T, selects, monkeypatch):
    print(f"[case] MLX-layout block decode E={E} k={k} T={T}", flush=True)
    g = torch.Generator(device=dev).manual_seed(E + k + T)
    H, I = 2048, 128
    gu, dn = _quant(g, (E, 2 * I), H, dev), _quant(g, (E, H), I, dev)
    router = (torch.randn(E, H, device=dev, generator=g) * H ** -0.5).to(torch.bfloat16)
    block = SparseMoeBlock(router, gu, dn, k, resident="both", sort_min_pairs=1 << 20)
    x = torch.randn(T, H, device=dev, generator=g).to(torch.bfloat16)
    calls = []
    fused, plain = ops.gate_up_silu_topk, ops.router_topk
    monkeypatch.setattr(ops, "gate_up_silu_topk", lambda *a, **kw: calls.append(True) or fused(*a, **kw))
    monkeypatch.setattr(ops, "router_topk", lambda *a, **kw: calls.append(False) or plain(*a, **kw))
    y = block(x)
    assert calls == [selects]
    assert torch.equal(y, block.experts(x, *block.route(x)))
