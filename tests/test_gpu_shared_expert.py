"""The shared expert as one more slot of the decode kernels
(qmoe_moe_gate_up_swiglu_tiles_topk_shared, qmoe_moe_down_wsum_tiles_shared) and
one more expert of the sorted path (qmoe_route_block and the *_shared entry points)
against the id-taking kernels and a 64-bit product."""

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


def _close_bf16(y, ref):
    """One bf16 rounding (2^-9 of a value) of sums in fp32: n * 2^-24 of the
    sum of magnitudes, far below 2^-14 of the largest output."""
    err = (y.double() - ref).abs()
    assert bool((err <= 2.0 ** -8 * ref.abs() + 2.0 ** -14 * ref.abs().max()).all()), float(err.max())


@pytest.mark.parametrize("norm", [True, False])
@pytest.mark.parametrize("T,k,H,E", [(1, 10, 2048, 256), (2, 1, 2048, 3), (16, 15, 4096, 300), (3, 4, 6144, 5),
                                     (5, 2, 8192, 64)])
def test_shared_slot_decode(dev, T, k, H, E, norm):
    print(f"[case] shared slot T={T} k={k} H={H} E={E} norm={norm}", flush=True)
    g = torch.Generator(device=dev).manual_seed(T * 100 + k)
    I = 512
    gu, dn = _quant(g, (E, 2 * I), H, dev), _quant(g, (E, H), I, dev)
    sgu, sdn = _quant(g, (1, 2 * I), H, dev), _quant(g, (1, H), I, dev)
    gate = (torch.randn(1, H, device=dev, generator=g) * H ** -0.5).to(torch.bfloat16)
    x = torch.randn(T, H, device=dev, generator=g).to(torch.bfloat16)
    logits = torch.randn(T, E, device=dev, generator=g)
    tw, stw = ops.repack_tiles(*gu, swiglu_pairs=True), ops.repack_tiles(*sgu, swiglu_pairs=True)
    td, std = ops.repack_tiles(*dn), ops.repack_tiles(*sdn)
    h, idx, sc = ops.gate_up_silu_tiles_topk_shared(x, tw, logits, k, stw, gate, norm)
    h0, idx0, sc0 = ops.gate_up_silu_tiles_topk(x, tw, logits, k, norm)
    assert torch.equal(h[:, :k], h0) and torch.equal(idx[:, :k], idx0) and torch.equal(sc[:, :k], sc0)
    zeros = torch.zeros(T, 1, dtype=torch.int32, device=dev)
    assert torch.equal(h[:, k:], ops.gate_up_silu_tiles(x, stw, zeros))
    assert bool((idx[:, k] == E).all())
    z = x.double() @ gate.double().t()
    # the logit's fp32 sum is within K * 2^-24 of sum |x w|; the sigmoid's slope is at most 1/4
    bound = 0.25 * H * 2.0 ** -24 * (x.double().abs() @ gate.double().abs().t()) + 4 * 2.0 ** -24
    assert bool(((sc[:, k:].double() - torch.sigmoid(z)).abs() <= bound).all())
    y = ops.down_wsum_tiles_shared(h, td, idx, sc, std)
    ref = torch.zeros(T, H, dtype=torch.float64, device=dev)
    dn64, sdn64 = _deq64(dn) if E <= 5 else None, _deq64(sdn)[0]
    for t in range(T):
        for j in range(k):
            e = int(idx[t, j])
            we = dn64[e] if dn64 is not None else _deq64(tuple(q[e] for q in dn))
            ref[t] += sc[t, j].double() * (we @ h[t, j].double())
        ref[t] += sc[t, k].double() * (sdn64 @ h[t, k].double())
    _close_bf16(y, ref)


@pytest.mark.parametrize("T", [1, 6, 7, 16, 17, 200])
@pytest.mark.parametrize("k,S", [(10, 512), (16, 512), (10, 768)])
def test_block_with_shared_expert_matches_its_parts(dev, T, k, S):
    """The block over every dispatch of its shared expert (a slot of the
    decode kernels, k at their limit, another width) against the routed part
    and the shared part on their own."""
    print(f"[case] block with shared expert T={T} k={k} S={S}", flush=True)
    g = torch.Generator(device=dev).manual_seed(T + k + S)
    E, H, I = 32, 2048, 512
    gu, dn = _quant(g, (E, 2 * I), H, dev), _quant(g, (E, H), I, dev)
    sgu, sdn = _quant(g, (1, 2 * S), H, dev), _quant(g, (1, H), S, dev)
    gate = (torch.randn(1, H, device=dev, generator=g) * H ** -0.5).to(torch.bfloat16)
    router = (torch.randn(E, H, device=dev, generator=g) * H ** -0.5).to(torch.bfloat16)
    x = torch.randn(T, H, device=dev, generator=g).to(torch.bfloat16)
    block = SparseMoeBlock(router, gu, dn, k, shared=SharedExpert(sgu, sdn, gate))
    y = block(x)
    idx, sc = block.route(x)
    routed = block.experts(x, idx, sc).double()
    gate_up = x.double() @ _deq64(sgu)[0].t()
    a, u = gate_up.chunk(2, dim=-1)
    shared = (torch.nn.functional.silu(a) * u) @ _deq64(sdn)[0].t()
    shared = torch.sigmoid(x.double() @ gate.double().t()) * shared
    ref = routed + shared
    # the routed part's bf16 rounding, h's, and the sum's: 3 * 2^-9 of the
    # parts' magnitudes, the block's own bar of 2^-7 of max|y|
    assert bool(((y.double() - ref).abs() <= 2.0 ** -7 * ref.abs().max()).all())


@pytest.mark.parametrize("sort_min_pairs", [0, 64])
@pytest.mark.parametrize("S", [None, 512, 768])
def test_block_of_no_tokens(dev, S, sort_min_pairs):
    print(f"[case] block of no tokens S={S} sort_min_pairs={sort_min_pairs}", flush=True)
    g = torch.Generator(device=dev).manual_seed(3)
    H, I, E = 2048, 512, 16
    shared = None
    if S:
        gate = torch.randn(1, H, device=dev, generator=g).to(torch.bfloat16)
        shared = SharedExpert(_quant(g, (1, 2 * S), H, dev), _quant(g, (1, H), S, dev), gate)
    rw = torch.randn(E, H, device=dev, generator=g).to(torch.bfloat16)
    blk = SparseMoeBlock(rw, _quant(g, (E, 2 * I), H, dev), _quant(g, (E, H), I, dev), 4, shared=shared,
                         sort_min_pairs=sort_min_pairs)
    x = torch.empty(0, H, dtype=torch.bfloat16, device=dev)
    assert blk(x).shape == (0, H)
    assert blk.experts(x, *blk.route(x)).shape == (0, H)


@pytest.mark.parametrize("T,k,E", [(1, 1, 1), (7, 10, 256), (64, 64, 100), (409, 10, 512), (410, 10, 256),
                                   (129, 3, 2048), (5, 4, 513), (3000, 10, 64)])
def test_route_block_matches_route(dev, T, k, E):
    """The block's routing on every path and edge of qmoe_route (one block,
    count and scatter, an expert count of its limit), with and without the
    shared expert's rows, against the plain tables."""
    print(f"[case] route_block T={T} k={k} E={E}", flush=True)
    g = torch.Generator(device=dev).manual_seed(T + k + E)
    idx = torch.randint(-1, E + 1, (T, k), dtype=torch.int32, device=dev, generator=g)  # a few out of range
    r = ops.route(idx, E)
    n, nt = T * k, int(r.tiles.ntiles)
    for shared in (False, True):
        x_rows, inv, t = ops.route_block(idx, E, shared)
        assert torch.equal(x_rows[:n], r.order // k) and torch.equal(inv[:n], r.inv_order)
        assert torch.equal(t.offsets[:E + 1], r.tiles.offsets)
        m = int(t.ntiles)
        assert torch.equal(t.tile_row[:nt], r.tiles.tile_row[:nt]) and torch.equal(t.tile_exp[:nt], r.tiles.tile_exp[:nt])
        if shared:
            rows = torch.arange(0, T, 128, dtype=torch.int32, device=dev)
            assert m == nt + rows.numel() and int(t.offsets[E + 1]) == n + T and t.rows == n + T
            assert torch.equal(t.tile_row[nt:m], n + rows) and bool((t.tile_exp[nt:m] == E).all())
            assert torch.equal(x_rows[n:n + T], torch.arange(T, dtype=torch.int32, device=dev))
        else:
            assert m == nt and t.rows == n


# (tile kernel; then, at six rows per expert or fewer, the rows kernel up to 320
# rows and either kernel past them, the shared expert's tiles of one to four
# subtiles and two tiles)
@pytest.mark.parametrize("T,E", [(17, 4), (128, 3), (129, 3), (300, 40), (17, 40), (33, 60), (65, 40), (100, 60),
                                 (129, 100), (140, 200), (200, 300)])
def test_gemm_with_shared_expert_is_the_two_gemms(dev, T, E):
    """Both epilogues over a table whose last expert is a tensor of its own:
    bit for bit the routed GEMM and the shared expert's own."""
    print(f"[case] GEMM with shared rows T={T} E={E}", flush=True)
    g = torch.Generator(device=dev).manual_seed(T + E)
    k, H, I = 2, 512, 256
    x = torch.randn(T, H, device=dev, generator=g).to(torch.bfloat16)
    idx = torch.randint(0, E, (T, k), dtype=torch.int32, device=dev, generator=g)
    x_rows, _, ts = ops.route_block(idx, E, shared=True)
    _, _, t0 = ops.route_block(idx, E)
    one = ops.build_tiles(torch.zeros(T, dtype=torch.int32, device=dev), 1)
    for pairs in (True, False):
        w, sw = _quant(g, (E, 2 * I), H, dev), _quant(g, (1, 2 * I), H, dev)
        tw, stw = ops.repack_tiles(*w, swiglu_pairs=pairs), ops.repack_tiles(*sw, swiglu_pairs=pairs)
        gemm = ops.gather_qmm_swiglu_sorted_tiles if pairs else ops.gather_qmm_sorted_tiles
        y = ops.gather_qmm_sorted_tiles_shared(x, tw, stw, ts, x_rows=x_rows)
        assert torch.equal(y[:T * k], gemm(x, tw, t0, x_rows=x_rows))
        assert torch.equal(y[T * k:], gemm(x, stw, one))


@pytest.mark.parametrize("mode", ["fast", "ops", "clone"])
@pytest.mark.parametrize("T,k,D", [(1, 1, 8), (3, 8, 2056), (70, 10, 2048), (5, 17, 512)])
def test_weighted_sum_with_shared_row(dev, mode, T, k, D):
    print(f"[case] weighted sum with shared row T={T} k={k} D={D} {mode}", flush=True)
    g = torch.Generator(device=dev).manual_seed(T + k)
    xs = torch.randn(T * k, D, device=dev, generator=g).to(torch.bfloat16)
    sh = torch.randn(T, D, device=dev, generator=g).to(torch.bfloat16)
    sc = torch.rand(T, k + 1, device=dev, generator=g)
    inv = torch.randperm(T * k, device=dev, generator=g).to(torch.int32)
    y = ops.moe_weighted_sum_shared(xs, inv, sc, sh, mode)
    if mode == "fast":
        ref = (xs.double()[inv.long()].reshape(T, k, D) * sc[:, :k, None].double()).sum(1)
        mag = (xs.double().abs()[inv.long()].reshape(T, k, D) * sc[:, :k, None].double()).sum(1)
    else:  # the k-slot sum as that mode rounds it
        ref = ops.moe_weighted_sum(xs, inv, sc[:, :k].contiguous(), (T, D), mode).double()
        mag = ref.abs()
    last = sc[:, k:].double() * sh.double()
    err = (y.double() - (ref + last)).abs()
    # one bf16 rounding, and k + 2 roundings of the sums in fp32
    assert bool((err <= 2.0 ** -8 * (ref + last).abs() + (k + 2) * 2.0 ** -24 * (mag + last.abs())).all())


@pytest.mark.parametrize("T,E,K", [(1, 8, 8), (5, 100, 2048), (300, 256, 2056), (9, 1000, 520)])
def test_topk_with_shared_score(dev, T, E, K):
    print(f"[case] top-k with shared score T={T} E={E} K={K}", flush=True)
    g = torch.Generator(device=dev).manual_seed(T + E)
    lg = torch.randn(T, E, device=dev, generator=g)
    x = torch.randn(T, K, device=dev, generator=g).to(torch.bfloat16)
    gate = (torch.randn(1, K, device=dev, generator=g) * K ** -0.5).to(torch.bfloat16)
    k = min(E, 10)
    for norm in (True, False):
        idx, sc = ops.router_topk_shared(lg, k, x, gate, norm)
        idx0, sc0 = ops.router_topk(lg, k, norm)
        assert torch.equal(idx, idx0) and torch.equal(sc[:, :k], sc0)
        z = x.double() @ gate.double().t()
        bound = 0.25 * K * 2.0 ** -24 * (x.double().abs() @ gate.double().abs().t()) + 4 * 2.0 ** -24
        assert bool(((sc[:, k:].double() - torch.sigmoid(z)).abs() <= bound).all())


@pytest.mark.parametrize("T,K,D", [(1, 8, 8), (5, 2048, 2048), (300, 520, 4104)])
def test_shared_combine(dev, T, K, D):
    print(f"[case] shared combine T={T} K={K} D={D}", flush=True)
    g = torch.Generator(device=dev).manual_seed(T + K)
    x, y, ys = (torch.randn(T, n, device=dev, generator=g).to(torch.bfloat16) for n in (K, D, D))
    gate = (torch.randn(1, K, device=dev, generator=g) * K ** -0.5).to(torch.bfloat16)
    out = ops.shared_combine(y, ys, x, gate).double()
    s = torch.sigmoid(x.double() @ gate.double().t())
    ref = y.double() + s * ys.double()
    # one bf16 rounding; the score's fp32 sum is within K * 2^-24 of sum |x w|, its sigmoid's slope at most 1/4
    off = 0.25 * K * 2.0 ** -24 * (x.double().abs() @ gate.double().abs().t()) + 4 * 2.0 ** -24
    assert bool(((out - ref).abs() <= 2.0 ** -8 * ref.abs() + off * ys.double().abs() + 2.0 ** -23 * y.double().abs()).all())


@pytest.mark.parametrize("n", [1, 5, 1023, 1024, 1025, 2047, 20480, 70001])
@pytest.mark.parametrize("E", [1, 7, 256, 1500])
def test_tiles_of_sorted_ids(dev, n, E):
    """Offsets and tiles over sorted ids at the edges of the sampled search."""
    print(f"[case] tiles of sorted ids n={n} E={E}", flush=True)
    g = torch.Generator(device=dev).manual_seed(n + E)
    for ids in (torch.randint(0, E, (n,), device=dev, generator=g), torch.full((n,), E - 1, device=dev),
                torch.zeros(n, dtype=torch.int64, device=dev)):
        ids = ids.sort()[0].to(torch.int32)
        t = ops.build_tiles(ids, E)
        edges = torch.searchsorted(ids.long(), torch.arange(E + 1, device=dev))
        assert torch.equal(t.offsets.long(), edges)
        per = (edges[1:] - edges[:-1] + 127) // 128
        assert int(t.ntiles) == int(per.sum())
        exp = torch.repeat_interleave(torch.arange(E, device=dev), per)
        assert torch.equal(t.tile_exp[:exp.numel()].long(), exp)


def _block_weights(g, dev, E, H, I):
    return ((torch.randn(E, H, device=dev, generator=g) * H ** -0.5).to(torch.bfloat16), _quant(g, (E, 2 * I), H, dev),
            _quant(g, (E, H), I, dev))


def _shared64(x, sgu, sdn, z):
    """sigmoid(z) * SwiGLU-MLP(x) in 64 bits, over the exact affine weights up to
    16 tokens and bf16-materialised ones above, as the block takes them."""
    wgu, wdn = (_deq64(q)[0] if x.shape[0] <= 16 else _deq64(q)[0].to(torch.bfloat16).double() for q in (sgu, sdn))
    a, u = (x.double() @ wgu.t()).chunk(2, dim=-1)
    return torch.sigmoid(z) * ((torch.nn.functional.silu(a) * u) @ wdn.t())


@pytest.mark.parametrize("T", [1, 16, 17, 100])
@pytest.mark.parametrize("S,resident", [(512, "tiles"), (512, "both"), (256, "tiles")])
def test_shared_expert_with_a_quantized_gate(dev, T, S, resident):
    """A gate of codes, which router_logits takes, over every dispatch."""
    print(f"[case] quantized gate T={T} S={S} {resident}", flush=True)
    g = torch.Generator(device=dev).manual_seed(T + S)
    E, H, I, k = 32, 2048, 512, 4
    router, gu, dn = _block_weights(g, dev, E, H, I)
    sgu, sdn = _quant(g, (1, 2 * S), H, dev), _quant(g, (1, H), S, dev)
    gate = _quant(g, (1,), H, dev)
    x = torch.randn(T, H, device=dev, generator=g).to(torch.bfloat16)
    block = SparseMoeBlock(router, gu, dn, k, resident=resident, shared=SharedExpert(sgu, sdn, gate))
    y = block(x)
    idx, sc = block.route(x)
    routed, shared = block.experts(x, idx, sc).double(), _shared64(x, sgu, sdn, x.double() @ _deq64(gate).t())
    # bf16 roundings, 2^-9 of a value each: of h (the down product of errors of
    # independent signs grows no faster than that of h itself), of the shared
    # expert's rows before and after the gate, and of the sum
    err = (y.double() - routed - shared).norm()
    bound = 2.0 ** -9 * (3 * shared.norm() + (routed + shared).norm())
    print(f"[parity] err/bound {float(err / bound):.3g}", flush=True)
    assert float(err) <= float(bound)


@pytest.mark.parametrize("T", [2, 40])
@pytest.mark.parametrize("resident,shared", [("tiles", True), ("both", True), ("both", False)])
@pytest.mark.parametrize("how", ["subclass", "instance", "class"])
def test_replaced_steps_are_called(dev, T, resident, shared, how, monkeypatch):
    """route, experts and shared_expert of a subclass, an instance or the patched
    class run where the block's own would, and make the result."""
    print(f"[case] replaced steps T={T} {resident} shared={shared} {how}", flush=True)
    g = torch.Generator(device=dev).manual_seed(T)
    E, H, I, k = 32, 2048, 512, 4
    router, gu, dn = _block_weights(g, dev, E, H, I)
    sh = SharedExpert(_quant(g, (1, 2 * I), H, dev), _quant(g, (1, H), I, dev),
                      (torch.randn(1, H, device=dev, generator=g) * H ** -0.5).to(torch.bfloat16)) if shared else None
    x = torch.randn(T, H, device=dev, generator=g).to(torch.bfloat16)
    plain = SparseMoeBlock(router, gu, dn, k, resident=resident, shared=sh)
    calls = []

    def route(self, x2):
        calls.append("route")
        idx, scores = SparseMoeBlock_route(self, x2)
        return idx.flip(-1).contiguous(), 0.5 * scores

    def experts(self, x2, idx, scores):
        calls.append("experts")
        return 2 * SparseMoeBlock_experts(self, x2, idx, scores)

    def shared_expert(self, x2):
        calls.append("shared_expert")
        return 3 * SparseMoeBlock_shared(self, x2)

    SparseMoeBlock_route, SparseMoeBlock_experts = SparseMoeBlock.route, SparseMoeBlock.experts
    SparseMoeBlock_shared = SparseMoeBlock.shared_expert
    steps = {"route": route, "experts": experts, "shared_expert": shared_expert}
    block = plain
    if how == "subclass":
        block = type("Mine", (SparseMoeBlock,), steps)(router, gu, dn, k, resident=resident, shared=sh)
    elif how == "class":
        for name, step in steps.items():
            monkeypatch.setattr(SparseMoeBlock, name, step)
    else:
        for name, step in steps.items():
            monkeypatch.setattr(block, name, lambda *a, step=step: step(block, *a))
    y = block(x)
    # the tile-layout decode call has its two launches in the place of route and experts
    routed = not (resident == "tiles" and T == 2)
    assert calls == ["route", "experts"] * routed + ["shared_expert"] * shared
    if routed:
        idx, scores = SparseMoeBlock_route(block, x)
        ref = 2 * SparseMoeBlock_experts(block, x, idx.flip(-1).contiguous(), 0.5 * scores)
    else:
        ref = SparseMoeBlock_experts(block, x, *SparseMoeBlock_route(block, x))
    if shared:
        ref = (ref.float() + (3 * SparseMoeBlock_shared(block, x)).float()).to(torch.bfloat16)
    assert torch.equal(y, ref)


@pytest.mark.parametrize("v", ["inf", "-inf", "nan"])
def test_shared_slot_decode_with_infinities(dev, v):
    """A token with an infinity or a NaN takes its own result with it and no
    other's; its shared score is the sigmoid's limit, or NaN."""
    print(f"[case] shared slot with {v}", flush=True)
    g = torch.Generator(device=dev).manual_seed(9)
    E, H, I, k, T = 24, 2048, 512, 4, 5
    router, gu, dn = _block_weights(g, dev, E, H, I)
    sgu, sdn = _quant(g, (1, 2 * I), H, dev), _quant(g, (1, H), I, dev)
    gate = (torch.randn(1, H, device=dev, generator=g) * H ** -0.5).to(torch.bfloat16)
    x = torch.randn(T, H, device=dev, generator=g).to(torch.bfloat16)
    logits = torch.randn(T, E, device=dev, generator=g)
    tw, stw = ops.repack_tiles(*gu, swiglu_pairs=True), ops.repack_tiles(*sgu, swiglu_pairs=True)
    td, std = ops.repack_tiles(*dn), ops.repack_tiles(*sdn)

    def run(x):
        h, idx, sc = ops.gate_up_silu_tiles_topk_shared(x, tw, logits, k, stw, gate)
        return h, idx, sc, ops.down_wsum_tiles_shared(h, td, idx, sc, std)

    h0, idx0, sc0, y0 = run(x)
    xb = x.clone()
    xb[2, 7] = float(v)
    h, idx, sc, y = run(xb)
    assert torch.equal(idx, idx0) and torch.equal(sc[:, :k], sc0[:, :k])
    rest = torch.tensor([0, 1, 3, 4], device=dev)
    assert torch.equal(h[rest], h0[rest]) and torch.equal(sc[rest], sc0[rest]) and torch.equal(y[rest], y0[rest])
    z = float(v) * float(gate[0, 7])  # the rest of the logit is finite
    lim = torch.sigmoid(torch.tensor(z))
    assert bool(torch.isnan(sc[2, k])) if v == "nan" else float(sc[2, k]) == float(lim)
    # the kernel that takes ids, slot for slot
    hi = ops.gate_up_silu_tiles(xb, tw, idx[:, :k].contiguous())
    assert torch.equal(h[:, :k].contiguous().view(torch.int16), hi.view(torch.int16))
    assert not bool(torch.isfinite(y[2]).any())


@pytest.mark.parametrize("E", [100, 600])
def test_selection_of_infinite_and_nan_logits(dev, E):
    """The kernels that select by themselves choose as router_topk does where
    logits are NaN, infinite, the lowest value or all equal."""
    print(f"[case] selection of infinite logits E={E}", flush=True)
    g = torch.Generator(device=dev).manual_seed(E)
    H, I, k, T = 2048, 512, 6, 8
    gu, sgu = _quant(g, (E, 2 * I), H, dev), _quant(g, (1, 2 * I), H, dev)
    gate = torch.randn(1, H, device=dev, generator=g).to(torch.bfloat16)
    x = torch.randn(T, H, device=dev, generator=g).to(torch.bfloat16)
    lg = torch.randn(T, E, device=dev, generator=g)
    lg[0, ::2] = float("nan")
    lg[1, 1:] = float("nan")
    lg[2, 5:] = float("-inf")
    lg[3] = float("-inf")
    lg[4, [1, 7]] = float("inf")
    lg[5] = torch.finfo(torch.float32).min
    lg[6] = 0.0
    lg[7] = float("nan")
    for norm in (True, False):
        idx, sc = ops.router_topk(lg, k, norm)
        bits = sc.view(torch.int32)
        _, i1, s1 = ops.gate_up_silu_topk(x, *gu, lg, k, norm)
        assert torch.equal(i1, idx) and torch.equal(s1.view(torch.int32), bits)
        tw, stw = ops.repack_tiles(*gu, swiglu_pairs=True), ops.repack_tiles(*sgu, swiglu_pairs=True)
        _, i2, s2 = ops.gate_up_silu_tiles_topk_shared(x, tw, lg, k, stw, gate, norm)
        assert torch.equal(i2[:, :k], idx) and torch.equal(s2[:, :k].contiguous().view(torch.int32), bits)
        i3, s3 = ops.router_topk_shared(lg, k, x, gate, norm)
        assert torch.equal(i3, idx) and torch.equal(s3[:, :k].contiguous().view(torch.int32), bits)
