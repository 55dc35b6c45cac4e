"""The tile-layout decode gate_up on both sides of its two dispatch lines (four
or eight indices per wave, one- or four-wave blocks), with ids and with the
top-k in the launch: the same bits from both, within the fp32 sums' error of
64-bit products."""

import pytest
import torch

from titan_amd import ops

pytestmark = pytest.mark.gpu


def _quant(g, lead, K, dev):
    w = torch.randint(-2 ** 31, 2 ** 31, (*lead, K // 8), dtype=torch.int32, device=dev, generator=g)
    s = (0.004 + 0.004 * torch.rand(*lead, K // 64, device=dev, generator=g)).to(torch.bfloat16)
    return w, s, (-7.5 * s.float()).to(torch.bfloat16)


# pairs x I / 8 on either side of the SIMDs (1024), pairs x I / 32 of three
# eighths of them (384): I = 512 turns at 16 and 24 pairs
@pytest.mark.parametrize("K", [2048, 4096])
@pytest.mark.parametrize("T,k", [(1, 1), (1, 15), (2, 8), (1, 11), (3, 5), (23, 1), (3, 8), (16, 10)])
def test_gate_up_tiles_over_its_dispatch(dev, K, T, k):
    print(f"[case] tile-layout gate_up T={T} k={k} K={K}", flush=True)
    g = torch.Generator(device=dev).manual_seed(K + 100 * T + k)
    E, I = 40, 512
    w = _quant(g, (E, 2 * I), K, dev)
    tw = ops.repack_tiles(*w, swiglu_pairs=True)
    x = torch.randn(T, K, device=dev, generator=g).to(torch.bfloat16)
    lg = torch.randn(T, E, device=dev, generator=g)
    idx, _ = ops.router_topk(lg, k)
    h = ops.gate_up_silu_tiles(x, tw, idx)
    ht, it, _ = ops.gate_up_silu_tiles_topk(x, tw, lg, k)
    assert torch.equal(it, idx) and torch.equal(ht, h)
    shifts = torch.arange(0, 32, 4, device=dev, dtype=torch.int32)
    for t in range(T):
        for j in range(k):
            e = int(idx[t, j])
            q = ((w[0][e].unsqueeze(-1) >> shifts) & 15).reshape(2 * I, K).double()
            s, b = (p[e].double().repeat_interleave(64, -1) for p in w[1:])
            xd = x[t].double()
            gu = (q * s + b) @ xd
            # a product enters as x * (128 + q), 128 x is taken off again, and
            # it meets at most K / 4 roundings of 2^-24
            mag = (K / 4 * 2.0 ** -24) * (((q + 256) * s + b.abs()) @ xd.abs())
            a, u = gu.chunk(2)
            da, du = mag.chunk(2)
            ref = torch.nn.functional.silu(a) * u
            # silu's slope is at most 1.1; exp and the reciprocal 2^-21
            bound = 2.0 ** -8 * ref.abs() + 1.1 * da * u.abs() + torch.nn.functional.silu(a).abs() * du + 1.1 * da * du \
                + 2.0 ** -21 * ref.abs()
            assert bool(((h[t, j].double() - ref).abs() <= bound).all())
