"""The fused down + weighted sum at every width with a kernel of its own, against
64-bit products."""

import pytest
import torch

from titan_amd import ops

pytestmark = pytest.mark.gpu


# I: 4, 8 or 16 lanes per row with one to three chunks each, and one past them
# (2048); slots up to the pair-parallel kernel's 16 and past it; ragged D
@pytest.mark.parametrize("gs", [32, 64, 128])
@pytest.mark.parametrize("I", [128, 256, 384, 512, 768, 1024, 1536, 2048])
@pytest.mark.parametrize("T,k,D", [(1, 8, 200), (2, 1, 72), (16, 16, 100), (3, 17, 64)])
def test_down_wsum_widths(dev, gs, I, T, k, D):
    print(f"[case] down + weighted sum I={I} gs={gs} T={T} k={k} D={D}", flush=True)
    g = torch.Generator(device=dev).manual_seed(I + gs + T + k)
    E = 20
    w = torch.randint(-2 ** 31, 2 ** 31, (E, D, I // 8), dtype=torch.int32, device=dev, generator=g)
    s = (0.004 + 0.004 * torch.rand(E, D, I // gs, device=dev, generator=g)).to(torch.bfloat16)
    b = (torch.randn(E, D, I // gs, device=dev, generator=g) * 0.05).to(torch.bfloat16)
    h = torch.randn(T, k, I, device=dev, generator=g).to(torch.bfloat16)
    idx = torch.rand(T, E, device=dev, generator=g).topk(k, dim=-1)[1].to(torch.int32)
    sc = torch.rand(T, k, device=dev, generator=g)
    y = ops.down_wsum(h, w, s, b, idx, sc, group_size=gs).double()
    shifts = torch.arange(0, 32, 4, device=dev, dtype=torch.int32)
    q = ((w.unsqueeze(-1) >> shifts) & 15).reshape(E, D, I).double()
    s64, b64 = s.double().repeat_interleave(gs, -1), b.double().repeat_interleave(gs, -1)
    we = (q * s64 + b64)[idx.long()]                        # [T, k, D, I]
    ref = ((we * h.double().unsqueeze(2)).sum(-1) * sc.double().unsqueeze(-1)).sum(1)
    wm = ((q + 256.0) * s64 + b64.abs())[idx.long()]        # a product enters as h * (q + 128), less 128 h
    mag = ((wm * h.double().abs().unsqueeze(2)).sum(-1) * sc.double().unsqueeze(-1)).sum(1)
    # one bf16 rounding, and the fp32 sums: 16 pairs per 32-code chunk, the chunks, the lanes, the slots
    err, bound = (y - ref).abs(), 2.0 ** -8 * ref.abs() + (32 + I // 128 + k) * 2.0 ** -24 * mag
    assert bool((err <= bound).all()), float((err / bound).max())
