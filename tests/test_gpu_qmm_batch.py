"""The dense quantized matmul for a batch of rows against 64-bit products."""

import pytest
import torch

from titan_amd import ops

pytestmark = pytest.mark.gpu


# row tiles of 16 up to 64 and more blocks of them, ragged columns, K of less
# than a batch of four units, a ragged last batch, one batch per wave and more
@pytest.mark.parametrize("bits,gs", [(4, 32), (4, 64), (4, 128), (8, 32), (8, 64), (8, 128)])
@pytest.mark.parametrize("M,N,K", [(3, 4096, 2048), (5, 4099, 1024), (16, 1000, 2048), (17, 999, 2048), (33, 600, 2560),
                                   (49, 700, 896), (64, 520, 768), (130, 257, 640), (1400, 100, 128), (8, 2048, 6144)])
def test_quantized_matmul_batch(dev, bits, gs, M, N, K):
    if bits == 8 and K > 4096 and K % 2048:
        pytest.skip("no 8-bit kernel for this K")
    print(f"[case] batched quantized_matmul bits={bits} gs={gs} M={M} N={N} K={K}", flush=True)
    g = torch.Generator(device=dev).manual_seed(M + N + K + bits + gs)
    w = torch.randint(-2 ** 31, 2 ** 31, (N, K * bits // 32), dtype=torch.int32, device=dev, generator=g)
    s = (0.004 + 0.004 * torch.rand(N, K // gs, device=dev, generator=g)).to(torch.bfloat16)
    b = (torch.randn(N, K // gs, device=dev, generator=g) * 0.05).to(torch.bfloat16)
    x = torch.randn(M, K, device=dev, generator=g).to(torch.bfloat16)
    y = ops.quantized_matmul(x, w, s, b, group_size=gs, bits=bits).double()
    shifts = torch.arange(0, 32, bits, device=dev, dtype=torch.int32)
    q = ((w.unsqueeze(-1) >> shifts) & (2 ** bits - 1)).reshape(N, K).double()
    s64, b64 = s.double().repeat_interleave(gs, -1), b.double().repeat_interleave(gs, -1)
    ref = x.double() @ (q * s64 + b64).t()
    # one bf16 rounding, and the fp32 sums: a product enters as x * (q + 128)
    # (4 bits) or x * q, and meets at most K / 4 roundings
    off = 128.0 if bits == 4 else 0.0
    mag = x.double().abs() @ ((q + 2 * off) * s64 + b64.abs()).t()
    err = (y - ref).abs()
    bound = 2.0 ** -8 * ref.abs() + K / 4 * 2.0 ** -24 * mag
    print(f"[parity] max err/bound {float((err / bound).max()):.3g}", flush=True)
    assert bool((err <= bound).all())
