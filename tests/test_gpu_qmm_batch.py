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


def _weights(g, dev, N, K, bits, gs):
    w = torch.randint(-2 ** 31, 2 ** 31, (N, K * bits // 32), dtype=torch.int32, device=dev, generator=g)
    s = (0.004 + 0.004 * torch.rand(N, K // gs, device=dev, generator=g)).to(torch.bfloat16)
    b = (torch.randn(N, K // gs, device=dev, generator=g) * 0.05).to(torch.bfloat16)
    return w, s, b


@pytest.mark.parametrize("bits,gs", [(4, 32), (4, 64), (4, 128), (8, 32), (8, 64), (8, 128)])
@pytest.mark.parametrize("K", [1024, 640, 2048])
def test_quantized_matmul_batch_of_large_values(dev, bits, gs, K):
    """Values whose products with the codes are finite but, for 4 bits, 128 times
    them are not (x up to 2^122, 5.3e36), in alternating signs, so that the sums
    are finite too."""
    print(f"[case] batched quantized_matmul of large values bits={bits} gs={gs} K={K}", flush=True)
    g = torch.Generator(device=dev).manual_seed(K + bits + gs)
    M, N = 16, 4096
    w, s, b = _weights(g, dev, N, K, bits, gs)
    s, b = s * 2.0 ** -8, b * 2.0 ** -8
    top = 122 if bits == 4 else 115
    x = (torch.randn(M, K, device=dev, generator=g).clamp(-1, 1) * 2.0 ** top).to(torch.bfloat16)
    x[:, ::2] = x[:, ::2].abs()
    x[:, 1::2] = -x[:, ::2]  # every partial sum stays small
    y = ops.quantized_matmul(x, w, s, b, group_size=gs, bits=bits).double()
    shifts = torch.arange(0, 32, bits, device=dev, dtype=torch.int32)
    q = ((w.unsqueeze(-1) >> shifts) & (2 ** bits - 1)).reshape(N, K).double()
    s64, b64 = s.double().repeat_interleave(gs, -1), b.double().repeat_interleave(gs, -1)
    ref = x.double() @ (q * s64 + b64).t()
    off = 128.0 if bits == 4 else 0.0
    mag = x.double().abs() @ ((q + 2 * off) * s64 + b64.abs()).t()
    assert bool(((y - ref).abs() <= 2.0 ** -8 * ref.abs() + K / 4 * 2.0 ** -24 * mag).all())


@pytest.mark.parametrize("bits,gs", [(4, 32), (4, 64), (4, 128), (8, 32), (8, 64), (8, 128)])
@pytest.mark.parametrize("K", [1024, 640])
def test_quantized_matmul_batch_of_infinities(dev, bits, gs, K):
    """A row with an infinity or a NaN, in its first or last columns (the last
    batch of 640 is ragged), has no finite result; no other row changes."""
    print(f"[case] batched quantized_matmul of infinities bits={bits} gs={gs} K={K}", flush=True)
    g = torch.Generator(device=dev).manual_seed(K + bits + gs)
    M, N = 20, 4099
    w, s, b = _weights(g, dev, N, K, bits, gs)
    x = torch.randn(M, K, device=dev, generator=g).to(torch.bfloat16)
    y0 = ops.quantized_matmul(x, w, s, b, group_size=gs, bits=bits)
    bad = {0: (3, "inf"), 2: (K - 1, "-inf"), 7: (K // 2, "nan"), 17: (K - 1, "nan"), 19: (0, "inf")}
    for row, (col, v) in bad.items():
        x[row, col] = float(v)
    y = ops.quantized_matmul(x, w, s, b, group_size=gs, bits=bits)
    rows = torch.tensor(sorted(bad), device=dev)
    rest = torch.tensor([r for r in range(M) if r not in bad], device=dev)
    assert torch.equal(y[rest], y0[rest])
    assert not bool(torch.isfinite(y[rows]).any())
    assert bool(torch.isnan(y[[7, 17]]).all())
