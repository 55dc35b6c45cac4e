"""The grouped GEMM's kernel for few rows per expert against its tile kernel:
the same rows and weights through a table of many experts (few rows per expert)
and through one of only the used experts give the same bits."""

import pytest
import torch

from titan_amd import ops

pytestmark = pytest.mark.gpu


def _quant(g, lead, K, dev):
    w = torch.randint(-2 ** 31, 2 ** 31, (*lead, K // 8), dtype=torch.int32, device=dev, generator=g)
    s = (0.004 + 0.004 * torch.rand(*lead, K // 64, device=dev, generator=g)).to(torch.bfloat16)
    return w, s, (-7.5 * s.float()).to(torch.bfloat16)


# rows of the used experts: one row, the 32-row subtile's and the 128-row
# tile's edges, several tiles; K of 1, 2, 3, 4 and 8 groups (the unrolled cycle
# is three)
@pytest.mark.parametrize("rows", [(1,), (31, 32, 33), (127, 128, 129), (64, 1, 300)])
@pytest.mark.parametrize("N,K", [(256, 64), (512, 128), (256, 192), (768, 256), (256, 512)])
@pytest.mark.parametrize("gathered", [False, True])
def test_rows_kernel_is_the_tile_kernel(dev, rows, N, K, gathered):
    print(f"[case] few rows {rows} N={N} K={K} gathered={gathered}", flush=True)
    R, n = sum(rows), len(rows)
    E = (R + 5) // 6 + n            # at most six rows per expert
    g = torch.Generator(device=dev).manual_seed(R + N + K)
    used = torch.randperm(E, device=dev, generator=g)[:n].sort()[0]
    few = torch.repeat_interleave(torch.arange(n, device=dev), torch.tensor(rows, device=dev))
    more = 7 * (n + 1)              # rows of one more expert, which put the second table past the limit
    T = R + more
    x = torch.randn(T, K, device=dev, generator=g).to(torch.bfloat16)
    x_rows = torch.randint(0, T, (T,), dtype=torch.int32, device=dev, generator=g) if gathered else None
    w = _quant(g, (E, N), K, dev)
    sub = tuple(t[torch.cat([used, used[:1]])].contiguous() for t in w)
    many_t = ops.build_tiles(used[few].to(torch.int32), E)
    few_t = ops.build_tiles(torch.cat([few, torch.full((more,), n, device=dev)]).to(torch.int32), n + 1)
    for pairs in (False, True):
        gemm = ops.gather_qmm_swiglu_sorted_tiles if pairs else ops.gather_qmm_sorted_tiles
        y = gemm(x, ops.repack_tiles(*w, swiglu_pairs=pairs), many_t, x_rows=None if x_rows is None else x_rows[:R])
        ref = gemm(x, ops.repack_tiles(*sub, swiglu_pairs=pairs), few_t, x_rows=x_rows)
        assert torch.equal(y, ref[:R])


# What decides between the two kernels, and the rows kernel's grid, on either
# side: the rows of a call (320 | more), the rows per tile (16 | more), more
# tiles and more 33-row tiles than the grid has blocks for at once, and a
# table past the limit of rows per expert.  (rows per used expert, experts, N)
@pytest.mark.parametrize("rows,E,N", [
    ((32,) * 10, 100, 512), ((33,) + (32,) * 9, 100, 512),   # 320 and 321 rows
    ((97, 65, 33, 1, 125), 60, 768),                         # 321 rows: every subtile, tile kernel
    ((16,) * 30, 100, 256), ((17,) + (16,) * 29, 100, 256),  # 16 rows per tile and a little more
    ((1,) * 40 + (100, 300, 33), 80, 512),                   # few rows per tile, several large tiles
    ((1,) * 2300, 2400, 256),                                # more tiles than 2048 blocks of one column block
    ((33, 1, 1) * 150, 900, 4096),                           # more large tiles than the 128 of one pass
])
def test_either_kernel_is_the_tile_kernel(dev, rows, E, N):
    print(f"[case] rows {len(rows)} x {max(rows)} of {E} experts, N={N}", flush=True)
    g = torch.Generator(device=dev).manual_seed(sum(rows) + E)
    n, R, K = len(rows), sum(rows), 64
    assert R <= 6 * E
    used = torch.randperm(E, device=dev, generator=g)[:n].sort()[0]
    ids = torch.repeat_interleave(torch.arange(n, device=dev), torch.tensor(rows, device=dev))
    more = 6 * (n + 1) + 1  # rows of one more expert, which put the second table past the limit
    x = torch.randn(R + more, K, device=dev, generator=g).to(torch.bfloat16)
    w = _quant(g, (E, N), K, dev)
    sub = tuple(t[torch.cat([used, used[:1]])].contiguous() for t in w)
    many_t = ops.build_tiles(used[ids].to(torch.int32), E)
    past_t = ops.build_tiles(torch.cat([ids, torch.full((more,), n, device=dev)]).to(torch.int32), n + 1)
    for pairs in (False, True):
        gemm = ops.gather_qmm_swiglu_sorted_tiles if pairs else ops.gather_qmm_sorted_tiles
        y = gemm(x[:R], ops.repack_tiles(*w, swiglu_pairs=pairs), many_t)
        ref = gemm(x, ops.repack_tiles(*sub, swiglu_pairs=pairs), past_t)
        assert torch.equal(y, ref[:R])


# T tokens of two experts each, one of them with an infinity or a NaN
@pytest.mark.parametrize("v", ["inf", "-inf", "nan"])
@pytest.mark.parametrize("T,E", [(40, 100), (170, 200)])
def test_rows_kernel_with_infinities(dev, T, E, v):
    """Such a row of x takes its own results with it and no other's, in the rows
    kernel and in the one that holds both, as in the tile kernel."""
    print(f"[case] rows kernel with {v} T={T} E={E}", flush=True)
    g = torch.Generator(device=dev).manual_seed(T)
    K, N, k = 256, 512, 2
    x = torch.randn(T, K, device=dev, generator=g).to(torch.bfloat16)
    idx = torch.randint(0, E, (T, k), dtype=torch.int32, device=dev, generator=g)
    x_rows, _, few = ops.route_block(idx, E)
    # the same rows in a table past the limit: many more of the last expert after them
    more = 6 * E + 6
    ids = torch.cat([idx.reshape(-1).long().sort()[0], torch.full((more,), E - 1, device=dev)]).to(torch.int32)
    many = ops.build_tiles(ids, E)
    rows2 = torch.cat([x_rows, torch.zeros(more, dtype=torch.int32, device=dev)])
    w = _quant(g, (E, N), K, dev)
    bad = x_rows == T // 2
    for pairs in (False, True):
        tw = ops.repack_tiles(*w, swiglu_pairs=pairs)
        gemm = ops.gather_qmm_swiglu_sorted_tiles if pairs else ops.gather_qmm_sorted_tiles
        y0 = gemm(x, tw, few, x_rows=x_rows)
        xb = x.clone()
        xb[T // 2, 5] = float(v)
        y = gemm(xb, tw, few, x_rows=x_rows)
        ref = gemm(xb, tw, many, x_rows=rows2)[:T * k]
        assert torch.equal(y[~bad], y0[~bad])
        assert torch.equal(y[bad].view(torch.int16), ref[bad].view(torch.int16))
        if not pairs:  # (silu takes a gate of minus infinity to zero or NaN)
            assert not bool(torch.isfinite(y[bad]).any())
