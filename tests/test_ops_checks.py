"""Wrong shapes that a wrapper turns into an error before any launch: the kernels
index what they are given by the sizes of the call.  CPU tensors, with the device
check taken out and a launch counted as a failure."""

import pytest
import torch

from titan_amd import _lib, ops


@pytest.fixture(autouse=True)
def no_launch(monkeypatch):
    def call(name, *args):
        raise AssertionError(f"{name} launched")

    monkeypatch.setattr(ops, "_dev", lambda t, name: None)
    monkeypatch.setattr(ops, "_stream", lambda t: 0)
    monkeypatch.setattr(ops, "tile_rows", lambda: 128)
    monkeypatch.setattr(_lib, "call", call)


def _tiles(E, N, K, pairs=False):
    return ops.TileWeights(torch.zeros(E, N // 64, K // 64, 2, 2, 32, 4, dtype=torch.int32),
                           torch.zeros(E, N // 64, K // 64, 64, dtype=torch.int32), E, N, K, swiglu_pairs=pairs)


# the ids or the scores of the k routed slots alone, one token's, none
@pytest.mark.parametrize("ids,scores", [((4, 3), (4, 4)), ((4, 4), (4, 3)), ((4,), (4, 4)), ((4, 4), (0, 4))])
def test_down_wsum_shared_needs_every_slot(ids, scores):
    T, slots, I, D = 4, 4, 512, 64
    h = torch.zeros(T, slots, I, dtype=torch.bfloat16)
    with pytest.raises(ValueError, match="slots"):
        ops.down_wsum_tiles_shared(h, _tiles(5, D, I), torch.zeros(ids, dtype=torch.int32), torch.zeros(scores),
                                   _tiles(1, D, I))
    with pytest.raises(AssertionError, match="launched"):  # the right ones reach the kernel
        ops.down_wsum_tiles_shared(h, _tiles(5, D, I), torch.zeros(T, slots, dtype=torch.int32),
                                   torch.zeros(T, slots), _tiles(1, D, I))


# the rows of the routed pairs alone, as a routing without shared rows gives them
@pytest.mark.parametrize("gathered", [False, True])
@pytest.mark.parametrize("pairs", [False, True])
def test_gemm_with_shared_expert_needs_every_row(gathered, pairs):
    T, k, E, K, N = 6, 3, 5, 128, 256
    i32 = torch.zeros(E + 2, dtype=torch.int32)
    table = ops.TileTable(i32, i32, i32, i32[:1], E + 2, 128, E + 1, T * k + T)

    def gemm(rows):
        x = torch.zeros(T if gathered else rows, K, dtype=torch.bfloat16)
        ops.gather_qmm_sorted_tiles_shared(x, _tiles(E, N, K, pairs), _tiles(1, N, K, pairs), table,
                                           x_rows=torch.zeros(rows, dtype=torch.int32) if gathered else None)

    for rows in (0, T * k, T * k + T - 1):
        with pytest.raises(ValueError, match="rows"):
            gemm(rows)
    with pytest.raises(AssertionError, match="launched"):
        gemm(T * k + T)


@pytest.mark.parametrize("width", [1, 17, 1025])
def test_swiglu_needs_both_halves(width):
    with pytest.raises(ValueError, match="2I"):
        ops.swiglu(torch.zeros(3, width, dtype=torch.bfloat16))
    with pytest.raises(AssertionError, match="launched"):
        ops.swiglu(torch.zeros(3, width + 15 + (width + 15) % 2, dtype=torch.bfloat16))
