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
