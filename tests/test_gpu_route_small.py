"""The routing step around the pair count where its single block changes width."""

import numpy as np
import pytest
import torch

from titan_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64, 65, 511, 512, 513, 1023, 1024, 1025])
@pytest.mark.parametrize("E", [1, 256, 512])
def test_route_widths(dev, n, E):
    print(f"[case] route n={n} E={E}", flush=True)
    rng = np.random.default_rng(n + E)
    ids = rng.integers(0, E, size=n).astype(np.int32)
    r = ops.route(torch.from_numpy(ids).to(dev), E)
    order = np.argsort(ids, kind="stable")
    assert np.array_equal(r.order.cpu().numpy(), order)
    assert np.array_equal(r.inv_order.cpu().numpy(), np.argsort(order, kind="stable"))
    assert np.array_equal(r.sorted_ids.cpu().numpy(), ids[order])
    assert np.array_equal(r.tiles.offsets.cpu().numpy(), np.searchsorted(ids[order], np.arange(E + 1)))
    assert int(r.bad_ids) == 0
