"""Address model of the four-wave blocks of the tile-layout gate_up decode
kernel (qmv64_paired_lines_kernel with W > 1): every access in bounds, every
byte of x staged once, every output stored once."""

import numpy as np
import pytest


def _blocks(E, T, k, n_out, NV, RG, W):
    """Per thread of the grid: block item, pair, first index, and lane split."""
    nblk = n_out // (RG * W)
    blocks = T * k * nblk
    b = np.repeat(np.arange(blocks, dtype=np.int64), 64 * W)
    t = np.tile(np.arange(64 * W, dtype=np.int64), blocks)
    item = b if blocks % 8 else (b % 8) * (blocks // 8) + b // 8
    pr = item // nblk
    lane, wave = t % 64, t // 64
    i0 = ((item - pr * nblk) * W + wave) * RG
    return blocks, b, t, pr, i0, lane & 7, lane >> 3


# one column block per pair, several, blocks a multiple of the XCDs and not,
# K = 2048 and 4096; eight indices in one- and four-wave blocks
@pytest.mark.parametrize("RG,W", [(8, 1), (8, 4)])
@pytest.mark.parametrize("E,T,k,n_out,NV", [(256, 4, 10, 512, 1), (64, 3, 7, 96, 1), (256, 3, 11, 512, 2), (4, 2, 1, 32, 1)])
def test_block_form_accesses(E, T, k, n_out, NV, RG, W):
    blocks, b, t, pr, i0, r, sl = _blocks(E, T, k, n_out, NV, RG, W)
    K, G, NC, NCH, NP = 2048 * NV, 32 * NV, 2 * n_out // 64, 64 * NV, 4 * NV
    e = (E - 1 - 7 * pr) % E
    c, l0 = i0 >> 5, i0 & 31
    cbase = (e * NC + c) * G
    assert np.all(l0 + RG <= 32)
    for pp in range(NP):
        for jj in range(2):
            word = (cbase + 8 * pp + sl) * 64 + l0 + r + 32 * jj
            assert word.min() >= 0 and word.max() < E * NC * G * 64
            for h in range(2):
                unit = (((cbase + 8 * pp + sl) * 2 + jj) * 2 + h) * 32 + l0 + r
                assert unit.min() >= 0 and (unit.max() + 1) * 16 <= E * 2 * n_out * K // 2
                # eight neighbouring lanes read consecutive units: one 128-byte line
                lines = unit.reshape(-1, 8)
                assert np.all(np.diff(lines, axis=1) == 1) and np.all(lines[:, 0] % 8 == 0)
    if W > 1:  # the block's threads stage its x row one 16-byte piece at a time
        pieces = np.concatenate([v * 64 * W + t[b == 0] for v in range(4 * NCH // (64 * W))])
        assert np.array_equal(np.sort(pieces), np.arange(4 * NCH))
        assert (np.max(pieces) + 1) * 16 == K * 2
    m = sl == 0
    out = pr[m] * n_out + i0[m] + r[m]
    assert np.array_equal(np.sort(out), np.arange(T * k * n_out))
