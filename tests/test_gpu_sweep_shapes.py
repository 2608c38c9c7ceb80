"""Executions of plans whose shape nobody set, of one to 16385 blocks and with few rows per tile, against
the C oracle (integer sums, so bit for bit). test_sweep_shape_rule.py asserts the shapes themselves."""

import numpy as np
import pytest

from oracle import c_oracle
from oracle import spp_oracle as O

pytestmark = pytest.mark.gpu

# (bits, channels, rows, 16-row blocks): a block covers 2048 (1/2-bit) or 1024 (4/8-bit) samples
CASES = [
    (1, 40, 16, 128), (1, 40, 16, 129),
    (2, 36, 5, 1), (2, 100, 17, 64), (2, 36, 9, 129),
    (4, 34, 16, 128), (4, 34, 16, 129), (4, 18, 7, 1024), (4, 18, 7, 1025),
    (8, 33, 12, 1), (8, 33, 9, 128), (8, 33, 9, 129), (8, 300, 8, 3),
    (8, 3, 2, 16384), (8, 3, 2, 16385),
]


def _check(rng, table, nsamps, nbits, tiles):
    from sigpyproc3_amd import _lib
    from sigpyproc3_amd.sweep import SweepPlan

    ndm, nchans = table.shape
    order = O.DEFAULT_BITORDER.get(nbits, "big")
    samples = rng.integers(0, 1 << nbits, nsamps * nchans, dtype=np.uint8)
    packed = samples if nbits == 8 else O.pack(samples, nbits, order)
    plan = SweepPlan(table, nsamps, nbits, 1 if order == "big" else 0)
    assert plan.info.ndm_tiles == tiles
    dev = _lib.to_device(packed)
    ref = c_oracle.sweep(samples, nchans, table, ld=plan.max_len)
    plane = plan.execute(dev).cpu().numpy()
    for i in range(ndm):
        n = int(plan.row_len[i])
        np.testing.assert_array_equal(plane[i, :n], ref[i, :n], err_msg=f"row {i}")
        assert not plane[i, n:].any()


@pytest.mark.parametrize("nbits,nchans,ndm,blocks", CASES)
def test_default_shape(nbits, nchans, ndm, blocks):
    T = 2048 if nbits <= 2 else 1024
    # delays rise by a sample a row at the band's far end; 16 rows share a DM tile
    table = (np.arange(ndm)[:, None] * np.linspace(0, 1, nchans)[None, :]).astype(np.int32)
    tiles = -(-ndm // 16)
    _check(np.random.default_rng(nbits * 1000 + blocks), table, (blocks // tiles) * T - T // 2, nbits, tiles)


@pytest.mark.parametrize("nbits", [1, 2, 4, 8])
@pytest.mark.parametrize("step,per_tile", [(60, 5), (250, 2), (300, 1), (17, 15), (20, 13)])
@pytest.mark.parametrize("nchans", [40, 136])
def test_tiles_with_few_rows(nbits, step, per_tile, nchans):
    # tiles hold the rows within 252 samples; each row ends `step` samples before the last, so whole
    # blocks of some rows lie past their ends
    ndm, T = 41, 2048 if nbits <= 2 else 1024
    table = np.round(step * np.arange(ndm)[:, None] * np.linspace(0, 1, nchans)[None, :]).astype(np.int32)
    tiles = -(-ndm // per_tile)
    _check(np.random.default_rng(nbits * 1000 + step), table, (128 // tiles + 12) * T + 333, nbits, tiles)
