"""spp_normalise_boxcar_mf in blocks of 16, 8, 4 and 2 segments of 2048 outputs (few rows take short
blocks), with a pulse across a block edge in every row, against the two-pass form."""

from __future__ import annotations

import numpy as np
import pytest

SEG = 2048
WIDTHS = [1, 2, 4, 8, 16, 32, 64]


def _segments(nrows, n):
    """Segments per block, restated: halved while fewer than 512 blocks result."""
    segs = 16
    while segs > 2 and nrows * -(-n // (segs * SEG)) < 512:
        segs //= 2
    return segs


@pytest.mark.gpu
@pytest.mark.parametrize("integer", [True, False])
@pytest.mark.parametrize(("nrows", "n", "segs"), [(520, 33001, 16), (172, 70003, 16), (260, 32768, 8), (129, 32770, 4),
                                                  (40, 34816, 2)])
def test_block_lengths(nrows, n, segs, integer):
    from sigpyproc3_amd.sweep import boxcar_mf, normalise_boxcar_mf, running_normalise

    assert _segments(nrows, n) == segs
    rng = np.random.default_rng(nrows)
    x = np.zeros((nrows, n + 1), np.float32)
    x[:, :n] = rng.integers(900, 1100, (nrows, n)) if integer else rng.normal(100.0, 7.0, (nrows, n))
    row_len = n - np.arange(nrows, dtype=np.int64) % 7
    edges = np.arange(segs * SEG, n - 64, segs * SEG)
    edges = np.concatenate([[n - 3], edges])  # and one round the row's end
    w = WIDTHS[3:]
    for i in range(nrows):
        start, width = int(edges[i % len(edges)]) - w[i % 4] // 2, w[i % 4]
        x[i, (start + np.arange(width)) % row_len[i]] += 600.0 if integer else 70.0
    one = normalise_boxcar_mf(x, row_len, 4096, WIDTHS)
    two = boxcar_mf(running_normalise(x, row_len, 4096), row_len, WIDTHS)
    np.testing.assert_array_equal(one[2], two[2])
    np.testing.assert_array_equal(one[1], two[1])
    # z may differ by a rounding of float32 where the window sums are not exact (6e-8 of it), and the
    # float64 sums by their order
    np.testing.assert_allclose(one[0], two[0], rtol=1e-6, atol=1e-6)
