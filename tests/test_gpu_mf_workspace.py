"""spp_normalise_boxcar_mf with a workspace sized once for the longest call: fewer and shorter rows,
which by themselves would take shorter blocks and more partials, must run in it."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from sigpyproc3_amd import _lib

WIDTHS = np.array([1, 2, 4, 8, 16, 32, 64], np.int32)


def _size(row_len):
    row_len = np.ascontiguousarray(row_len, np.int64)
    return _lib.workspace_size("spp_normalise_boxcar_mf_workspace_size", len(row_len), _lib.ptr(row_len),
                               _lib.ptr(WIDTHS), len(WIDTHS))


def _run(x, row_len, nbytes):
    row_len = np.ascontiguousarray(row_len, np.int64)
    n = len(row_len)
    snr, peak, widx = _lib.empty((n,), "float32"), _lib.empty((n,), "int32"), _lib.empty((n,), "int32")
    ws = _lib.workspace(nbytes)
    _lib.call("spp_normalise_boxcar_mf", _lib.ptr(x), x.shape[1], n, _lib.ptr(row_len), 4096, _lib.ptr(WIDTHS),
              len(WIDTHS), _lib.ptr(snr), _lib.ptr(peak), _lib.ptr(widx), _lib.ptr(ws), ctypes.c_int64(nbytes),
              _lib.stream_handle())
    return snr.cpu().numpy(), peak.cpu().numpy(), widx.cpu().numpy()


@pytest.mark.gpu
@pytest.mark.parametrize(("nrows", "n"), [(127, 131072), (128, 98304), (64, 131072), (3, 40000), (1, 70000)])
def test_workspace_of_a_longer_call_serves(nrows, n):
    rng = np.random.default_rng(nrows)
    longest = _size(np.full(128, 131072))
    x = rng.integers(900, 1100, (nrows, 131072)).astype(np.float32)
    for i in range(nrows):
        x[i, 100 + 300 * i : 108 + 300 * i] += 400.0
    row_len = np.full(nrows, n)
    own = _run(_lib.to_device(x), row_len, _size(row_len))
    got = _run(_lib.to_device(x), row_len, longest)
    np.testing.assert_array_equal(got[1], own[1])
    np.testing.assert_array_equal(got[2], own[2])
    # integer samples: the same z whatever the blocks, float64 sums in another order, one rounding
    # to float32 each
    np.testing.assert_allclose(got[0], own[0], rtol=2.4e-7)


@pytest.mark.gpu
def test_workspace_below_the_longest_blocks_is_refused():
    row_len = np.full(2, 70000)
    x = _lib.to_device(np.ones((2, 70000), np.float32))
    with pytest.raises(ValueError, match="workspace too small"):
        _run(x, row_len, 1024)
