"""The DM-time transform: which calls its tiles take (host rule), and, on the GPU, the forms at the
edges of that rule: valid columns only in tiles, rows whose offsets no window holds, and calls of few
rows or short blocks. Channels are added in order in float32, so equality is exact."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from sigpyproc3_amd import _lib


def _in_tiles(ncols, ndm, out_cols):
    fn = _lib.load()._ZN3spp12dmt_in_tilesElll  # spp::dmt_in_tiles(ncols, ndm, out_cols)
    fn.restype = ctypes.c_bool
    fn.argtypes = [ctypes.c_int64] * 3
    return fn(ncols, ndm, out_cols)


CASES = [
    # channels, columns, rows, offset step a row at the band's end, output columns, in tiles
    (7, 1535, 1100, 1.1, 1535, False),    # no window fits: a thread per output
    (7, 1024, 2100, 0.3, 1024, False),
    (7, 1536, 1100, 1.1, 1536, True),
    (11, 6000, 416, 2.0, 5000, True),     # valid columns only
    (11, 6000, 416, 90.0, 4097, True),    # of these most windows do not fit
    (13, 5000, 416, 611.0, 5000, True),   # offsets far apart in every tile
    (9, 70000, 32, 9001.0, 70000, True),
    (9, 300000, 4, 70001.0, 300000, True),
    (9, 300000, 3, 70001.0, 300000, False),  # few rows: a thread per output
    (9, 300000, 1, 1.0, 300000, False),
    (483, 5000, 416, 55.0, 5000, True),   # more channels than are planned at a time, some out of a window
]


@pytest.mark.parametrize(("nchans", "ncols", "ndm", "step", "out_cols", "tiles"), CASES)
def test_rule(nchans, ncols, ndm, step, out_cols, tiles):
    assert _in_tiles(ncols, ndm, out_cols) == tiles


@pytest.mark.gpu
@pytest.mark.parametrize(("nchans", "ncols", "ndm", "step", "out_cols", "tiles"), CASES)
def test_transform(nchans, ncols, ndm, step, out_cols, tiles):
    rng = np.random.default_rng(nchans + ncols)
    x = rng.normal(10.0, 3.0, (nchans, ncols)).astype(np.float32)
    delays = np.round(step * np.arange(ndm)[:, None] * np.linspace(0, 1, nchans)[None, ::-1]).astype(np.int64)
    off = np.ascontiguousarray(np.mod(-delays, ncols) if out_cols == ncols else delays % (ncols - out_cols + 1))
    dev = [_lib.to_device(x), _lib.to_device(off)]
    out = _lib.empty((ndm, out_cols), "float32")
    assert _in_tiles(ncols, ndm, out_cols) == tiles
    _lib.call("spp_dmt", _lib.ptr(dev[0]), nchans, ncols, _lib.ptr(off), _lib.ptr(dev[1]), ndm, out_cols,
              _lib.ptr(out), _lib.stream_handle())
    got = out.cpu().numpy()
    t = np.arange(out_cols)
    for a in range(0, ndm, 64):
        want = np.zeros((min(64, ndm - a), out_cols), np.float32)
        for c in range(nchans):
            want += x[c][(t[None, :] + off[a : a + 64, c : c + 1]) % ncols]
        np.testing.assert_array_equal(got[a : a + 64], want, err_msg=f"rows from {a}")
