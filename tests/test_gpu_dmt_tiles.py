"""spp_dmt on grids about as large as the tiled kernel takes: windows that wrap, do not fit, or come
from rows of very different offsets (test_dmt_routes.py asserts which calls take tiles). Channels are
added in order in float32, so equality is exact."""

from __future__ import annotations

import numpy as np
import pytest

from sigpyproc3_amd import _lib


def _expected(x, off, out_cols):
    t = np.arange(out_cols)
    acc = np.zeros((off.shape[0], out_cols), np.float32)
    for c in range(x.shape[0]):
        acc += x[c][(t[None, :] + off[:, c : c + 1]) % x.shape[1]]
    return acc


@pytest.mark.gpu
@pytest.mark.parametrize(
    ("nchans", "ncols", "ndm", "step", "out_cols"),
    [
        (1, 1536, 1021, 0.3, 1536),      # one channel, a last tile of 5 rows
        (5, 1535, 1024, 1.1, 1535),      # rows shorter than a window: read from memory
        (7, 4097, 420, 9.7, 4097),       # a partial stage; offsets wrap many times over
        (13, 5000, 416, 73.0, 5000),     # 511 apart in a tile: the widest window
        (13, 5000, 416, 74.0, 5000),     # 518 apart: read from memory
        (483, 2050, 690, 0.9, 2050),     # more channels than are planned at a time
        (11, 6000, 360, 2.0, 5000),      # valid columns only
        (6, 8192, 256, -3.0, 8192),
    ],
)
def test_dmt_tiles(nchans, ncols, ndm, step, out_cols):
    rng = np.random.default_rng(nchans + ncols)
    x = rng.normal(10.0, 3.0, (nchans, ncols)).astype(np.float32)
    delays = np.round(step * np.arange(ndm)[:, None] * np.linspace(0, 1, nchans)[None, ::-1]).astype(np.int64)
    off = np.ascontiguousarray(np.mod(-delays, ncols) if out_cols == ncols else delays % (ncols - out_cols + 1))
    dev = [_lib.to_device(x), _lib.to_device(off)]
    out = _lib.empty((ndm, out_cols), "float32")
    _lib.call("spp_dmt", _lib.ptr(dev[0]), nchans, ncols, _lib.ptr(off), _lib.ptr(dev[1]), ndm, out_cols,
              _lib.ptr(out), _lib.stream_handle())
    np.testing.assert_array_equal(out.cpu().numpy(), _expected(x, off, out_cols))
