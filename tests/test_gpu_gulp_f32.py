"""spp_dedisperse on float32 gulps at the edges of the kernel's chunks, tiles and windows.

The reference value is the float64 sum in channel order, rounded once to float32, so equality
is exact."""

from __future__ import annotations

import numpy as np
import pytest

from sigpyproc3_amd import _lib


def _expected(x, delays, md):
    nsamps = x.shape[0]
    acc = np.zeros(nsamps - md, np.float64)
    for c, d in enumerate(delays):
        rows = np.arange(nsamps - md) + int(d)
        rows = np.where(rows < 0, rows + nsamps, rows)
        ok = (rows >= 0) & (rows < nsamps)
        acc += np.where(ok, x[np.where(ok, rows, 0), c], np.float32(0)).astype(np.float64)
    return acc.astype(np.float32)


@pytest.mark.gpu
@pytest.mark.parametrize(
    ("nchans", "nsamps", "lo", "hi"),
    [
        (1, 65, 0, 0),           # one channel: rows narrower than a 16-byte load
        (3, 200, 0, 40),
        (4, 64 + 96, 0, 96),     # one pass of the widest window
        (5, 64 + 97, 0, 97),     # one sample wider: two passes
        (31, 1000, 0, 300),
        (33, 777, 0, 20),        # a chunk of one channel
        (64, 5000, 0, 2500),     # every channel a pass of its own
        (130, 3001, 0, 130),
        (1002, 4097, 0, 1700),
        (96, 3000, -500, 400),   # negative delays wrap inside the gulp
        (4097, 400, 0, 120),     # more channels than the delays kept in LDS
        (48, 66000, 0, 300),
        (48, 65536 + 128, -100, 128),
    ],
)
def test_dedisperse_f32_edges(nchans, nsamps, lo, hi):
    rng = np.random.default_rng(nchans * 131 + nsamps)
    x = (rng.normal(size=(nsamps, nchans)) * 37.0 + 11.0).astype(np.float32)
    delays = np.round(np.linspace(lo, hi, nchans)).astype(np.int32)
    if nchans == 130:
        rng.shuffle(delays)  # windows that jump between channels
    md = int(np.abs(delays).max())
    out = _lib.to_device(np.full(nsamps - md + 7, -1.0, np.float32))
    xd, dd = _lib.to_device(x), _lib.to_device(delays)
    _lib.call("spp_dedisperse", _lib.ptr(xd), 32, 0, nchans, nsamps, _lib.ptr(dd), md, _lib.ptr(out), 5,
              _lib.stream_handle())
    got = out.cpu().numpy()
    np.testing.assert_array_equal(got[5 : 5 + nsamps - md], _expected(x, delays, md))
    assert (got[:5] == -1).all() and (got[5 + nsamps - md :] == -1).all()
