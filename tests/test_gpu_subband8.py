"""spp_subband on 8-bit gulps of many outputs: band maps, delays and sizes at the edges of the
whole-band kernel's stages, some of which the byte-staged kernel takes (test_subband8_bands.py asserts
which calls take which). Sums are integers below 2^24, so equality is exact."""

from __future__ import annotations

import numpy as np
import pytest

from sigpyproc3_amd import _lib


def _expected(x, delays, bands, md, nsubs, out_size):
    nsamps, nchans = x.shape
    nout = nsamps - md
    acc = np.zeros(max(out_size, (nout + 2) * nsubs + int(bands.max()) + 1), np.int64)
    t = np.arange(nout)
    for c in range(nchans):
        rows = t + int(delays[c])
        rows = np.where(rows < 0, rows + nsamps, rows)
        ok = (rows >= 0) & (rows < nsamps)
        if bands[c] >= 0:
            acc[t * nsubs + int(bands[c])] += np.where(ok, x[np.where(ok, rows, 0), c], 0)
    return acc[:out_size].astype(np.float32)


def _run(x, delays, bands, md, nsubs, out_size):
    out = _lib.to_device(np.full(out_size + 5, -1.0, np.float32))
    dev = [_lib.to_device(a) for a in (x, delays, bands)]
    _lib.call("spp_subband", _lib.ptr(dev[0]), 8, 0, x.shape[1], x.shape[0], _lib.ptr(dev[1]), _lib.ptr(dev[2]), md,
              nsubs, _lib.ptr(out), out_size, _lib.stream_handle())
    got = out.cpu().numpy()
    assert (got[out_size:] == -1).all()
    return got[:out_size]


@pytest.mark.gpu
@pytest.mark.parametrize(
    ("nchans", "nsubs", "nsamps", "lo", "hi"),
    [
        (16, 8, 26000, 0, 40),       # less than a stage
        (20, 10, 21000, 0, 700),     # a partial 16-channel group
        (68, 17, 12900, 0, 300),     # a second stage of 4 channels
        (136, 8, 26500, 0, 1200),    # 17-channel bands
        (192, 64, 4096 + 7, 0, 0),
        (256, 128, 2800, 0, 1100),   # delays wider than the output tile
        (520, 8, 26100, -300, 900),  # 65 channels per band on average; negative delays wrap
        (1024, 64, 5000, 0, 800),
        (2052, 36, 7000, 0, 1024),   # 57-channel bands over every stage boundary
        (4096, 32, 6600, 0, 257),
    ],
)
def test_subband8_sizes(nchans, nsubs, nsamps, lo, hi):
    rng = np.random.default_rng(nchans * 7 + nsubs)
    x = rng.integers(0, 256, (nsamps, nchans), dtype=np.uint8)
    delays = np.round(np.linspace(lo, hi, nchans)).astype(np.int32)
    bands = (np.arange(nchans) // (nchans // nsubs)).clip(max=nsubs - 1).astype(np.int32)
    md = int(np.abs(delays).max())
    size = (nsamps - md) * nsubs
    np.testing.assert_array_equal(_run(x, delays, bands, md, nsubs, size),
                                  _expected(x, delays, bands, md, nsubs, size))


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["interleaved", "shuffled", "gaps", "dropped", "beyond", "short"])
def test_subband8_maps(kind):
    rng = np.random.default_rng(len(kind))
    nchans, nsubs, nsamps, md = 132, 12, 18001, 411
    x = rng.integers(0, 256, (nsamps, nchans), dtype=np.uint8)
    delays = rng.integers(0, md + 1, nchans).astype(np.int32)
    delays[5] = md
    bands = (np.arange(nchans) // 11).astype(np.int32)
    size = (nsamps - md) * nsubs
    if kind == "interleaved":
        bands = (np.arange(nchans) % nsubs).astype(np.int32)
    elif kind == "shuffled":
        rng.shuffle(bands)
    elif kind == "gaps":  # uneven bands, some without channels
        bands = np.sort(rng.choice([0, 1, 4, 5, 6, 7, 11], nchans)).astype(np.int32)
    elif kind == "dropped":  # channels of no band
        bands[::9] = -1
    elif kind == "beyond":  # a band index past the row lands in the next row
        bands[-7:] = nsubs
    else:  # a result buffer that ends inside a row
        size -= 5 * nsubs + 2
    np.testing.assert_array_equal(_run(x, delays, bands, md, nsubs, size),
                                  _expected(x, delays, bands, md, nsubs, size))
