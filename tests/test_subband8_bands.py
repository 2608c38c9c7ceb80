"""8-bit subbands: which calls the whole-band kernel takes (host rule, both sides of its lines), and,
on the GPU, maps with bands too wide for one block, falling maps and negative delays in it. Sums are
integers below 2^24, so equality is exact."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from sigpyproc3_amd import _lib


def _applies(nchans, nsamps, md, nsubs, address=4096):
    fn = _lib.load()._ZN3spp16subband8_appliesEPKvllll  # spp::subband8_applies(in, nchans, nsamps, nout, nsubs)
    fn.restype = ctypes.c_bool
    fn.argtypes = [ctypes.c_void_p] + [ctypes.c_int64] * 4
    return fn(address, nchans, nsamps, nsamps - md, nsubs)


@pytest.mark.parametrize(
    ("nchans", "nsamps", "md", "nsubs", "whole"),
    [
        # times measured with whole bands and with atomics, in us
        (1024, 131072, 5077, 64, True),    # 69, 407
        (512, 32768, 0, 8, True),          # 23, 33: a short gulp's channel groups add atomics
        (64, 32768, 0, 8, False),          # 23, 12.5
        (32, 32768, 0, 16, True),          # 25, 31
        (16, 131072, 4096, 8, True),       # 36, 39
        (16, 131072, 13107, 8, False),     # 71, 44: the delay spread of 16 channels
        (64, 262144, 60000, 8, False),     # 137, 93
        (64, 262144, 131072, 8, False),    # 264, 57
        (64, 131072, 13107, 32, True),     # 64, 194: spread, but more bands
        (1024, 262144, 100000, 64, True),  # 246, 747
        (4096, 65536, 2500, 32, True),     # 128-channel bands
        (4096, 65536, 2500, 16, False),    # 256-channel bands
        (1026, 131072, 0, 64, False),      # rows that are not whole dwords
        (64, 524288, 0, 1, False),         # 20, 15: few bands
        (64, 524288, 800, 1, True),        # 19, 37
        (64, 131072, 800, 2, False),       # 18, 10
        (128, 131072, 12000, 2, True),     # 29, 49
        (64, 131072, 0, 4, False),         # 20, 13
        (64, 524288, 0, 4, True),          # 24, 37
        (24, 131072, 0, 6, True),          # 16, 21
    ],
)
def test_rule(nchans, nsamps, md, nsubs, whole):
    assert _applies(nchans, nsamps, md, nsubs) == whole
    assert not _applies(nchans, nsamps, md, nsubs, address=4098)


def _runs(*widths):
    """The map of bands 0, 1, ... of these widths."""
    return np.repeat(np.arange(len(widths)), widths).astype(np.int32)


ONES = [1] * 20
MAPS = {
    "wide first": (640, 32, _runs(400, *ONES, *([22] * 10))),
    "wide last": (640, 32, _runs(*ONES, *([20] * 11), 400)),
    "wide inside": (640, 32, _runs(*ONES, 60, 500, *([6] * 10))),
    "two wide": (640, 32, _runs(300, *ONES, 300, *([2] * 10))),
    "wide next to wide": (640, 16, _runs(*([2] * 10), 310, 310)),
    "256 and 257": (640, 16, _runs(10, 256, 30, 257, *([8] * 9), 15)),
    "one band": (512, 8, np.full(512, 5, np.int32)),
    "last channel alone": (516, 16, _runs(515, 1)),
    "within the last stage": (524, 16, _runs(*([30] * 8), 270, 14)),
    "57 channels": (2052, 36, _runs(*([57] * 36))),
}


def _expected(x, delays, bands, md, nsubs, out_size):
    nsamps, nchans = x.shape
    t = np.arange(nsamps - md)
    acc = np.zeros((nsamps - md) * nsubs, np.int64)
    for c in range(nchans):
        rows = t + int(delays[c])
        rows = np.where(rows < 0, rows + nsamps, rows)
        ok = rows < nsamps
        acc[t * nsubs + int(bands[c])] += np.where(ok, x[np.where(ok, rows, 0), c], 0)
    return acc[:out_size].astype(np.float32)


def _compare(nchans, nsubs, nsamps, delays, bands, cut=0):
    x = np.random.default_rng(nchans + nsubs).integers(0, 256, (nsamps, nchans), dtype=np.uint8)
    md = int(np.abs(delays).max())
    size = (nsamps - md) * nsubs - cut
    out = _lib.to_device(np.full(size + 5, -1.0, np.float32))
    dev = [_lib.to_device(np.ascontiguousarray(a)) for a in (x, delays, bands)]
    assert _applies(nchans, nsamps, md, nsubs, dev[0].data_ptr())
    _lib.call("spp_subband", _lib.ptr(dev[0]), 8, 0, nchans, nsamps, _lib.ptr(dev[1]), _lib.ptr(dev[2]), md, nsubs,
              _lib.ptr(out), size, _lib.stream_handle())
    got = out.cpu().numpy()
    assert (got[size:] == -1).all()
    np.testing.assert_array_equal(got[:size], _expected(x, delays, bands, md, nsubs, size))


@pytest.mark.gpu
@pytest.mark.parametrize("falling", [False, True])
@pytest.mark.parametrize("name", sorted(MAPS))
def test_band_widths(name, falling):
    nchans, nsubs, bands = MAPS[name]
    assert len(bands) == nchans and bands.max() < nsubs
    delays = np.round(np.linspace(0, 300, nchans)).astype(np.int32)
    _compare(nchans, nsubs, 20000, delays, bands[::-1] if falling else bands, cut=7 if falling else 0)


@pytest.mark.gpu
@pytest.mark.parametrize("widths", [(10, 128, 30, 129, *([8] * 40), 23), (250, 250, *([4] * 35))])
def test_widest_band_of_one_block_by_gulp_length(widths):
    """Bands of 129 to 256 channels are shared in short gulps only."""
    bands = _runs(*widths)
    delays = np.round(np.linspace(0, 300, len(bands))).astype(np.int32)
    for nsamps in (20000, 60000):
        _compare(len(bands), 48, nsamps, delays, bands)


@pytest.mark.gpu
def test_many_outputs_per_block_group():
    """Enough outputs that a block takes several stages of channels."""
    nchans, nsubs = 512, 32
    bands = _runs(*([4] * 20), 400, *([32] * 1))
    delays = np.round(np.linspace(0, 900, nchans)).astype(np.int32)
    _compare(nchans, nsubs, 700000 // 4, delays, bands)


@pytest.mark.gpu
@pytest.mark.parametrize(("nchans", "nsubs", "lo", "hi"), [(512, 8, -300, 900), (640, 32, -1000, -3), (16, 8, -40, 40)])
def test_negative_delays(nchans, nsubs, lo, hi):
    delays = np.round(np.linspace(lo, hi, nchans)).astype(np.int32)
    bands = (np.arange(nchans) * nsubs // nchans).astype(np.int32)
    _compare(nchans, nsubs, 46000 if nchans == 16 else 20000, delays, bands)
