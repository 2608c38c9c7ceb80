"""One-DM dedispersion of packed gulps: which ones the word-parallel kernel takes (host rule, at sizes
timed on both kernels), and 1/2-bit rows of any bytes on the GPU in either. Sums are integers."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from sigpyproc3_amd import _lib


def _word_parallel(nbits, nchans, nsamps, md, aligned=False):
    # spp::gulp_swar_applies(nbits, aligned, nchans, nout, max_delay)
    fn = _lib.load()._ZN3spp17gulp_swar_appliesEiblll
    fn.restype = ctypes.c_bool
    fn.argtypes = [ctypes.c_int, ctypes.c_bool] + [ctypes.c_int64] * 3
    return fn(nbits, aligned, nchans, nsamps - md, md)


@pytest.mark.parametrize(
    ("nbits", "nchans", "nsamps", "md", "word"),
    [
        # times measured in the word-parallel and in the byte-staged kernel, in us
        (1, 336, 20011, 500, False),      # 17, 9
        (1, 336, 65536, 500, True),       # 17, 20
        (2, 132, 65536, 0, False),        # 14, 10
        (1, 72, 262144, 20000, False),    # 202, 86
        (1, 1040, 4096, 0, False),        # 17, 10
        (1, 1000, 262144, 5000, True),    # 49, 201
        (2, 36, 262144, 20000, False),    # 135, 52
        (2, 260, 20011, 500, False),      # 14, 10
        (2, 1004, 262144, 5000, True),    # 58, 203
        (4, 10, 262144, 1000, True),      # 7, 12
        (4, 66, 4096, 0, True),           # 10, 10
        (4, 1002, 100003, 40000, True),   # 52, 148
        (8, 5, 262144, 60000, True),      # 9, 12
        (8, 1001, 16384, 300, True),      # 14, 26
        (8, 3, 262144, 1000, False),      # less than a dword
    ],
)
def test_rule(nbits, nchans, nsamps, md, word):
    assert _word_parallel(nbits, nchans, nsamps, md) == word
    if nchans * nbits >= 32:
        assert _word_parallel(nbits, nchans, nsamps, md, aligned=True)


def _by_lines(nbits, nchans, nsamps, md):
    fn = _lib.load()._ZN3spp18gulp_swar_by_linesEilll  # spp::gulp_swar_by_lines(nbits, nchans, nout, max_delay)
    fn.restype = ctypes.c_bool
    fn.argtypes = [ctypes.c_int] + [ctypes.c_int64] * 3
    return fn(nbits, nchans, nsamps - md, md)


@pytest.mark.parametrize(
    ("nbits", "nchans", "nsamps", "md", "lines"),
    [
        # times measured by lines and in contiguous groups, in us
        (8, 1024, 65536, 2000, True),     # whole lines
        (8, 1000, 200000, 5000, True),    # 86, 200
        (8, 160, 524288, 100, True),      # 40, 48
        (8, 160, 262144, 100, False),     # 26, 21
        (8, 192, 262144, 8000, False),    # 40, 37
        (8, 124, 1 << 20, 0, False),      # less than a line
        (4, 1000, 200000, 5000, False),   # 68, 62
        (2, 896, 524288, 100, True),      # 57, 66
        (2, 640, 524288, 100, False),     # 58, 49
        (2, 1152, 262144, 8000, True),    # 53, 70
        (1, 2560, 524288, 100, True),     # 113, 132
        (1, 2176, 524288, 100, False),    # 115, 107
        (1, 2304, 262144, 8000, True),    # 67, 80
    ],
)
def test_line_rule(nbits, nchans, nsamps, md, lines):
    assert _by_lines(nbits, nchans, nsamps, md) == lines


@pytest.mark.gpu
@pytest.mark.parametrize(("nbits", "nchans", "nsamps", "hi", "lines"), [
    (8, 160, 380000, 100, True), (8, 160, 100000, 100, False), (8, 192, 400000, 9000, True), (8, 300, 100003, 9000, False),
    (2, 640, 640000, 900, True), (2, 640, 100000, 900, False), (2, 1152, 100000, 8000, True), (1, 1312, 200000, 3000, True),
    (1, 1312, 200000, 300, False)])
def test_cut_lines(nbits, nchans, nsamps, hi, lines):
    import torch

    assert _by_lines(nbits, nchans, nsamps, hi) == lines
    gen = torch.Generator(device="cuda")
    gen.manual_seed(nchans)
    packed = torch.randint(0, 256, (nsamps, nchans * nbits // 8), generator=gen, device="cuda", dtype=torch.uint8)
    delays = np.round(np.linspace(0, 1, nchans) ** 2 * hi).astype(np.int32)
    per = 8 // nbits
    want = torch.zeros(nsamps - hi, dtype=torch.int64, device="cuda")
    for c in range(nchans):
        byte = packed[int(delays[c]) : int(delays[c]) + nsamps - hi, c // per]
        want += (byte >> (8 - (c % per + 1) * nbits)) & ((1 << nbits) - 1)  # big bit order
    out = torch.full((nsamps - hi + 2,), -1.0, device="cuda")
    d = _lib.to_device(delays)
    _lib.call("spp_dedisperse", _lib.ptr(packed), nbits, 1, nchans, nsamps, _lib.ptr(d), hi, _lib.ptr(out), 1,
              _lib.stream_handle())
    got = out.cpu().numpy()
    assert got[0] == -1 and got[-1] == -1
    np.testing.assert_array_equal(got[1:-1], want.cpu().numpy().astype(np.float32))


def _samples(packed_rows, nbits, nchans, big):
    per = 8 // nbits
    shifts = [(8 - (k + 1) * nbits) if big else k * nbits for k in range(per)]
    x = np.stack([(packed_rows >> s) & ((1 << nbits) - 1) for s in shifts], axis=-1)
    return x.reshape(len(packed_rows), -1)[:, :nchans]


@pytest.mark.gpu
@pytest.mark.parametrize("nbits", [1, 2])
@pytest.mark.parametrize("big", [0, 1])
@pytest.mark.parametrize(
    ("row_bytes", "nsamps", "lo", "hi", "shift", "word"),
    [
        (127, 90000, 0, 700, 0, True), (129, 90000, 0, 700, 3, True), (66, 150000, -90, 300, 1, True),
        (127, 9000, 0, 700, 0, False), (42, 20011, 0, 500, 0, False), (9, 30000, -200, 9000, 2, False),
        (5, 5000, 0, 0, 1, False),
    ],
)
def test_rows_of_any_bytes(nbits, big, row_bytes, nsamps, lo, hi, shift, word):
    nchans = row_bytes * 8 // nbits
    rng = np.random.default_rng(row_bytes)
    rows_host = rng.integers(0, 256, (nsamps, row_bytes), dtype=np.uint8)
    delays = np.round(np.linspace(lo, hi, nchans)).astype(np.int32)
    md = int(np.abs(delays).max())
    assert _word_parallel(nbits, nchans, nsamps, md) == word
    x = _samples(rows_host, nbits, nchans, big)
    t = np.arange(nsamps - md)
    want = np.zeros(nsamps - md, np.int64)
    for c in range(nchans):
        rows = t + int(delays[c])
        rows = np.where(rows < 0, rows + nsamps, rows)
        want += np.where(rows < nsamps, x[rows % nsamps, c], 0)
    dev = _lib.to_device(np.concatenate([np.full(shift, 255, np.uint8), rows_host.reshape(-1)]))
    out = _lib.to_device(np.full(nsamps - md + 3, -1.0, np.float32))
    d = _lib.to_device(delays)
    _lib.call("spp_dedisperse", _lib.ptr(dev[shift:]), nbits, big, nchans, nsamps, _lib.ptr(d), md, _lib.ptr(out), 1,
              _lib.stream_handle())
    got = out.cpu().numpy()
    assert got[0] == -1 and (got[nsamps - md + 1 :] == -1).all()
    np.testing.assert_array_equal(got[1 : nsamps - md + 1], want.astype(np.float32))
