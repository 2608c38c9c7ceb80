"""spp_dedisperse on packed rows of any byte length and stream start, at the edges of the word-
parallel kernel's columns, and on gulps long enough for its wide stages. Sums are integers."""

from __future__ import annotations

import numpy as np
import pytest

from sigpyproc3_amd import _lib


def _run(packed, nbits, big, nchans, nsamps, delays, md):
    out = _lib.to_device(np.full(nsamps - md + 3, -1.0, np.float32))
    d = _lib.to_device(delays)
    _lib.call("spp_dedisperse", _lib.ptr(packed), nbits, big, nchans, nsamps, _lib.ptr(d), md, _lib.ptr(out), 1,
              _lib.stream_handle())
    got = out.cpu().numpy()
    assert got[0] == -1 and (got[nsamps - md + 1 :] == -1).all()
    return got[1 : nsamps - md + 1]


@pytest.mark.gpu
@pytest.mark.parametrize("nbits", [1, 2, 4, 8])
@pytest.mark.parametrize("row_bytes", [4, 5, 6, 7, 9, 15, 17, 31, 33, 66, 127, 129, 259])
def test_swar_rows_of_any_bytes(nbits, row_bytes):
    from oracle import spp_oracle as O

    nchans, nsamps = row_bytes * 8 // nbits, 4500
    rng = np.random.default_rng(nbits * 1000 + row_bytes)
    order = O.DEFAULT_BITORDER.get(nbits, "big")
    x = rng.integers(0, 1 << nbits, (nsamps, nchans), dtype=np.uint8)
    packed = x.reshape(-1) if nbits == 8 else O.pack(x.reshape(-1), nbits, order)
    for lo, hi, shift in ((0, 700, 0), (-90, 300, 1), (0, 2300, 3)):
        delays = np.round(np.linspace(lo, hi, nchans)).astype(np.int32)
        md = int(np.abs(delays).max())
        t = np.arange(nsamps - md)
        want = np.zeros(nsamps - md, np.int64)
        for c in range(nchans):
            rows = t + int(delays[c])
            rows = np.where(rows < 0, rows + nsamps, rows)
            want += np.where(rows < nsamps, x[rows % nsamps, c], 0)
        dev = _lib.to_device(np.concatenate([np.full(shift, 255, np.uint8), packed]))
        got = _run(dev[shift:], nbits, 1 if order == "big" else 0, nchans, nsamps, delays, md)
        np.testing.assert_array_equal(got, want.astype(np.float32), err_msg=f"delays {lo}..{hi}, start {shift}")


@pytest.mark.gpu
@pytest.mark.parametrize(("nbits", "nchans", "hi"), [(2, 4096, 2500), (2, 2064, 0), (8, 1000, 900), (8, 1056, 7000)])
def test_swar_long_gulps(nbits, nchans, hi):
    """At least 1e8 packed bytes: the wide stages (the last one with delays too wide for them)."""
    import torch

    nsamps = 100_000_000 * 8 // (nchans * nbits) + hi + 777
    gen = torch.Generator(device="cuda")
    gen.manual_seed(nchans)
    packed = torch.randint(0, 256, (nsamps, nchans * nbits // 8), generator=gen, device="cuda", dtype=torch.uint8)
    delays = np.round(np.linspace(0, 1, nchans) ** 2 * hi).astype(np.int32)
    md = int(delays.max())
    want = torch.zeros(nsamps - md, dtype=torch.int64, device="cuda")
    per = 8 // nbits
    for c in range(nchans):
        byte = packed[int(delays[c]) : int(delays[c]) + nsamps - md, c // per]
        want += (byte >> (8 - (c % per + 1) * nbits)) & ((1 << nbits) - 1)  # big order at 2 bits
    got = _run(packed.reshape(-1), nbits, 1, nchans, nsamps, delays, md)
    np.testing.assert_array_equal(got, want.cpu().numpy().astype(np.float32))
