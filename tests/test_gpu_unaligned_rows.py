"""The sweep's stage-1 copy of streams whose rows are not whole dwords, or start at any byte:
rows narrower than a dword, one byte past a dword, and past a 64-byte column block."""

from __future__ import annotations

import numpy as np
import pytest

from oracle import spp_oracle as O


@pytest.mark.gpu
@pytest.mark.parametrize("nbits", [1, 2, 4, 8])
@pytest.mark.parametrize("row_bytes", [1, 2, 3, 4, 5, 7, 63, 65, 66, 127, 130])
def test_sweep_rows_of_any_bytes(nbits, row_bytes):
    from sigpyproc3_amd import _lib
    from sigpyproc3_amd.sweep import SweepPlan

    nchans, nsamps = row_bytes * 8 // nbits, 2311
    rng = np.random.default_rng(nbits * 1000 + row_bytes)
    order = O.DEFAULT_BITORDER.get(nbits, "big")
    x = rng.integers(0, 1 << nbits, (nsamps, nchans), dtype=np.uint8)
    packed = x.reshape(-1) if nbits == 8 else O.pack(x.reshape(-1), nbits, order)
    table = np.round(np.linspace(0, 1, 5)[:, None] * np.linspace(0, 90, nchans)[None, :]).astype(np.int32)
    plan = SweepPlan(table, nsamps, nbits, 1 if order == "big" else 0)
    for shift in (0, 1, 3):
        dev = _lib.to_device(np.concatenate([np.full(shift, 255, np.uint8), packed]))
        plane = plan.execute(dev[shift:]).cpu().numpy()
        for i, d in enumerate(table):
            n = nsamps - int(d.max())
            want = np.zeros(n, np.int64)
            for c in range(nchans):
                want += x[d[c] : d[c] + n, c]
            np.testing.assert_array_equal(plane[i, :n], want.astype(np.float32), err_msg=f"row {i} shift {shift}")
