"""Stage-1 columns of the batch kernel: rows around the 32- and 64-byte column widths, in a block
shape of each, against the C oracle (integer sums, so bit for bit)."""

import numpy as np
import pytest

from oracle import c_oracle
from oracle import spp_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [2, 4])
@pytest.mark.parametrize("row_bytes", [1, 31, 33, 63, 64, 65, 96, 97, 128, 130])
def test_batch_rows_of_any_bytes(shape, row_bytes):
    from sigpyproc3_amd import _lib
    from sigpyproc3_amd.batch import SweepBatch
    from sigpyproc3_amd.sweep import SweepPlan

    rng = np.random.default_rng(row_bytes)
    plans, packed, refs = [], [], []
    for nbits, nsamps in [(1, 2311), (2, 1500), (4, 1025), (8, 700)]:
        nchans = row_bytes * 8 // nbits
        order = O.DEFAULT_BITORDER.get(nbits, "big")
        samples = rng.integers(0, 1 << nbits, nsamps * nchans, dtype=np.uint8)
        table = np.round(np.linspace(0, 1, 6)[:, None] * np.linspace(0, 90, nchans)[None, :]).astype(np.int32)
        plans.append(SweepPlan(table, nsamps, nbits, 1 if order == "big" else 0, allocate=False))
        packed.append(_lib.to_device(samples if nbits == 8 else O.pack(samples, nbits, order)))
        refs.append(c_oracle.sweep(samples, nchans, table, ld=plans[-1].max_len))
    batch = SweepBatch(plans)
    batch.set_shape(shape)
    planes = batch.execute(packed)
    batch.check()
    for plan, plane, ref in zip(plans, planes, refs):
        plane = plane.cpu().numpy()
        for i in range(plan.ndm):
            n = int(plan.row_len[i])
            np.testing.assert_array_equal(plane[i, :n], ref[i, :n], err_msg=f"{plan.nbits}-bit row {i}")
