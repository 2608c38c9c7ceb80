"""Results brought to the host in pieces: sizes around the staging buffers, views, threads."""

from __future__ import annotations

import threading

import numpy as np
import pytest

from sigpyproc3_amd import _lib

B = _lib.STAGE_BYTES


@pytest.mark.gpu
@pytest.mark.parametrize(("n", "dtype"), [(0, "float32"), (3, "uint8"), (B - 1, "uint8"), (B, "uint8"), (2 * B, "uint8"),
                                          (2 * B + 1, "uint8"), (3 * B // 4, "float32"), (5 * B // 4 + 1, "int32"),
                                          (B, "float64")])
def test_to_host_sizes(n, dtype):
    want = np.random.default_rng(n).integers(0, 100, n).astype(dtype)
    got = _lib.to_host(_lib.to_device(want))
    assert got.dtype == want.dtype and got.flags.writeable
    np.testing.assert_array_equal(got, want)


@pytest.mark.gpu
def test_to_host_views_and_threads():
    import torch

    x = torch.arange(6 * B // 4, dtype=torch.int32, device="cuda").reshape(-1, 64)
    np.testing.assert_array_equal(_lib.to_host(x.t()), x.cpu().numpy().T)
    np.testing.assert_array_equal(_lib.to_host(x[5:, :60]), x.cpu().numpy()[5:, :60])
    got = [None] * 6

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            y = torch.full((B + 17,), float(i), device="cuda")
            y += 1
            got[i] = _lib.to_host(y)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(got))]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    for i, y in enumerate(got):
        assert y.shape == (B + 17,) and (y == i + 1).all()
