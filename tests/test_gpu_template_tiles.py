"""spp_convolve_templates at the edges of its tiles: tap counts around the groups of four taps and
up to the longest, series shorter and longer than a block.

The convolution is float64 rounded once to float32 (half an ulp, 6e-8 relative); the float64
sums of at most 2048 products err by about 1e-12 of their terms."""

from __future__ import annotations

import numpy as np
import pytest

from sigpyproc3_amd.core import kernels


@pytest.mark.gpu
@pytest.mark.parametrize("n", [2048, 2050, 5000, 1024 * 9 + 216])
def test_template_tiles(n):
    rng = np.random.default_rng(n)
    z = rng.normal(size=n).astype(np.float32)
    lens = [1, 2, 3, 4, 5, 7, 8, 9, 255, 1023, 1026, 2047, 2048]
    temps = [rng.uniform(0.1, 1.0, m).astype(np.float32) for m in lens]
    refs = [0, 1, 2, 0, 4, 3, 7, 0, 100, 1022, 5, 2046, 1000]
    ng = kernels.good_size_real(n)
    assert ng % 2 == 0
    zt = z.astype(np.float64)[np.arange(ng) % n]
    got = kernels.convolve_templates(z, temps, refs)
    for k, (h, ref) in enumerate(zip(temps, refs)):
        h = h.astype(np.float64)
        mu, var = h.sum() / ng, (h**2).sum() - h.sum() ** 2 / ng
        acc = np.zeros(n)
        for m in range(h.size):
            acc += h[m] * zt[(np.arange(n) - ref + m) % ng]
        want = (acc - mu * zt.sum()) / np.sqrt(var)
        np.testing.assert_allclose(got[k], want, rtol=1.2e-7, atol=1e-9, err_msg=f"{h.size} taps")
