"""The block shape an execution takes when nobody set one: both sides of every line of the rule, by the
plan's own report (host code only)."""

from __future__ import annotations

import contextlib
import ctypes

import numpy as np
import pytest

from sigpyproc3_amd import _lib


@contextlib.contextmanager
def _plan(table, nsamps, nbits):
    lib = _lib.load()
    h = ctypes.c_void_p()
    _lib.check(lib.spp_sweep_plan_create(_lib.ptr(table), table.shape[0], table.shape[1], nsamps, nbits, 1,
                                         ctypes.byref(h)))
    try:
        yield h
    finally:
        lib.spp_sweep_plan_destroy(h)


def _info(h):
    info = _lib.SweepInfo()
    _lib.check(_lib.load().spp_sweep_plan_info(h, ctypes.byref(info)))
    return info


def _shape(nbits, nchans, ndm, blocks, per_tile=16):
    """The shape of a plan of `blocks` 16-row blocks whose DM tiles hold `per_tile` rows."""
    step = 252 // per_tile + 1 if per_tile < 16 else 1
    table = np.round(step * np.arange(ndm)[:, None] * np.linspace(0, 1, nchans)[None, :]).astype(np.int32)
    T = 2048 if nbits <= 2 else 1024
    tiles = -(-ndm // per_tile)
    with _plan(table, blocks // tiles * T, nbits) as h:
        info = _info(h)
        assert info.ndm_tiles == tiles and tiles * -(-info.max_len // T) == blocks
        return int(info.mode) // 64


@pytest.mark.parametrize("nbits", [1, 2])
@pytest.mark.parametrize("nchans", [40, 400])
def test_nibble_shapes(nbits, nchans):
    assert [_shape(nbits, nchans, 16, b) for b in (1, 64, 65, 128, 129, 5000)] == [6, 6, 8, 8, 4, 4]
    # 13 of 16 rows in a tile are more than 4/5, 12 are not
    assert [_shape(nbits, nchans, 13, b) for b in (128, 129)] == [8, 4]
    assert [_shape(nbits, nchans, 12, b) for b in (128, 129)] == [8, 7]


def test_4bit_shapes():
    assert [_shape(4, 128, 16, b) for b in (1, 128, 129, 1024, 1025)] == [6, 6, 4, 4, 3]
    assert [_shape(4, 126, 16, b) for b in (128, 129, 1024, 1025)] == [6, 3, 3, 3]
    assert [_shape(4, 128, n, 200) for n in (13, 12)] == [4, 7]  # more than 3/4 of a tile, and not


def test_8bit_shapes():
    assert [_shape(8, 128, 16, b) for b in (1, 128, 129, 16384, 16385)] == [6, 6, 4, 4, 0]
    assert [_shape(8, 127, 16, b) for b in (128, 129, 16385)] == [6, 0, 0]
    assert [_shape(8, 128, n, 200) for n in (13, 12)] == [4, 7]


@pytest.mark.parametrize(("nbits", "full"), [(4, 3), (8, 0)])
def test_narrow_bands_in_sparse_tiles(nbits, full):
    # fewer than 128 channels: two rows a wave only in tiles more than half full
    assert [_shape(nbits, 126, n, 200) for n in (16, 9, 8, 1)] == [full, full, 7, 7]
    assert [_shape(nbits, 126, 64, 64 // per * 20, per) for per in (8, 4, 2, 1)] == [7, 7, 7, 7]


def test_a_shape_that_was_set_stays():
    lib = _lib.load()
    with _plan(np.zeros((4, 16), np.int32), 4096, 2) as h:
        for v in range(lib.spp_sweep_variant_count()):
            _lib.check(lib.spp_sweep_plan_set_variant(h, v))
            assert int(_info(h).mode) // 64 == v
        with pytest.raises(ValueError):
            _lib.check(lib.spp_sweep_plan_set_variant(h, lib.spp_sweep_variant_count()))
