"""Results brought to the host under the callers' torch modes, and after a call that did not end."""

from __future__ import annotations

import threading

import numpy as np
import pytest

from sigpyproc3_amd import _lib

pytestmark = pytest.mark.gpu
N = _lib.STAGE_BYTES  # floats: four pieces


def _in_new_thread(fn):
    """Run fn in a thread without staging buffers of its own yet."""
    out = []

    def work():
        try:
            out.append(fn())
        except BaseException as e:  # noqa: BLE001 - handed to the test
            out.append(e)

    th = threading.Thread(target=work)
    th.start()
    th.join()
    if isinstance(out[0], BaseException):
        raise out[0]
    return out[0]


def _series(k: float):
    import torch

    return torch.arange(N, dtype=torch.float32, device="cuda") + k


def _check(got, k: float):
    np.testing.assert_array_equal(got, np.arange(N, dtype=np.float32) + np.float32(k))
    assert got.flags.writeable


@pytest.mark.parametrize("first_inside", [True, False])
def test_inference_mode_and_after_it(first_inside):
    import torch

    def work():
        results = []
        for inside in (first_inside, not first_inside, first_inside):
            with torch.inference_mode(inside):
                results.append(_lib.to_host(_series(len(results))))
        with torch.inference_mode():
            x = _series(3)  # an inference tensor brought over outside the mode
        results.append(_lib.to_host(x))
        return results

    for k, got in enumerate(_in_new_thread(work)):
        _check(got, k)


@pytest.mark.parametrize("first_inside", [True, False])
def test_default_device(first_inside):
    import torch

    def work():
        results = []
        for inside in (first_inside, not first_inside):
            with torch.device("cuda" if inside else "cpu"):
                results.append(_lib.to_host(_series(len(results))))
        return results

    for k, got in enumerate(_in_new_thread(work)):
        _check(got, k)


def test_after_a_call_that_did_not_end(monkeypatch):
    import torch

    def work():
        _lib.to_host(_series(1))
        kept = _lib._staging.buffers
        calls = []
        with monkeypatch.context() as m:
            real = torch.cuda.Event.synchronize

            def interrupted(self):
                calls.append(self)
                if len(calls) == 2:
                    raise KeyboardInterrupt
                real(self)

            m.setattr(torch.cuda.Event, "synchronize", interrupted)
            with pytest.raises(KeyboardInterrupt):
                _lib.to_host(_series(2))
        # its copies may still be under way: another call must not fill the same buffers
        assert getattr(_lib._staging, "buffers", None) is None
        got = _lib.to_host(_series(5))
        assert _lib._staging.buffers[0] is not kept[0]
        return got

    _check(_in_new_thread(work), 5)
