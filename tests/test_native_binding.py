"""csrc/pynative.cpp: the CPython binding of the device entries."""
import ctypes as C

import numpy as np
import pytest

import rustorch_amd as ra
from rustorch_amd import _lib as L


def test_native_binding_converts_arguments_and_reports_errors():
    """Addresses, streams and shapes as objects, errors as the tuple errors.check takes."""
    class Buf:
        ptr = 16

    class Handle:
        _as_parameter_ = C.c_void_p(0)

    call = L.native.rt_gqa_decode_online_bf16
    for stream in (None, 0, C.c_void_p(), Handle()):
        for buf in (16, np.int64(16), Buf()):
            assert call(stream, buf, buf, buf, buf, 8, 3, 1, 64, 10)[:4] == (L.RT_ERR_HEAD_COUNT_MISMATCH, -1, 8, 3)
    with pytest.raises(ra.Overflow) as e:
        ra.LlmKernels.gqa_decode_online_bf16(None, 16, 16, 16, 16, 8, 2, 11, 64, 10)
    assert (e.value.requested, e.value.max) == (11, 10)
    with pytest.raises(ra.ZeroDim):
        ra.flash_forward_bf16_dev(ra.AttentionShape.new(1, 1, 4, 0), 16, 16, 16, 16)
    for bad in ("x", 1.5, [16]):
        with pytest.raises(TypeError):
            call(None, bad, 16, 16, 16, 8, 2, 1, 64, 10)
    with pytest.raises(TypeError):
        call(None, 16, 16, 16, 16, 8, 2, 1, 64)
    with pytest.raises(TypeError):
        call(None, 16, 16, 16, 16, 8, 2, 1.0, 64, 10)
