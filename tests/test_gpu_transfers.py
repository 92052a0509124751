"""Uploads and downloads around the lengths where pieces and the host's copies change form, from and to unaligned memory."""
import ctypes

import numpy as np
import pytest

from webdnn_amd import capi

pytestmark = pytest.mark.gpu

MIB = 1 << 20


@pytest.mark.parametrize("bytes_", [4, 100, MIB - 4, MIB, MIB + 36, 2 * MIB, 2 * MIB + 4, 3 * MIB + 20, 8 * MIB - 4, 8 * MIB, 15 * MIB + 68, 70 * MIB + 4])
@pytest.mark.parametrize("shift", [0, 1, 4, 63])
def test_every_byte_arrives(ctx, bytes_, shift):
    rng = np.random.default_rng(bytes_ + shift)
    source = rng.integers(0, 256, bytes_ + 128, dtype=np.uint8)
    target = np.full(bytes_ + 256, 0xA5, dtype=np.uint8)
    handle = capi.load().wdh_alloc(bytes_ + 64)
    assert handle > 0
    try:
        for round_ in range(2):  # (the second finds the staging memory used)
            source[shift:shift + bytes_] ^= 0x3C
            capi.call("wdh_write", handle, 4 * round_, source[shift:].ctypes.data_as(ctypes.c_void_p), bytes_)
            at = 128 - shift
            capi.call("wdh_read", handle, 4 * round_, target[at:].ctypes.data_as(ctypes.c_void_p), bytes_)
            assert (target[at:at + bytes_] == source[shift:shift + bytes_]).all()
            assert (target[:at] == 0xA5).all() and (target[at + bytes_:] == 0xA5).all()
    finally:
        capi.call("wdh_free", handle)
