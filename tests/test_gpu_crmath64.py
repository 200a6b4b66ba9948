"""The sweeps' float64 roots and quotients (geoswe_amd/csrc/gs_wave.h) equal the general ones on the
device: 2^30 seeded operands within their bounds, every other one of a significand whose root or
reciprocal lies next to a midpoint."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_wave_float64_forms_equal_general(gpu):
    from geoswe_amd import _lib as L
    counts = L.DeviceArray((4,), np.uint64, zero=True)
    L.call("gs_crmath_check", 5, counts.ptr, None)
    L.sync(None)
    c = counts.download()
    assert c[0] == 0, f"root: {int(c[0])} mismatches, last index {int(c[1]) - 1:#x}"
    assert c[2] == 0, f"quotients: {int(c[2])} mismatches, last index {int(c[3]) - 1:#x}"
