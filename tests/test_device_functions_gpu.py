"""The device's reciprocals, inverse square roots, rcpps and depth keys for
every float: the corrected estimates equal the correctly rounded operators,
rcpps and the key their definitions, bit for bit."""
import ctypes
import os

import pytest
import torch  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("which", [0, 1, 2, 3], ids=["recip", "recip_sqrt", "rcpps", "depth_order"])
def test_every_float(which):
    from rsr_amd import build
    if not os.path.exists(build.CHECKS_LIB):
        build.build_checks()
    L = ctypes.CDLL(build.CHECKS_LIB)
    out = (ctypes.c_ulonglong * 2)()
    assert L.rgl_check_all(which, out) == 0
    assert out[0] == 0, f"{out[0]} inputs differ, {out[1]:#010x} among them"
