"""Device functions whose exactness is claimed for every input of a range,
on all of it: the one-step reciprocal against the IEEE quotient (it holds only
through what v_rcp_f32 returns), exp2f_fast against the form that
oracle/exp2_check.c holds against libm."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from conftest import REPO

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def math():
    lib = C.CDLL(str(REPO / "tests" / "device_math" / "libdevice_math.so"))
    for f in (lib.device_math_rcp_ge1, lib.device_math_exp2_mismatches):
        f.argtypes = [C.c_uint32, C.c_uint32, C.c_void_p, C.c_void_p]
        f.restype = C.c_int
    return lib


@pytest.mark.parametrize("exponent", [0, 1, 2, 24, 63, 100, 124, 125])
def test_rcp_ge1_every_significand(cuda, math, exponent):
    """1 / d for all 2^23 significands of d in [2^exponent, 2^(exponent + 1))."""
    first, n = (127 + exponent) << 23, 1 << 23
    out = torch.empty(n, dtype=torch.float32, device=cuda)
    stream = torch.cuda.current_stream().cuda_stream
    assert math.device_math_rcp_ge1(first, n, out.data_ptr(), stream) == 0
    d = np.arange(first, first + n, dtype=np.uint32).view(np.float32)
    ref = (np.float32(1) / d).view(np.uint32)
    bad = np.flatnonzero(out.cpu().numpy().view(np.uint32) != ref)
    assert bad.size == 0, (bad.size, d[bad[:4]])


def test_exp2f_fast_every_float(cuda, math):
    count = torch.zeros(2, dtype=torch.int64, device=cuda)
    stream = torch.cuda.current_stream().cuda_stream
    for first in range(0, 1 << 32, 1 << 28):
        assert math.device_math_exp2_mismatches(first, 1 << 28, count.data_ptr(), stream) == 0
    # [0, 200], [-151, -0]: bit patterns up to and with the last
    last = [int(np.float32(v).view(np.uint32)) & 0x7FFFFFFF for v in (200, 151)]
    assert count.tolist() == [sum(last) + 2, 0]
