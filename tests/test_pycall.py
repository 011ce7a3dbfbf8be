"""The wrappers' call path (madi_amd/csrc/pycall.c): what it accepts and
refuses, against functions called through ctypes as well."""
import ctypes

import numpy as np
import pytest

from madi_amd import _lib, q8

FAKE = 0x100000  # never dereferenced: every call below fails validation first


class Buffer:
    def data_ptr(self):
        return FAKE


@pytest.mark.parametrize("p", [FAKE, Buffer()])
def test_errors_carry_the_librarys_code(p):
    with pytest.raises(_lib.MadiError) as e:
        _lib.calls.madi_q8_gemv(p, p, p, p, np.int64(100), np.uint32(96))
    assert e.value.code == -5 and "madi_q8_gemv" in str(e.value)  # k % 64
    with pytest.raises(_lib.MadiError) as e:
        _lib.calls.madi_q8_gemv(None, p, p, p, 64, 64)
    assert e.value.code == -6
    with pytest.raises(_lib.MadiError) as e:
        _lib.calls.madi_matmul_f16(p, p, p, -1, 4, 4, 1, 0.0)
    assert e.value.code == -5


@pytest.mark.parametrize("args", [(1, 2), (FAKE,) * 4 + (64, 96.0), (FAKE,) * 4 + (64, None),
                                  ("x", FAKE, FAKE, FAKE, 64, 64), (1.5, FAKE, FAKE, FAKE, 64, 64)])
def test_wrong_arguments_are_refused(args):
    with pytest.raises((TypeError, AttributeError)):
        _lib.calls.madi_q8_gemv(*args)


def test_no_such_entry_point():
    for name in ("madi_nothing", "madi_alloc"):  # not of the int-returning form
        with pytest.raises(AttributeError):
            getattr(_lib.calls, name)


def test_arguments_arrive_in_order():
    """Every call form (up to ten integers, six and two floats) hands each
    argument to its place."""
    from madi_amd import _pycall
    seen = []

    def collect(*a):
        seen.append(a)
        return 0

    fail = lambda code, name: pytest.fail("no error here")
    for n in range(11):
        f = ctypes.CFUNCTYPE(ctypes.c_int, *[ctypes.c_uint64] * n)(collect)
        vals = [(1 << 40) * (i + 1) + i for i in range(n)]
        assert _pycall.bind(ctypes.cast(f, ctypes.c_void_p).value, "p" * n, "f", fail)(*vals) is None
        assert list(seen.pop()) == vals
    types = [ctypes.c_uint64] * 3 + [ctypes.c_int] * 3 + [ctypes.c_float] * 2
    f = ctypes.CFUNCTYPE(ctypes.c_int, *types)(collect)
    call = _pycall.bind(ctypes.cast(f, ctypes.c_void_p).value, "pppiiiff", "f", fail)
    call(1, None, Buffer(), -4, 5, 6, 0.5, 2)
    assert seen.pop() == (1, 0, FAKE, -4, 5, 6, 0.5, 2.0)
    with pytest.raises(ValueError):
        _pycall.bind(1, "pf", "f", fail)
    assert q8.calls is _lib.calls
