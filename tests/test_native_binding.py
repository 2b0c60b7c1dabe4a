"""The CPython binding of the launch entry points: what it accepts and raises
(no GPU needed: the calls below are refused, or have nothing to do)."""
import ctypes as C

import numpy as np
import pytest

from glow_amd import capi


class _Buffer:
    ptr = 64


@pytest.mark.parametrize("pointer", [None, 64, _Buffer(), np.zeros(4, np.int8)[::2],
                                     (C.c_int32 * 3)(), np.int64(64), C.c_void_p(64).value])
def test_pointer_forms(pointer):
    capi.launch_quantize_i8(pointer, pointer, 0, np.float32(0.5), np.int64(-3))   # nothing to do


@pytest.mark.parametrize("kind", [np.int64, np.uint64, np.intp, np.int32, np.uint8])
def test_numpy_integers_are_addresses(kind):
    """The number itself, not the memory of the scalar object: zero is NULL."""
    a = np.zeros(16, np.float32)
    for d, s in ((kind(0), a), (a, kind(0))):
        with pytest.raises(capi.MI355XError) as e:
            capi.launch_quantize_i8(d, s, 16, 0.5, 0)
        assert e.value.code == -1 and "NULL" in str(e.value)


@pytest.mark.parametrize("pointer", [C.c_void_p(64), C.c_void_p(0), C.c_int64(64), "no address"])
def test_what_is_no_pointer_is_refused(pointer):
    """A ctypes integer is neither a number nor memory to read from."""
    with pytest.raises((TypeError, ValueError)):
        capi.launch_quantize_i8(pointer, 64, 0, 0.5, 0)


def test_status_becomes_the_librarys_error():
    with pytest.raises(capi.MI355XError) as e:
        capi.launch_rescale_i8(64, 64, 16, 0, 0, 32, 0, 1)
    assert e.value.code == -1 and "shift" in str(e.value)
    with pytest.raises(capi.MI355XError) as e:
        capi.launch_rwq_fc_i8(64, 64, 64, 64, False, None, *[64] * 6, 2, 3, 4, 0, 0, 0)
    assert e.value.code == -1


def test_per_call_options_reach_the_library():
    with pytest.raises(capi.MI355XError) as e:
        capi.launch_frwq_slws(64, False, 64, 1, 0, None, False, 64, True, 0, 64, 0, 12, 4,
                              opts=capi.LaunchOpts(slws_math=3))
    assert "slws_math" in str(e.value)


def test_wrong_arguments_are_type_errors():
    with pytest.raises(TypeError):
        capi.native().quantize_i8(64, 64)
    with pytest.raises((TypeError, ValueError)):
        capi.launch_quantize_i8(64, 64, "many", 0.5, 0)
