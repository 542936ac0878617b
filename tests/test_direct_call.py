"""The native callables in front of the C ABI's ctypes functions: what they pass on, and that everything else still ends at ctypes, with its
results and its errors."""
import ctypes as C
import os

import numpy as np
import pytest

from attention_amd import hip

LIB = os.path.join(os.path.dirname(hip.LIB_PATH), "_direct_call.so")


@pytest.fixture()
def calls():
    """(native callable bound to a Python function of ahpc_hip_flash_fwd_gqa's type, what arrived there)."""
    from importlib import machinery, util
    spec = util.spec_from_file_location("_direct_call", LIB, loader=machinery.ExtensionFileLoader("_direct_call", LIB))
    direct = util.module_from_spec(spec)
    spec.loader.exec_module(direct)
    seen = []
    res, args = hip.SIGNATURES["ahpc_hip_flash_fwd_gqa"]
    target = C.CFUNCTYPE(res, *args)(lambda *a: seen.append(a) or 7)
    slow_calls = []

    def slow(*a):
        slow_calls.append(a)
        return target(*a)

    fn = direct.bind("ahpc_hip_flash_fwd_gqa", C.cast(target, C.c_void_p).value, slow)
    yield fn, seen, slow_calls, target
    del fn, target


ARGS = (2 ** 47 + 1, 5, 6, 7, 1, 2 ** 40, 3, -4, 8, 9, 10, 11, 12, 13, 14, 15, 0.125, 1, None, 2 ** 63 + 5)


def test_arguments_arrive(calls):
    fn, seen, slow, _ = calls
    assert fn(*ARGS) == 7 and not slow
    assert seen == [ARGS]
    assert fn(*ARGS[:16], np.float64(0.5), *ARGS[17:]) == 7 and not slow and seen[1][16] == 0.5


@pytest.mark.parametrize("at,value", [(0, C.c_void_p(3)), (4, True), (16, 1), (5, np.int64(3))])
def test_everything_else_goes_to_ctypes(calls, at, value):
    fn, seen, slow, target = calls
    args = list(ARGS)
    args[at] = value
    try:
        want = target(*args)
    except C.ArgumentError:
        with pytest.raises(C.ArgumentError):
            fn(*args)
    else:
        assert fn(*args) == want and seen[0] == seen[1]
    assert len(slow) == 1


def test_wrong_counts_and_types_raise(calls):
    fn = calls[0]
    with pytest.raises(TypeError):
        fn(*ARGS[:-1])
    with pytest.raises(C.ArgumentError):
        fn("text", *ARGS[1:6], "text", *ARGS[7:])
