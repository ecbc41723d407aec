"""The traversal's stacks, run on the host beside a plain list: entries come back
in order from LDS and the overflow area, and one beyond the limit is dropped
without a later pop reading past the area."""
import ctypes
import os

import pytest

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "bin", "libkernel_checks.so")


@pytest.mark.parametrize("grow", [45, 55, 70, 95])
@pytest.mark.parametrize("which", ["lane", "quad", "quad after a lane"])
def test_stack_against_a_list(which, grow):
    assert os.path.exists(LIB), "tests/bin/libkernel_checks.so missing: build with `make -C lighthouse2_amd/csrc`"
    check = ctypes.CDLL(LIB).check_stack
    check.argtypes = [ctypes.c_int, ctypes.c_uint32, ctypes.c_int]
    for seed in range(1, 40):
        assert check(["lane", "quad", "quad after a lane"].index(which), seed * 2654435761 % (1 << 32), grow) == -1, seed
