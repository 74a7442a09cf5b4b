"""Which form of the BF16 kernel of several rows a launch takes: the library holds the forms that the rule gives and no others, and
the tests on the GPU run each of them."""
import ctypes
import re

import pytest

from mykuiperllama_amd.build import KX_LIB
from tests.test_gpu_bf16_held import FORMS

# a block and its neighbours where the rule looks at their number, and numbers between
BLOCKS = sorted({1, 255, 256, 257, 1023, 1024, 1025, 5119, 5120, 5121, *range(1026, 12000, 97)})


def form(lib, on_lines, M, K, N):
    """(waves, elements per unit, units, waves to a block, runs)"""
    fields = (ctypes.c_int32 * 5)()
    assert lib.kx_bf16_held_form(on_lines, M, K, N, fields), (M, K, N)
    return tuple(fields)


@pytest.fixture(scope="module")
def reached():
    lib = ctypes.CDLL(KX_LIB)
    return {form(lib, on_lines, M, K, 16 * blocks) for K in range(8, 8193, 8) for on_lines in ((0, 1) if K % 64 == 0 else (0,))
            for blocks in BLOCKS for M in (5, 6)}


def test_the_library_holds_what_the_rule_gives(reached):
    with open(KX_LIB, "rb") as f:
        names = re.findall(rb"bf16_gemv_held_kernelILi(\d+)ELi(\d+)ELi(\d+)ELi(\d+)ELb(\d)E", f.read())
    assert {tuple(int(n) for n in name) for name in names} == reached


def test_the_tests_on_the_gpu_run_every_form(reached):
    lib = ctypes.CDLL(KX_LIB)
    assert all(K % 64 == 0 for K, _, on_lines in FORMS if on_lines)
    assert {form(lib, on_lines, M, K, 16 * blocks - 5) for K, blocks, on_lines in FORMS for M in (3, 16)} == reached


def test_sizes_that_the_kernel_does_not_take():
    lib = ctypes.CDLL(KX_LIB)
    fields = (ctypes.c_int32 * 5)()
    assert not any(lib.kx_bf16_held_form(1, M, K, N, fields) for M, K, N in ((1, 64, 64), (17, 64, 64), (3, 8200, 64), (3, 12, 64), (3, 0, 64), (3, 64, 0)))
