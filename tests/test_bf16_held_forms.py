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
            for blocks in BLOCKS for M in (4, 5, 6, 16)}


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


# (on lines, rows, K, N) -> waves to a block, and runs of four blocks
@pytest.mark.parametrize("on_lines,M,K,N,parts,runs", [
    (1, 16, 3072, 32768, 8, 0), (1, 8, 4096, 24000, 8, 0), (1, 3, 4096, 151936, 4, 0), (1, 5, 4096, 151936, 8, 1), (1, 16, 2560, 32768, 4, 0),
    (1, 16, 1536, 32768, 4, 0), (1, 16, 1280, 32768, 2, 0), (1, 8, 6144, 24000, 8, 0), (1, 16, 6144, 40000, 8, 1), (1, 8, 6144, 151936, 8, 1),
    (1, 16, 2048, 16384, 8, 1), (1, 5, 2048, 16384, 8, 0), (0, 8, 3592, 32768, 8, 0), (0, 16, 3592, 65000, 8, 1), (0, 8, 5000, 32768, 4, 1)])
def test_form_of_a_size(on_lines, M, K, N, parts, runs):
    assert form(ctypes.CDLL(KX_LIB), on_lines, M, K, N)[3:] == (parts, runs)


@pytest.mark.parametrize("K,N,taken", [(4096, 8192, 1), (4096, 8383, 0), (5000, 9000, 0), (5000, 11177, 1), (3072, 12400, 0), (768, 8192, 1), (768, 8383, 0),
                                       (768, 16500, 0), (768, 24000, 1), (1000, 40000, 0), (4096, 6400, 0), (8200, 40000, 0)])
def test_two_rows(K, N, taken):
    assert ctypes.CDLL(KX_LIB).kx_bf16_held_form(0, 2, K, N, (ctypes.c_int32 * 5)()) == taken
