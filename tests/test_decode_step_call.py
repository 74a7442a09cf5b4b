"""The decode step in one native call: what it refuses before anything is launched (no GPU needed), and that the binding's
structures have the sizes the library was compiled with."""
import array
import ctypes

import pytest


@pytest.fixture(scope="module")
def capi():
    from mykuiperllama_amd import capi
    capi.load()
    return capi


def test_null_pointers_are_refused(capi):
    step = capi.load().kx_decode_step_bf16
    assert step(None, None, None) == -1
    empty = capi.StepDesc(layers=1, hidden=256)
    assert step(ctypes.addressof(empty), None, None) == -1  # a layer count without layers
    layers = array.array("q", [0] * capi.STEP_LAYER_WORDS)
    assert step(ctypes.addressof(empty), layers.buffer_info()[0], None) == -1  # the embedding table is missing


def test_structures_match_the_header(capi):
    # thirteen pointers, two workspaces with their sizes, twelve 32-bit integers, two floats
    assert ctypes.sizeof(capi.StepDesc) == 17 * 8 + 14 * 4
    assert capi.STEP_LAYER_WORDS == 4 * 3 + 4 + 2 + 1
