"""Where a decode step merges the chunks of the attention, on both sides of each line."""
import ctypes

import pytest

from mykuiperllama_amd import capi
from mykuiperllama_amd.build import KX_LIB


@pytest.mark.parametrize("hidden,n_q,positions,where", [
    (4096, 32, 1, 1), (4096, 32, 10240, 1), (4096, 32, 10241, -1),   # 256 workgroups
    (5120, 40, 3072, 1), (5120, 40, 3073, 0), (5120, 40, 8192, 0),   # 400: 48 chunks of 40 heads, 64 chunks of 128 positions
    (5120, 32, 3840, 1), (5120, 32, 3841, 0), (5120, 32, 5121, 1), (5120, 32, 7681, 0),  # 320: up to 60 chunks of 32 heads
    (5120, 64, 64, 0), (5120, 64, 10241, -1),                        # 640
    (1024, 1, 100, 1), (64, 2, 100, 1)])
def test_where_the_chunks_are_merged(hidden, n_q, positions, where):
    assert ctypes.CDLL(KX_LIB).kx_step_merges_in_o(hidden, n_q, positions) == where


def test_the_longest_cache_that_a_projection_merges():
    rule = ctypes.CDLL(KX_LIB).kx_step_merges_in_o
    assert rule(4096, 32, capi.FUSED_MERGE_MAX_POSITIONS) >= 0 > rule(4096, 32, capi.FUSED_MERGE_MAX_POSITIONS + 1)
