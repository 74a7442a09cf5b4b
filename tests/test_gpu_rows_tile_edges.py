"""The matrix-core GEMV of several rows at the edges of a column tile: where the sums of the waves and the partial sums of the
K tiles are laid out by word halves (whole tiles) or by columns (a narrower last one), for every row count that is packed
differently, against the CPU oracle."""
import numpy as np
import pytest

from mykuiperllama_amd import synth
from tests import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,group", [(1056, 96), (1024, 128)])
@pytest.mark.parametrize("N", [16, 120, 248, 256, 264, 520, 1016])
@pytest.mark.parametrize("M", [2, 3, 4, 7, 8, 9, 13, 16])
def test_tile_edges_match_the_oracle(oracle, M, N, K, group):
    import torch
    from mykuiperllama_amd import capi
    p = synth.make_awq_problem(f"edges_{K}x{N}", M, K, N, group)
    x, qw = H.to_dev_bf16(p["x"], torch), H.to_dev_i32(p["qweight"], torch)
    sc, qz = H.to_dev_f16(p["scales"], torch), H.to_dev_i32(p["qzeros"], torch)
    y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    capi.gemv_awq_bf16(x, qw, sc, qz, y, group, capi.make_workspace(M, K, N))
    torch.cuda.synchronize()
    ref = oracle.gemv_awq_f64(p["x"], p["qweight"], p["scales"], p["qzeros"], group)
    rounded = H.bf16_to_f64(oracle.f32_to_bf16(ref.astype(np.float32)))
    # a bf16 output whose fp32 sum falls next to a rounding boundary may flip: 2^-8 of its value in at most a few per cent
    assert H.rel_l2(H.bf16_to_f64(H.bf16_bits(y, torch)), rounded) <= 1e-3
