"""The matrix-core GEMV at five and more rows, whose workgroups finish a column tile together (each a share of its rows)
where they fit on the chip: shapes at the edges of that rule, odd word counts and group sizes that are no power of two,
against the CPU oracle; and the same bits when no workgroup is willing to wait for the others."""
import numpy as np
import pytest

from mykuiperllama_amd import synth
from tests import helpers as H

pytestmark = pytest.mark.gpu

# K, N, group: one K tile; two column tiles; tiles whose number has no divisor near eight; an odd number of words and
# groups of 96; more K tiles than slices; the largest grid that still shares (512 workgroups); one workgroup too many
SHAPES = [(128, 256, 128), (1024, 512, 64), (1024, 2816, 128), (1152, 1000, 96), (8192, 256, 32), (4096, 16384, 128),
          (4096, 16640, 128)]


@pytest.mark.parametrize("K,N,group", SHAPES)
@pytest.mark.parametrize("M", [5, 8, 9, 16])
def test_rows_finished_together_match_the_oracle(oracle, K, N, group, M):
    import torch
    from mykuiperllama_amd import capi
    p = synth.make_awq_problem(f"slices_{K}x{N}", M, K, N, group)
    x, qw = H.to_dev_bf16(p["x"], torch), H.to_dev_i32(p["qweight"], torch)
    sc, qz = H.to_dev_f16(p["scales"], torch), H.to_dev_i32(p["qzeros"], torch)
    ws = capi.make_workspace(M, K, N)
    results = []
    for policy in (0, 3, 0):  # by shape; the same kernel without waiting; and once more on the same workspace
        y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
        assert capi.load().kx_gemv_awq_bf16_policy(
            x.data_ptr(), qw.data_ptr(), sc.data_ptr(), qz.data_ptr(), y.data_ptr(), M, K, N, group, ws.data_ptr(),
            ws.numel(), torch.cuda.current_stream().cuda_stream, policy) == 0
        torch.cuda.synchronize()
        results.append(H.bf16_bits(y, torch))
    assert np.array_equal(results[0], results[1]) and np.array_equal(results[0], results[2])
    ref = oracle.gemv_awq_f64(p["x"], p["qweight"], p["scales"], p["qzeros"], group)
    rounded = H.bf16_to_f64(oracle.f32_to_bf16(ref.astype(np.float32)))
    assert H.rel_l2(H.bf16_to_f64(results[0]), rounded) <= 1e-3
