"""Packed rows whose 128-byte pieces do not start on a memory line: column tiles taken in another order, the same sums."""
import numpy as np
import pytest

from mykuiperllama_amd import synth
from tests import helpers as H

pytestmark = pytest.mark.gpu


def run(torch, capi, M, K, N, group, shift):
    p = synth.make_awq_problem(f"order_{M}_{K}_{N}", M, K, N, group)
    words = torch.zeros(K * N // 8 + 64, dtype=torch.int32, device="cuda")
    qw = words[shift:shift + K * N // 8].view(K, N // 8)
    qw.copy_(H.to_dev_i32(p["qweight"], torch))
    y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    capi.gemv_awq_bf16(H.to_dev_bf16(p["x"], torch), qw, H.to_dev_f16(p["scales"], torch), H.to_dev_i32(p["qzeros"], torch), y,
                       group, capi.make_workspace(M, K, N))
    torch.cuda.synchronize()
    return p, H.bf16_bits(y, torch)


# one column short of, at and past groups of 32 column tiles, with one and several K tiles; fewer tiles than it takes
@pytest.mark.parametrize("M", [1, 2, 5, 16])
@pytest.mark.parametrize("K,N,group", [(512, 31 * 256 - 8, 128), (512, 32 * 256 + 128, 32), (640, 33 * 256 + 16, 64), (2048, 1048, 32),
                                       (1024, 264, 128)])
def test_against_the_oracle(oracle, M, K, N, group):
    import torch
    from mykuiperllama_amd import capi
    p, bits = run(torch, capi, M, K, N, group, 0)
    ref = oracle.gemv_awq_f64(p["x"], p["qweight"], p["scales"], p["qzeros"], group)
    ref = H.bf16_to_f64(oracle.f32_to_bf16(ref.astype(np.float32)))
    assert H.rel_l2(H.bf16_to_f64(bits), ref) <= 1e-3


# grids that finish together, on both sides of the rule that keeps the order of the numbers: eight column tiles and more with one,
# two and four steps and with 12 M workgroups and more, two and four with K tiles that do and do not divide by eight, four,
# six, twelve and sixteen whose rows start on half lines
@pytest.mark.parametrize("M,K,N", [(16, 4096, 24 * 256), (16, 4608, 24 * 256), (16, 1024, 8 * 256), (9, 4096, 16 * 256), (8, 4096, 16 * 256),
                                   (5, 1024, 24 * 256), (6, 6144, 512), (6, 4096, 512), (12, 2304, 1024), (12, 2048, 1024), (16, 8192, 8 * 256),
                                   (6, 2048, 896), (6, 12288, 896), (9, 12288, 896), (6, 6144, 896), (15, 7680, 3968), (7, 3328, 3968),
                                   (5, 4352, 3968), (10, 3968, 2944), (7, 5632, 1408)])
def test_few_workgroups_that_finish_together(M, K, N):
    import torch
    from mykuiperllama_amd import capi
    on, off = (run(torch, capi, M, K, N, 128, shift)[1] for shift in (0, 1))
    assert np.array_equal(on, off)


# grids of more than two workgroups per compute unit, which one workgroup reads back, on both sides of that rule (steps across groups)
@pytest.mark.parametrize("M,K,N", [(9, 22528, 12 * 256), (9, 23552, 12 * 256), (8, 24576, 12 * 256), (8, 16384, 17 * 256), (10, 16384, 17 * 256)])
def test_grids_with_one_reader(M, K, N):
    import torch
    from mykuiperllama_amd import capi
    on, off = (run(torch, capi, M, K, N, 64, shift)[1] for shift in (0, 1))
    assert np.array_equal(on, off)


@pytest.mark.parametrize("M", [1, 3, 9])
def test_weights_off_a_line_return_the_same_bits(M):
    import torch
    from mykuiperllama_amd import capi
    on = run(torch, capi, M, 1024, 33 * 256, 128, 0)[1]
    off = run(torch, capi, M, 1024, 33 * 256, 128, 1)[1]
    assert np.array_equal(on, off)
