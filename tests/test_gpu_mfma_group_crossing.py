"""The matrix-core GEMV whose waves take four 32-row steps across quantisation groups (groups that are no multiple of 128 and
many K tiles otherwise), for every row count that is laid out differently, with a last block of K that is partly past its
end, with whole and odd numbers of words in the last column tile, against the CPU oracle."""
import numpy as np
import pytest

from mykuiperllama_amd import synth
from tests import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,group", [(6432, 32), (6432, 96), (6560, 160), (16000, 64), (15552, 192)])
@pytest.mark.parametrize("N", [248, 272])
def test_waves_across_groups_match_the_oracle(oracle, N, K, group):
    import torch
    from mykuiperllama_amd import capi
    p = synth.make_awq_problem(f"cross_{K}x{N}x{group}", 16, K, N, group)
    ref = oracle.gemv_awq_f64(p["x"], p["qweight"], p["scales"], p["qzeros"], group)
    rounded = H.bf16_to_f64(oracle.f32_to_bf16(ref.astype(np.float32)))
    qw, sc, qz = H.to_dev_i32(p["qweight"], torch), H.to_dev_f16(p["scales"], torch), H.to_dev_i32(p["qzeros"], torch)
    for M in (2, 3, 4, 6, 8, 9, 16):
        x = H.to_dev_bf16(np.ascontiguousarray(p["x"][:M]), torch)
        y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
        capi.gemv_awq_bf16(x, qw, sc, qz, y, group, capi.make_workspace(M, K, N))
        torch.cuda.synchronize()
        # a bf16 output whose fp32 sum falls next to a rounding boundary may flip: 2^-8 of its value in at most a few per cent
        assert H.rel_l2(H.bf16_to_f64(H.bf16_bits(y, torch)), rounded[:M]) <= 1e-3, M
        # the form that produces its activations, and the same sums: bit for bit
        both, act = torch.randn((M, 2 * K), device="cuda").bfloat16(), torch.empty((M, K), dtype=torch.bfloat16, device="cuda")
        fused, gate, up = torch.empty_like(y), both[:, :K], both[:, K:]
        capi.swiglu_bf16(gate.contiguous(), up.contiguous(), act)
        capi.gemv_awq_bf16(act, qw, sc, qz, y, group, capi.make_workspace(M, K, N))
        capi.gemv_awq_swiglu_bf16(gate, up, qw, sc, qz, fused, group, capi.make_workspace(M, K, N))
        torch.cuda.synchronize()
        assert torch.equal(y, fused), M
