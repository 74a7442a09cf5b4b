"""Waves across groups whose last block of K is partly past its end: the steps that are not there add nothing, whatever the
scales of the last group are.  An infinite scale makes a column infinite, not NaN."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,N,group", [(6528, 272, 32), (6432, 248, 32), (6528, 272, 96), (16128, 272, 64)])
def test_an_infinite_scale_of_the_last_group(K, N, group):
    import torch
    from mykuiperllama_amd import capi
    for M in (2, 4, 8, 16):
        x = torch.ones((M, K), dtype=torch.bfloat16, device="cuda")
        qw = torch.full((K, N // 8), 0x33333333, dtype=torch.int32, device="cuda")
        qz = torch.full((K // group, N // 8), 0x22222222, dtype=torch.int32, device="cuda")  # every weight is its scale
        sc = torch.full((K // group, N), 2.0 ** -8, dtype=torch.float16, device="cuda")
        sc[-1, 5], sc[-1, 130], sc[0, 7] = float("inf"), float("-inf"), float("inf")
        want = torch.full((M, N), K * 2.0 ** -8, dtype=torch.bfloat16, device="cuda")
        want[:, 5], want[:, 130], want[:, 7] = float("inf"), float("-inf"), float("inf")
        y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
        capi.gemv_awq_bf16(x, qw, sc, qz, y, group, capi.make_workspace(M, K, N))
        torch.cuda.synchronize()
        assert torch.equal(y, want), M
