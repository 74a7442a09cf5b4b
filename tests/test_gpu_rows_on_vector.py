"""Several rows that stay on the vector kernel (an odd number of words, groups that leave a wave of the matrix-core kernel one
step, long and narrow or two rows): its sums, bit for bit, whose rounding error is the smaller one, and the same behind SwiGLU."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,N,group,rows", [(12288, 1288, 32, (2, 3, 4, 5, 8, 16)), (9216, 520, 32, (2, 4, 8, 9, 16)),
                                            (9216, 2040, 96, (3, 4, 16)), (8224, 24, 32, (2, 3, 4, 16)), (2080, 3000, 32, (2,))])
def test_sums_are_those_of_the_vector_kernel(K, N, group, rows):
    import torch
    from mykuiperllama_amd import capi
    gen = torch.Generator(device="cuda")
    gen.manual_seed(K + N)
    codes = lambda r: torch.randint(-2**31, 2**31, (r, N // 8), dtype=torch.int32, device="cuda", generator=gen)
    w = codes(K), torch.rand((K // group, N), device="cuda", generator=gen).mul_(0.019).add_(0.001).half(), codes(K // group)
    for M in rows:
        gate, up = (torch.randn((M, K), device="cuda", generator=gen).bfloat16() for _ in range(2))
        act, plain, vector, fused = torch.empty_like(gate), *(torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
                                                              for _ in range(3))
        ws = capi.make_workspace(M, K, N)
        capi.swiglu_bf16(gate, up, act)
        capi.gemv_awq_bf16(act, *w, plain, group, ws)
        capi.gemv_awq_swiglu_bf16(gate, up, *w, fused, group, ws)
        capi.set_awq_kernel_policy(1)
        try:
            capi.gemv_awq_bf16(act, *w, vector, group, ws)
        finally:
            capi.set_awq_kernel_policy(0)
        torch.cuda.synchronize()
        assert torch.equal(plain, vector), M
        assert torch.equal(fused, vector), M
