"""BF16 GEMV at several activation rows: lengths of K at the edges of the units and parts it is cut into and of 8192, output
counts at the edges of a block of sixteen and of one block per compute unit, against fp64."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [8, 1016, 1024, 1032, 5120, 6400, 8192, 8200])
@pytest.mark.parametrize("N", [1, 17, 4096, 8209, 40001])
def test_several_rows_match_fp64(K, N):
    import torch
    from mykuiperllama_amd import capi
    gen = torch.Generator(device="cuda")
    gen.manual_seed(K + N)
    w = torch.randn((N, K), device="cuda", generator=gen).bfloat16()
    for M in (2, 3, 8, 16):
        x = torch.randn((M, K), device="cuda", generator=gen).bfloat16()
        y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
        again = torch.full_like(y, float("nan"))
        capi.gemv_bf16(x, w, y)
        capi.gemv_bf16(x, w, again)
        ref = (x.double() @ w.double().t().contiguous()).to(torch.bfloat16).double()
        torch.cuda.synchronize()
        assert torch.equal(y.view(torch.int16), again.view(torch.int16))
        assert ((y.double() - ref).norm() / ref.norm()).item() <= 1e-3, (M, K, N)
