"""The matrix-core GEMV at five and more rows where a workgroup walks over several blocks of K (long K, many column
tiles): against float64, with and without waiting for the others, and behind a SwiGLU prologue and a residual epilogue."""
import pytest

pytestmark = pytest.mark.gpu

# K, N: two blocks each; a last workgroup with one block of four; the last block partly past K and an odd word count;
# seventeen blocks (the fewest that walk at nine rows and more) and one fewer; thirty-three (at five to eight) and one fewer
SHAPES = [(25600, 2816), (8704, 22016), (16512, 7432), (8704, 8192), (8192, 8448), (16896, 4352), (16384, 4352)]


def rand(torch, shape, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.randn(shape, device="cuda", generator=g).bfloat16()


def weights(torch, K, N):
    g = torch.Generator(device="cuda")
    g.manual_seed(K + N)
    codes = lambda rows: torch.randint(-2**31, 2**31, (rows, N // 8), dtype=torch.int32, device="cuda", generator=g)
    return codes(K), torch.rand((K // 128, N), device="cuda", generator=g).mul_(0.019).add_(0.001).half(), codes(K // 128)


@pytest.mark.parametrize("K,N", SHAPES)
@pytest.mark.parametrize("M", [5, 8, 9, 16])
def test_walk_matches_float64(K, N, M):
    import torch
    from mykuiperllama_amd import capi
    x, (qw, sc, qz) = rand(torch, (M, K), M), weights(torch, K, N)
    ws = capi.make_workspace(M, K, N)
    results = []
    for policy in (0, 3, 0):  # by shape; the same kernel without waiting; and once more on the same workspace
        y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
        assert capi.load().kx_gemv_awq_bf16_policy(
            x.data_ptr(), qw.data_ptr(), sc.data_ptr(), qz.data_ptr(), y.data_ptr(), M, K, N, 128, ws.data_ptr(),
            ws.numel(), torch.cuda.current_stream().cuda_stream, policy) == 0
        torch.cuda.synchronize()
        results.append(y)
    assert torch.equal(results[0], results[1]) and torch.equal(results[0], results[2])
    # the weights in double from their definition: nibble i of a word holds column order[i]
    ref = torch.zeros((M, N), dtype=torch.float64, device="cuda")
    order = (0, 2, 4, 6, 1, 3, 5, 7)
    for i, col in enumerate(order):
        q = ((qw >> (4 * i)) & 15).double()
        z = ((qz >> (4 * i)) & 15).double().repeat_interleave(128, 0)
        w = (q - z) * sc[:, col::8].double().repeat_interleave(128, 0)
        ref[:, col::8] = x.double() @ w
    got, rounded = results[0].double(), ref.bfloat16().double()
    assert ((got - rounded).norm() / rounded.norm()).item() <= 1e-3


@pytest.mark.parametrize("K,N,M", [(25600, 2816, 5), (25600, 2816, 16), (16896, 4352, 8), (16896, 4352, 16)])
def test_walk_behind_swiglu_and_into_the_residual_stream(K, N, M):
    import torch
    from mykuiperllama_amd import capi
    gate, up, res, (qw, sc, qz) = rand(torch, (M, K), 1), rand(torch, (M, K), 2), rand(torch, (M, N), 3), weights(torch, K, N)
    ws = capi.make_workspace(M, K, N)
    act, plain, fused, out = (torch.empty((M, n), dtype=torch.bfloat16, device="cuda") for n in (K, N, N, N))
    capi.swiglu_bf16(gate, up, act)
    capi.gemv_awq_bf16(act, qw, sc, qz, plain, 128, ws)
    capi.gemv_awq_swiglu_bf16(gate, up, qw, sc, qz, fused, 128, ws)
    ssq = torch.empty((M, (N + 255) // 256, 4), dtype=torch.float32, device="cuda")
    capi.gemv_awq_chain_bf16({"in_kind": capi.IN_SWIGLU, "gate": gate, "up": up, "act_ld": K, "rows": M,
                              "out_kind": capi.OUT_RESIDUAL, "residual_in": res, "residual_out": out, "sumsq_out": ssq},
                             qw, sc, qz, K, N, 128, ws)
    torch.cuda.synchronize()
    assert torch.equal(plain, fused)
    expect = (res.float() + plain.float()).bfloat16()
    assert torch.equal(out, expect)
    total = expect.double().square().sum(1)
    assert ((ssq.double().sum((1, 2)) - total).abs() / total).max().item() <= 1e-5  # fp32 sums of squares
