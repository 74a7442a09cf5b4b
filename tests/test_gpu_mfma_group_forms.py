"""Waves across quantisation groups in every form of a launch: the norm in front, the residual add and the rotation behind, one
reader of many workgroups' sums, and a single row on the matrix cores.  Each against the stand-alone operators around the plain
launch, bit for bit, and the plain launch against float64."""
import pytest

pytestmark = pytest.mark.gpu

# twelve and a half K tiles that finish together; three column tiles, the last a narrow one; more than 512 workgroups at
# eleven K tiles, whose sums one workgroup of a tile reads; groups of 96, which a wave's steps do not divide
SHAPES = [(6400, 512, 32), (16000, 768, 64), (5472, 12304, 32), (6432, 528, 96)]
ROWS = [2, 4, 5, 8, 9, 16]


def problem(torch, M, K, N, group):
    g = torch.Generator(device="cuda")
    g.manual_seed(M + K + N)
    codes = lambda rows: torch.randint(-2**31, 2**31, (rows, N // 8), dtype=torch.int32, device="cuda", generator=g)
    w = codes(K), torch.rand((K // group, N), device="cuda", generator=g).mul_(0.019).add_(0.001).half(), codes(K // group)
    return w, lambda *shape: torch.randn(shape, device="cuda", generator=g).bfloat16()


def empty(torch, *shape):
    return torch.full(shape, float("nan"), dtype=torch.bfloat16, device="cuda")


def rounded_sum(torch, x, w, N, group):
    qw, sc, qz = w
    ref = torch.empty((x.shape[0], N), dtype=torch.float64, device="cuda")
    for i, col in enumerate((0, 2, 4, 6, 1, 3, 5, 7)):  # nibble i of a word holds column col of its eight
        q, z = ((qw >> (4 * i)) & 15).double(), ((qz >> (4 * i)) & 15).double().repeat_interleave(group, 0)
        ref[:, col::8] = x.double() @ ((q - z) * sc[:, col::8].double().repeat_interleave(group, 0))
    return ref.bfloat16().double()


def rel(a, b):
    return ((a.double() - b).norm() / b.norm()).item()


@pytest.mark.parametrize("K,N,group", SHAPES)
@pytest.mark.parametrize("M", ROWS)
def test_store_norm_and_residual_forms(M, K, N, group):
    import torch
    from mykuiperllama_amd import capi
    w, rand = problem(torch, M, K, N, group)
    x, gate, up, res = rand(M, K), rand(M, K), rand(M, K), rand(M, N)
    plain, normed, act, behind = empty(torch, M, N), empty(torch, M, N), empty(torch, M, K), empty(torch, M, N)
    ws = capi.make_workspace(M, K, N)
    capi.gemv_awq_bf16(x, *w, plain, group, ws)
    # a bf16 output whose fp32 sum falls next to a rounding boundary may flip: 2^-8 of its value in at most a few per cent
    assert rel(plain, rounded_sum(torch, x, w, N, group)) <= 1e-3

    # sums of squares that add up to K, no epsilon and gains of one: the normalised row is the row
    tiles = (K + 255) // 256
    sums = torch.zeros((M, tiles, 4), dtype=torch.float32, device="cuda")
    sums[:, 0, 0] = K
    norm = {"in_kind": capi.IN_NORM, "norm_row": x, "norm_sumsq": sums, "norm_parts": tiles, "norm_eps": 0.0,
            "norm_gain": torch.ones(K, dtype=torch.bfloat16, device="cuda")}
    capi.gemv_awq_chain_bf16(dict(norm, rows=M, out_kind=capi.OUT_ROW, y=normed), *w, K, N, group, ws)
    torch.cuda.synchronize()
    assert torch.equal(plain, normed)

    capi.swiglu_bf16(gate, up, act)
    capi.gemv_awq_bf16(act, *w, behind, group, ws)
    for source, product in ((norm, plain), ({"in_kind": capi.IN_ROW, "x": x}, plain),
                            ({"in_kind": capi.IN_SWIGLU, "gate": gate, "up": up}, behind)):
        out, added = empty(torch, M, N), empty(torch, M, N)
        ssq = torch.full((M, (N + 255) // 256, 4), float("nan"), dtype=torch.float32, device="cuda")
        capi.add_bf16(res, product, added)
        capi.gemv_awq_chain_bf16(dict(source, rows=M, out_kind=capi.OUT_RESIDUAL, residual_in=res, residual_out=out,
                                      sumsq_out=ssq), *w, K, N, group, ws)
        torch.cuda.synchronize()
        assert torch.equal(out, added)
        # fp32 sums of 64 squares each: 64 roundings of 2^-24 at most
        assert rel(ssq.sum((1, 2)), added.double().pow(2).sum(1)) <= 1e-5


@pytest.mark.parametrize("K,N,group", [(6400, 512, 32), (16000, 768, 64), (5472, 12544, 32)])
@pytest.mark.parametrize("M", ROWS)
def test_rotary_forms(M, K, N, group):
    import torch
    from mykuiperllama_amd import capi
    w, rand = problem(torch, M, K, N, group)
    x, gate, up, q_gain, k_gain = rand(M, K), rand(M, K), rand(M, K), rand(128), rand(128)
    n_kv, positions = 1, 4
    n_q = N // 128 - 2
    pos = torch.arange(M, dtype=torch.int32, device="cuda") % positions
    ws = capi.make_workspace(M, K, N)
    outputs = lambda: (empty(torch, M, n_q * 128), torch.zeros((M, positions, n_kv, 128), dtype=torch.bfloat16, device="cuda"),
                       torch.zeros((M, positions, n_kv, 128), dtype=torch.bfloat16, device="cuda"))
    act, product = empty(torch, M, K), empty(torch, M, N)
    capi.swiglu_bf16(gate, up, act)
    tiles = (K + 255) // 256
    sums = torch.zeros((M, tiles, 4), dtype=torch.float32, device="cuda")
    sums[:, 0, 0] = K
    for row, source in ((x, {"in_kind": capi.IN_NORM, "norm_row": x, "norm_sumsq": sums, "norm_parts": tiles, "norm_eps": 0.0,
                             "norm_gain": torch.ones(K, dtype=torch.bfloat16, device="cuda")}),
                        (x, {"in_kind": capi.IN_ROW, "x": x}), (act, {"in_kind": capi.IN_SWIGLU, "gate": gate, "up": up})):
        want, got = outputs(), outputs()
        capi.gemv_awq_bf16(row, *w, product, group, ws)
        capi.qk_norm_rope_batch_bf16(product, q_gain, k_gain, *want, n_q, n_kv, pos, 1e6, 1e-6)
        capi.gemv_awq_chain_bf16(dict(source, rows=M, out_kind=capi.OUT_QKV_ROPE, q_gain=q_gain, k_gain=k_gain, q_out=got[0],
                                      k_cache=got[1], v_cache=got[2], pos=pos, rope_n_q_heads=n_q, rope_n_kv_heads=n_kv,
                                      cache_positions=positions, rope_theta=1e6, qk_eps=1e-6,
                                      cache_stride=positions * n_kv * 128), *w, K, N, group, ws)
        torch.cuda.synchronize()
        for a, b in zip(got, want):
            assert torch.equal(a, b)


@pytest.mark.parametrize("K,N,group", [(6432, 272, 32), (6432, 248, 96), (16000, 520, 64)])
def test_one_row_on_the_matrix_cores(K, N, group):
    import torch
    from mykuiperllama_amd import capi
    w, rand = problem(torch, 1, K, N, group)
    x, y = rand(1, K), empty(torch, 1, N)
    capi.set_awq_kernel_policy(2)
    try:
        capi.gemv_awq_bf16(x, *w, y, group, capi.make_workspace(1, K, N))
    finally:
        capi.set_awq_kernel_policy(0)
    torch.cuda.synchronize()
    assert rel(y, rounded_sum(torch, x, w, N, group)) <= 1e-3
