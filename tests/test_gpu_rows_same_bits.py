"""Several activation rows: every launch of a shape adds the K tiles in the same order, whether its workgroups walk over
several blocks of K or not, so that SwiGLU, residual and rotary forms return the bits of the stand-alone kernels around
the plain GEMV.  Shapes whose plain launch walks (a grid of more than 512 workgroups and, at nine rows and more, more
than 16 blocks of 512 rows, at five to eight more than 32) on both sides of what the other forms do."""
import pytest

pytestmark = pytest.mark.gpu

# K, N: 27 and 24 blocks; a last block half past K; runs of three blocks whose last is shorter; 32 blocks and 33, where
# the SwiGLU form walks as well; 34 in whole tiles of heads; 43 blocks in runs of three, 40 in runs of four, over which the
# SwiGLU form at nine rows does not walk
SHAPES = [(13824, 5120), (12288, 8192), (8960, 10240), (10240, 16384), (16384, 4352), (16896, 4352), (17408, 4352),
          (22016, 8192), (20096, 9616)]
ROWS = [5, 8, 9, 16]


def problem(torch, M, K, N, group=128):
    g = torch.Generator(device="cuda")
    g.manual_seed(M + K + N)
    codes = lambda rows: torch.randint(-2**31, 2**31, (rows, N // 8), dtype=torch.int32, device="cuda", generator=g)
    w = codes(K), torch.rand((K // group, N), device="cuda", generator=g).mul_(0.019).add_(0.001).half(), codes(K // group)
    return w, lambda *shape: torch.randn(shape, device="cuda", generator=g).bfloat16()


def empty(torch, *shape):
    return torch.full(shape, float("nan"), dtype=torch.bfloat16, device="cuda")


@pytest.mark.parametrize("K,N", SHAPES)
@pytest.mark.parametrize("M", ROWS)
def test_swiglu_and_residual_forms(M, K, N):
    import torch
    from mykuiperllama_amd import capi
    w, rand = problem(torch, M, K, N)
    gate, up, res = rand(M, K), rand(M, K), rand(M, N)
    act, plain, fused, added = empty(torch, M, K), empty(torch, M, N), empty(torch, M, N), empty(torch, M, N)
    ws = capi.make_workspace(M, K, N)
    capi.swiglu_bf16(gate, up, act)
    capi.gemv_awq_bf16(act, *w, plain, 128, ws)
    capi.gemv_awq_swiglu_bf16(gate, up, *w, fused, 128, ws)
    torch.cuda.synchronize()
    assert torch.equal(plain, fused)
    capi.add_bf16(res, plain, added)
    ssq = torch.empty((M, (N + 255) // 256, 4), dtype=torch.float32, device="cuda")
    for source in ({"in_kind": capi.IN_SWIGLU, "gate": gate, "up": up}, {"in_kind": capi.IN_ROW, "x": act}):
        out = empty(torch, M, N)
        capi.gemv_awq_chain_bf16(dict(source, rows=M, out_kind=capi.OUT_RESIDUAL, residual_in=res, residual_out=out,
                                      sumsq_out=ssq), *w, K, N, 128, ws)
        torch.cuda.synchronize()
        assert torch.equal(out, added)


# two to four rows at the edges of "four steps per wave": sixteen K tiles of two steps and one more; too few workgroups, one
# and two per compute unit and just past either; thirty and thirty-two K tiles of two steps; one more than two batches
@pytest.mark.parametrize("K,N", [(4096, 5120), (4352, 5120), (5120, 1024), (6400, 4864), (6400, 5120), (5120, 13056),
                                 (7680, 5120), (8192, 8448), (8448, 5120)])
@pytest.mark.parametrize("M", [2, 3, 4])
def test_two_to_four_rows(M, K, N):
    import torch
    from mykuiperllama_amd import capi
    w, rand = problem(torch, M, K, N)
    x, res = rand(M, K), rand(M, N)
    plain, out, added = empty(torch, M, N), empty(torch, M, N), empty(torch, M, N)
    ssq = torch.empty((M, (N + 255) // 256, 4), dtype=torch.float32, device="cuda")
    ws = capi.make_workspace(M, K, N)
    capi.gemv_awq_bf16(x, *w, plain, 128, ws)
    capi.add_bf16(res, plain, added)
    capi.gemv_awq_chain_bf16({"in_kind": capi.IN_ROW, "x": x, "rows": M, "out_kind": capi.OUT_RESIDUAL, "residual_in": res,
                              "residual_out": out, "sumsq_out": ssq}, *w, K, N, 128, ws)
    torch.cuda.synchronize()
    assert torch.equal(out, added)
    qw, sc, qz = w
    ref = torch.empty((M, N), dtype=torch.float64, device="cuda")
    for i, col in enumerate((0, 2, 4, 6, 1, 3, 5, 7)):  # nibble i of a word holds column col of its eight
        q, z = ((qw >> (4 * i)) & 15).double(), ((qz >> (4 * i)) & 15).double().repeat_interleave(128, 0)
        ref[:, col::8] = x.double() @ ((q - z) * sc[:, col::8].double().repeat_interleave(128, 0))
    rounded = ref.bfloat16().double()
    assert ((plain.double() - rounded).norm() / rounded.norm()).item() <= 1e-3


# N an odd multiple of eight (one word of a row has no partner): three words in all, groups of 96 and 32, shapes whose plain
# launch walks over two and three blocks; and what stays on the vector kernel: eight columns, many short K tiles
@pytest.mark.parametrize("K,N,group", [(256, 24, 128), (1152, 1000, 96), (5472, 9000, 32), (17408, 4360, 128),
                                       (8704, 22024, 128), (512, 8, 128),
                                       (9216, 520, 32)])
@pytest.mark.parametrize("M", [2, 3] + ROWS)
def test_swiglu_form_of_odd_word_counts(M, K, N, group):
    import torch
    from mykuiperllama_amd import capi
    w, rand = problem(torch, M, K, N, group)
    both = rand(M, 2 * K)
    act, plain, fused = empty(torch, M, K), empty(torch, M, N), empty(torch, M, N)
    ws = capi.make_workspace(M, K, N)
    gate, up = both[:, :K], both[:, K:]
    capi.swiglu_bf16(gate.contiguous(), up.contiguous(), act)
    capi.gemv_awq_bf16(act, *w, plain, group, ws)
    capi.gemv_awq_swiglu_bf16(gate, up, *w, fused, group, ws)
    torch.cuda.synchronize()
    assert torch.equal(plain, fused)


@pytest.mark.parametrize("K,N", [(8704, 8704), (13824, 5120), (16384, 4352), (17408, 4352), (25600, 2816)])
@pytest.mark.parametrize("M", ROWS)
def test_rotary_form(M, K, N):
    import torch
    from mykuiperllama_amd import capi
    w, rand = problem(torch, M, K, N)
    gate, up, q_gain, k_gain = rand(M, K), rand(M, K), rand(128), rand(128)
    act, plain = empty(torch, M, K), empty(torch, M, N)
    n_kv, positions = 1, 4
    n_q = N // 128 - 2
    pos = torch.arange(M, dtype=torch.int32, device="cuda") % positions
    ws = capi.make_workspace(M, K, N)
    outputs = lambda: (empty(torch, M, n_q * 128), torch.zeros((M, positions, n_kv, 128), dtype=torch.bfloat16, device="cuda"),
                       torch.zeros((M, positions, n_kv, 128), dtype=torch.bfloat16, device="cuda"))
    ref = outputs()
    capi.swiglu_bf16(gate, up, act)
    capi.gemv_awq_bf16(act, *w, plain, 128, ws)
    capi.qk_norm_rope_batch_bf16(plain, q_gain, k_gain, *ref, n_q, n_kv, pos, 1e6, 1e-6)
    for source in ({"in_kind": capi.IN_SWIGLU, "gate": gate, "up": up}, {"in_kind": capi.IN_ROW, "x": act}):
        q, kc, vc = outputs()
        capi.gemv_awq_chain_bf16(dict(source, rows=M, out_kind=capi.OUT_QKV_ROPE, q_gain=q_gain, k_gain=k_gain, q_out=q,
                                      k_cache=kc, v_cache=vc, pos=pos, rope_n_q_heads=n_q, rope_n_kv_heads=n_kv,
                                      cache_positions=positions, rope_theta=1e6, qk_eps=1e-6,
                                      cache_stride=positions * n_kv * 128), *w, K, N, 128, ws)
        torch.cuda.synchronize()
        for got, want in zip((q, kc, vc), ref):
            assert torch.equal(got, want)


@pytest.mark.parametrize("K,N", [(4096, 4096), (8704, 8192), (12288, 8192), (16384, 4352), (1152, 23040), (1280, 26112),
                                 (2304, 14592)])  # the last three: a last block mostly idle, 450, 510 and 513 workgroups without it
@pytest.mark.parametrize("M", ROWS)
def test_norm_form_where_the_norm_changes_nothing(M, K, N):
    """Sums of squares that add up to K, no epsilon and gains of one: the normalised row is the row."""
    import torch
    from mykuiperllama_amd import capi
    w, rand = problem(torch, M, K, N)
    row = rand(M, K)
    plain, out = empty(torch, M, N), empty(torch, M, N)
    tiles = (K + 255) // 256
    sums = torch.zeros((M, tiles, 4), dtype=torch.float32, device="cuda")
    sums[:, 0, 0] = K
    ws = capi.make_workspace(M, K, N)
    capi.gemv_awq_bf16(row, *w, plain, 128, ws)
    capi.gemv_awq_chain_bf16({"in_kind": capi.IN_NORM, "norm_row": row, "norm_sumsq": sums, "norm_parts": tiles,
                              "norm_gain": torch.ones(K, dtype=torch.bfloat16, device="cuda"), "norm_eps": 0.0, "rows": M,
                              "out_kind": capi.OUT_ROW, "y": out}, *w, K, N, 128, ws)
    torch.cuda.synchronize()
    assert torch.equal(plain, out)
