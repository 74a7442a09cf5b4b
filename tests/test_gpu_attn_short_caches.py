"""Attention over caches that are not full: chunks behind the last position, at every form of the first stage (asking for the
position first or not, chunks of 64 and 128, chunks or heads side by side) and of the merge (chunks covered by its first flight)."""
import pytest

pytestmark = pytest.mark.gpu


def reference(torch, q, k, v, n_q, n_kv, last):
    """Softmax attention of one sequence in float64: [n_q * 128]."""
    k, v = (t[:last + 1].double().repeat_interleave(n_q // n_kv, dim=1) for t in (k, v))  # [positions, n_q, 128]
    w = torch.softmax((k * q.double().view(1, n_q, 128)).sum(-1) / 128 ** 0.5, 0)
    return (w.unsqueeze(-1) * v).sum(0).reshape(-1)


# (query heads, KV heads, cache positions, last positions of the sequences); the merge's first flight covers 32, 48, 80 or 128 chunks
CASES = [(4, 2, 64, [0, 63]), (4, 2, 200, [0, 62, 63, 64, 127, 128, 199]), (6, 2, 2048, [700, 2047]), (6, 2, 2049, [2048, 64]),
         (6, 2, 3072, [3071, 1]), (6, 2, 3073, [3072, 1000]), (8, 1, 5120, [5119, 5]), (4, 4, 4097, [4096, 4095, 127, 128, 255]),
         (16, 1, 130, [129, 127, 128, 0]),
         # many KV heads, whose chunks lie side by side in the grid from 1024 positions on
         (16, 16, 1023, [1022, 5]), (16, 16, 1024, [1023, 0, 64]), (32, 32, 1100, [1099, 63, 64, 700]), (64, 32, 1024, [1000]),
         (32, 32, 5120, [700]), (48, 48, 5121, [5120]),
         (8, 8, 1000, [999]), (8, 8, 32768, [32767]), (8, 8, 32769, [32768]), (8, 8, 32769, [700]), (8, 8, 32769, [0])]


@pytest.mark.parametrize("n_q,n_kv,positions,last", CASES)
def test_chunks_behind_the_context(n_q, n_kv, positions, last):
    torch = pytest.importorskip("torch")
    from mykuiperllama_amd import capi
    batch = len(last)
    g = torch.Generator(device="cuda")
    g.manual_seed(positions + n_q)
    rand = lambda *shape: torch.randn(shape, device="cuda", generator=g).bfloat16()
    q, kc, vc = rand(batch, n_q * 128), rand(batch, positions, n_kv, 128), rand(batch, positions, n_kv, 128)
    for b, p in enumerate(last):  # what lies behind the context may be anything
        kc[b, p + 1:] = float("nan")
        vc[b, p + 1:] = float("inf")
    pos = torch.tensor(last, dtype=torch.int32, device="cuda")
    ws = capi.attn_decode_batch_workspace(batch, n_q, positions)
    ws.fill_(255)  # NaN: nothing that was not written may be used
    out = torch.full((batch, n_q * 128), float("nan"), dtype=torch.bfloat16, device="cuda")
    capi.attn_decode_batch_bf16(q, kc, vc, out, n_q, n_kv, pos, positions, ws)
    one = torch.full_like(out, float("nan"))
    for b in range(batch):
        capi.attn_decode_bf16(q[b], kc[b], vc[b], one[b], n_q, n_kv, pos[b:b + 1], positions, ws)
    torch.cuda.synchronize()
    for b, p in enumerate(last):
        ref = reference(torch, q[b], kc[b], vc[b], n_q, n_kv, p)
        for got in (out[b], one[b]):
            assert (got.double() - ref).norm() <= 2.0 ** -8 * ref.norm(), f"sequence {b}"  # one rounding to bf16: at most 2^-9
    if batch < 4:  # the same chunks for one sequence as for several
        assert torch.equal(out.view(torch.int16), one.view(torch.int16))


def test_no_position_to_attend_to():
    torch = pytest.importorskip("torch")
    from mykuiperllama_amd import capi
    n_q, n_kv, positions = 8, 2, 300
    kc, vc = (torch.full((2, positions, n_kv, 128), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(2))
    q = torch.ones((2, n_q * 128), dtype=torch.bfloat16, device="cuda")
    out = torch.full_like(q, float("nan"))
    ws = capi.attn_decode_batch_workspace(2, n_q, positions)
    ws.fill_(255)
    capi.attn_decode_batch_bf16(q, kc, vc, out, n_q, n_kv, torch.tensor([-1, -1], dtype=torch.int32, device="cuda"), positions, ws)
    torch.cuda.synchronize()
    assert not out.any()


# 32 KV heads at 5120 positions: a first stage that asks for the position and leaves the chunks behind it unwritten
@pytest.mark.parametrize("positions,last,n_q,n_kv", [(64, 63, 4, 2), (300, 5, 4, 2), (2048, 2047, 4, 2), (2049, 2048, 4, 2), (2049, 63, 4, 2),
                                                     (3072, 3071, 4, 2), (3073, 3072, 4, 2), (4096, 4095, 4, 2), (4097, 700, 4, 2),
                                                     (5120, 5119, 4, 2), (6144, 6143, 4, 2), (6145, 6144, 4, 2),
                                                     (5120, 63, 32, 32), (5120, 700, 32, 32), (5120, 5119, 32, 32)])
def test_merge_on_the_way_into_a_projection(positions, last, n_q, n_kv):
    """At the edges of 32, 48 and 64 chunks the projection returns the bits of the merge followed by the projection."""
    torch = pytest.importorskip("torch")
    from mykuiperllama_amd import capi
    N, group = 512, 128
    K = n_q * 128
    g = torch.Generator(device="cuda")
    g.manual_seed(positions)
    rand = lambda *shape: torch.randn(shape, device="cuda", generator=g).bfloat16()
    q, kc, vc = rand(1, K), rand(positions, n_kv, 128), rand(positions, n_kv, 128)
    qw = torch.randint(-2**31, 2**31, (K, N // 8), dtype=torch.int32, device="cuda", generator=g)
    qz = torch.randint(-2**31, 2**31, (K // group, N // 8), dtype=torch.int32, device="cuda", generator=g)
    sc = torch.rand((K // group, N), device="cuda", generator=g).half()
    pos = torch.tensor([last], dtype=torch.int32, device="cuda")
    ws, attn_ws = capi.make_workspace(1, K, N), capi.attn_decode_workspace(n_q, positions)
    attn, residual = torch.empty((1, K), dtype=torch.bfloat16, device="cuda"), rand(1, N)
    capi.attn_decode_bf16(q, kc, vc, attn, n_q, n_kv, pos, positions, attn_ws)
    outs = []
    for inputs in ({"in_kind": capi.IN_ROW, "x": attn},
                   {"in_kind": capi.IN_ATTN, "attn_workspace": attn_ws, "attn_workspace_bytes": attn_ws.numel(),
                    "n_q_heads": n_q, "n_kv_heads": n_kv, "max_positions": positions}):
        if "x" not in inputs:
            attn_ws.fill_(255)
            capi.attn_decode_partial_bf16(q, kc, vc, n_q, n_kv, pos, positions, attn_ws)
        out = torch.full_like(residual, float("nan"))
        sums = torch.empty((N // 256, 4), dtype=torch.float32, device="cuda")
        capi.gemv_awq_chain_bf16({**inputs, "out_kind": capi.OUT_RESIDUAL, "residual_in": residual, "residual_out": out,
                                  "sumsq_out": sums}, qw, sc, qz, K, N, group, ws)
        outs.append((out, sums))
    torch.cuda.synchronize()
    assert torch.isfinite(outs[0][0]).all()
    assert all(torch.equal(a.view(torch.int16), b.view(torch.int16)) for a, b in zip(*outs))
