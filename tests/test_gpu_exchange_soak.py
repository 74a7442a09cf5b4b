"""Many split-K launches back to back on ONE workspace, cycling the seven Qwen3-8B projection shapes: every
output must equal, bit for bit, what the same shape returned the first time.

The split-K exchange orders its partial sums before the arrival counter by waiting for the stores'
acknowledgement, not by a release/acquire pair (an acquire-release counter update costs 3 to 27 us per launch
on this machine: it writes back and invalidates whole caches).  That is a contract with the hardware rather
than with the language's memory model, so it is watched: a stale partial sum or a counter left non-zero by
one launch shows up here as a changed bit in a later one.  The run stops at the first mismatch.
"""
import pytest

from mykuiperllama_amd import synth

pytestmark = pytest.mark.gpu

LAUNCHES = 2000
CHUNK = 100  # launches between comparisons


@pytest.mark.parametrize("policy", [0, 1, 2], ids=["by_shape", "vector_ordered", "mfma"])
def test_two_thousand_launches_on_one_workspace_repeat_their_first_results(policy):
    import torch
    from mykuiperllama_amd import capi
    capi.load()
    assert torch.cuda.is_available()
    names = ["q_proj", "k_proj", "v_proj", "o_proj", "gate_proj", "up_proj", "down_proj"]
    shapes = [synth.QWEN3_8B[n] for n in names]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(synth.BASE_SEED + 5)
    probs = []
    for K, N in shapes:
        qw = torch.randint(-2**31, 2**31 - 1, (K, N // 8), dtype=torch.int32, device="cuda", generator=gen)
        qz = torch.randint(-2**31, 2**31 - 1, (K // 128, N // 8), dtype=torch.int32, device="cuda", generator=gen)
        sc = (torch.rand((K // 128, N), device="cuda", generator=gen) * 0.019 + 0.001).half()
        x = torch.randn((1, K), device="cuda", generator=gen).bfloat16()
        probs.append((x, qw, sc, qz, N))
    ws = capi.make_workspace(1, max(k for k, _ in shapes), max(n for _, n in shapes))  # one workspace for all
    capi.set_awq_kernel_policy(policy)
    try:
        first = []
        for x, qw, sc, qz, N in probs:
            y = torch.empty((1, N), dtype=torch.bfloat16, device="cuda")
            capi.gemv_awq_bf16(x, qw, sc, qz, y, 128, ws)
            first.append(y)
        torch.cuda.synchronize()
        outs = [[torch.empty((1, N), dtype=torch.bfloat16, device="cuda") for _ in range(CHUNK // len(probs) + 1)]
                for (_, _, _, _, N) in probs]
        done = 0
        while done < LAUNCHES:
            used = [0] * len(probs)
            batch = []
            for i in range(done, min(done + CHUNK, LAUNCHES)):
                s = i % len(probs)
                x, qw, sc, qz, _ = probs[s]
                y = outs[s][used[s]]
                used[s] += 1
                capi.gemv_awq_bf16(x, qw, sc, qz, y, 128, ws)  # no synchronisation in between
                batch.append((i, s, y))
            torch.cuda.synchronize()
            for i, s, y in batch:
                assert torch.equal(y.view(torch.int16), first[s].view(torch.int16)), \
                    f"launch {i} ({names[s]}) differs from the first {names[s]} launch"
            done += len(batch)
    finally:
        capi.set_awq_kernel_policy(0)


def test_chained_launches_on_one_workspace_repeat_their_first_results():
    """The same watch over the exchanges of the fused epilogues: the o and down projections with the residual
    output (every wave of 64 columns finishes for itself) and the q|k|v projection with the rotary output (the two
    waves of a head share a counter), 1 400 launches cycling over the three on one workspace together with plain
    launches of the same shapes, which index the counter area differently."""
    import torch
    from mykuiperllama_amd import capi
    capi.load()
    gen = torch.Generator(device="cuda")
    gen.manual_seed(synth.BASE_SEED + 6)
    H, I, n_q, n_kv, max_pos, pos_value = 4096, 12288, 32, 8, 64, 17

    def weights(K, N):
        qw = torch.randint(-2**31, 2**31 - 1, (K, N // 8), dtype=torch.int32, device="cuda", generator=gen)
        qz = torch.randint(-2**31, 2**31 - 1, (K // 128, N // 8), dtype=torch.int32, device="cuda", generator=gen)
        sc = (torch.rand((K // 128, N), device="cuda", generator=gen) * 0.019 + 0.001).half()
        return qw, sc, qz

    def bf16(shape, scale=1.0):
        return (torch.randn(shape, device="cuda", generator=gen) * scale).bfloat16()

    w_o, w_down, w_qkv = weights(H, H), weights(I, H), weights(H, (n_q + 2 * n_kv) * 128)
    x_o, gate, up, x_qkv, resid = bf16((1, H)), bf16((1, I)), bf16((1, I)), bf16((1, H)), bf16((1, H), 2.0)
    q_gain, k_gain = 1 + bf16((128,), 0.1), 1 + bf16((128,), 0.1)
    pos = torch.tensor([pos_value], dtype=torch.int32, device="cuda")
    ws = capi.make_workspace(1, I, (n_q + 2 * n_kv) * 128)

    def run_residual(kind, out, sumsq):
        if kind == "o":
            capi.gemv_awq_chain_bf16({"in_kind": capi.IN_ROW, "x": x_o, "out_kind": capi.OUT_RESIDUAL,
                                      "residual_in": resid, "residual_out": out, "sumsq_out": sumsq},
                                     *w_o, H, H, 128, ws)
        else:
            capi.gemv_awq_chain_bf16({"in_kind": capi.IN_SWIGLU, "gate": gate, "up": up,
                                      "out_kind": capi.OUT_RESIDUAL, "residual_in": resid, "residual_out": out,
                                      "sumsq_out": sumsq}, *w_down, I, H, 128, ws)

    def run_rope(q_out, kc, vc):
        capi.gemv_awq_chain_bf16({"in_kind": capi.IN_ROW, "x": x_qkv, "out_kind": capi.OUT_QKV_ROPE,
                                  "q_gain": q_gain, "k_gain": k_gain, "q_out": q_out, "k_cache": kc, "v_cache": vc,
                                  "pos": pos, "rope_n_q_heads": n_q, "rope_n_kv_heads": n_kv, "rope_theta": 1e6,
                                  "qk_eps": 1e-6}, *w_qkv, H, (n_q + 2 * n_kv) * 128, 128, ws)

    def fresh():
        return {"o": (torch.empty((1, H), dtype=torch.bfloat16, device="cuda"),
                      torch.empty((H // 256, 4), dtype=torch.float32, device="cuda")),
                "down": (torch.empty((1, H), dtype=torch.bfloat16, device="cuda"),
                         torch.empty((H // 256, 4), dtype=torch.float32, device="cuda")),
                "rope": (torch.empty((1, n_q * 128), dtype=torch.bfloat16, device="cuda"),
                         torch.zeros((max_pos, n_kv, 128), dtype=torch.bfloat16, device="cuda"),
                         torch.zeros((max_pos, n_kv, 128), dtype=torch.bfloat16, device="cuda")),
                "plain": (torch.empty((1, H), dtype=torch.bfloat16, device="cuda"),)}

    def launch(kind, bufs):
        if kind in ("o", "down"):
            run_residual(kind, *bufs[kind])
        elif kind == "rope":
            run_rope(*bufs["rope"])
        else:
            capi.gemv_awq_bf16(x_o, *w_o, bufs["plain"][0], 128, ws)

    order = ["o", "rope", "plain", "down"]
    first = fresh()
    for kind in order:
        launch(kind, first)
    torch.cuda.synchronize()
    rounds, per_round = 14, 25   # 14 x 25 x 4 = 1 400 launches
    for r in range(rounds):
        sets = [fresh() for _ in range(per_round)]
        for bufs in sets:
            for kind in order:
                launch(kind, bufs)       # no synchronisation in between
        torch.cuda.synchronize()
        for i, bufs in enumerate(sets):
            for kind in order:
                for got, ref in zip(bufs[kind], first[kind]):
                    same = torch.equal(got.view(torch.int32) if got.dtype == torch.float32 else got.view(torch.int16),
                                       ref.view(torch.int32) if ref.dtype == torch.float32 else ref.view(torch.int16))
                    assert same, f"round {r}, set {i}: a {kind} launch differs from the first one"


def _rows_problem(torch, gen, M, K, N):
    codes = lambda rows: torch.randint(-2**31, 2**31, (rows, N // 8), dtype=torch.int32, device="cuda", generator=gen)
    w = codes(K), (torch.rand((K // 128, N), device="cuda", generator=gen) * 0.019 + 0.001).half(), codes(K // 128)
    return w, torch.randn((M, K), device="cuda", generator=gen).bfloat16()


@pytest.mark.parametrize("M", [2, 3, 8, 16])
def test_several_row_launches_on_one_workspace_repeat_their_first_results(M):
    """Two and more rows: counters per wave, per workgroup and, from five rows on, arrivals, departures and masks of column
    tiles that are finished together, all in the same area of one workspace.  About a thousand launches cycle over
    shapes that finish together with few and with many K tiles, that have one reader, and that walk over blocks of K;
    over the residual, rotary and norm forms; and over launches whose workgroups do not wait for each other."""
    import torch
    from mykuiperllama_amd import capi
    lib = capi.load()
    gen = torch.Generator(device="cuda")
    gen.manual_seed(synth.BASE_SEED + 20 + M)
    H, n_q, n_kv, positions = 4096, 32, 8, 32
    wide = (n_q + 2 * n_kv) * 128
    shapes = {"narrow": (H, 1024), "square": (H, H), "long": (12288, H), "wide": (H, 24576), "walk": (8704, 8192),
              "longest": (25600, 2816), "qkv": (H, wide)}
    probs = {name: _rows_problem(torch, gen, M, K, N) for name, (K, N) in shapes.items()}
    ws = capi.make_workspace(M, 25600, 24576)
    resid = torch.randn((M, H), device="cuda", generator=gen).bfloat16()
    gains = [1 + 0.1 * torch.randn((n,), device="cuda", generator=gen) for n in (128, 128, H)]
    q_gain, k_gain, norm_gain = (g.bfloat16() for g in gains)
    pos = torch.arange(M, dtype=torch.int32, device="cuda") + 3
    sums = torch.rand((M, H // 256, 4), device="cuda", generator=gen) * 64 + 1

    def bf16(*shape):
        return torch.zeros(shape, dtype=torch.bfloat16, device="cuda")

    def plain(name, policy):
        (K, N), (w, x) = shapes[name], probs[name]
        y = bf16(M, N)
        assert lib.kx_gemv_awq_bf16_policy(x.data_ptr(), *(t.data_ptr() for t in w), y.data_ptr(), M, K, N, 128,
                                           ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream, policy) == 0
        return (y,)

    def residual(name):
        (K, N), (w, x) = shapes[name], probs[name]
        out, ssq = bf16(M, N), torch.zeros((M, N // 256, 4), dtype=torch.float32, device="cuda")
        capi.gemv_awq_chain_bf16({"in_kind": capi.IN_ROW, "x": x, "rows": M, "out_kind": capi.OUT_RESIDUAL,
                                  "residual_in": resid, "residual_out": out, "sumsq_out": ssq}, *w, K, N, 128, ws)
        return out, ssq

    def rotary():
        w, x = probs["qkv"]
        q, kc, vc = bf16(M, n_q * 128), bf16(M, positions, n_kv, 128), bf16(M, positions, n_kv, 128)
        capi.gemv_awq_chain_bf16({"in_kind": capi.IN_ROW, "x": x, "rows": M, "out_kind": capi.OUT_QKV_ROPE, "q_gain": q_gain,
                                  "k_gain": k_gain, "q_out": q, "k_cache": kc, "v_cache": vc, "pos": pos,
                                  "rope_n_q_heads": n_q, "rope_n_kv_heads": n_kv, "cache_positions": positions,
                                  "rope_theta": 1e6, "qk_eps": 1e-6, "cache_stride": positions * n_kv * 128}, *w, H, wide, 128, ws)
        return q, kc, vc

    def norm():
        w, x = probs["wide"]
        y = bf16(M, shapes["wide"][1])
        capi.gemv_awq_chain_bf16({"in_kind": capi.IN_NORM, "norm_row": x, "norm_sumsq": sums, "norm_parts": H // 256,
                                  "norm_gain": norm_gain, "norm_eps": 1e-6, "rows": M, "out_kind": capi.OUT_ROW, "y": y},
                                 *w, H, shapes["wide"][1], 128, ws)
        return (y,)

    launches = [lambda n=n, p=p: plain(n, p) for p in (0, 3) for n in ("narrow", "square", "long", "wide", "walk", "longest")]
    launches += [lambda: residual("square"), lambda: residual("long"), rotary, norm]
    first = [launch() for launch in launches]
    torch.cuda.synchronize()
    for r in range(16):
        sets = [[launch() for launch in launches] for _ in range(4)]  # no synchronisation in between
        torch.cuda.synchronize()
        for got in sets:
            for i, (a, b) in enumerate(zip(got, first)):
                assert all(torch.equal(x, y) for x, y in zip(a, b)), f"round {r}: launch {i} differs from its first result"
    for i in range(6):  # waiting or not, the same sums
        assert torch.equal(first[i][0], first[i + 6][0])


@pytest.mark.parametrize("M", [5, 16])
def test_two_streams_with_a_workspace_each(M):
    """Grids that fill the chip on two streams at once, so that workgroups hold the places their neighbours need: the wait of
    the shared finishing is bounded for this, whoever gives up hands its share on, and every launch still returns its bits."""
    import torch
    from mykuiperllama_amd import capi
    gen = torch.Generator(device="cuda")
    gen.manual_seed(synth.BASE_SEED + 40 + M)
    shapes = [(4096, 16384), (25600, 2816), (12288, 4096), (1024, 2048)]  # 512 and 550 workgroups (walking), 384, small ones
    probs = [_rows_problem(torch, gen, M, K, N) for K, N in shapes]
    spaces = [capi.make_workspace(M, 25600, 16384) for _ in range(2)]

    def launch(i, ws):
        (w, x), y = probs[i], torch.zeros((M, shapes[i][1]), dtype=torch.bfloat16, device="cuda")
        capi.gemv_awq_bf16(x, *w, y, 128, ws)
        return y

    first = [launch(i, spaces[0]) for i in range(len(shapes))]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in spaces]
    for r in range(12):
        got = [[], []]
        for j in range(12):
            for s, stream in enumerate(streams):
                with torch.cuda.stream(stream):
                    i = (j + s * (r % 4)) % len(shapes)  # the same shapes side by side, and different ones
                    got[s].append((i, launch(i, spaces[s])))
        torch.cuda.synchronize()
        for s in range(2):
            for i, y in got[s]:
                assert torch.equal(y, first[i]), f"round {r}, stream {s}: {shapes[i]} differs"
