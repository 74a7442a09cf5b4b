"""Attention over long caches: the merge at the edges of its first flights (128 chunks of 128 positions, 320, 512) and of the
rule that takes a head in quarters (more chunks, the more heads there are)."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("max_pos", [16384, 16385, 40960, 40961, 65536])
@pytest.mark.parametrize("batch", [1, 2])
def test_long_merge_against_float64(max_pos, batch):
    torch = pytest.importorskip("torch")
    from mykuiperllama_amd import capi
    n_q, n_kv = 6, 2
    g = torch.Generator(device="cuda")
    g.manual_seed(max_pos + batch)
    rand = lambda *shape: torch.randn(shape, device="cuda", generator=g).bfloat16()
    q, kc, vc = rand(batch, n_q * 128), rand(batch, max_pos, n_kv, 128), rand(batch, max_pos, n_kv, 128)
    out = torch.full((batch, n_q * 128), float("nan"), dtype=torch.bfloat16, device="cuda")
    last = [max_pos - 1, max_pos // 3][:batch]  # a full cache, and one with empty chunks at the end
    pos = torch.tensor(last, dtype=torch.int32, device="cuda")
    ws = capi.attn_decode_batch_workspace(batch, n_q, max_pos)
    ws.fill_(255)  # NaN: nothing that was not written may be used
    capi.attn_decode_batch_bf16(q, kc, vc, out, n_q, n_kv, pos, max_pos, ws)
    torch.cuda.synchronize()
    for b, p in enumerate(last):
        for h in range(n_q):
            k, v = kc[b, :p + 1, h // 3].cpu().double(), vc[b, :p + 1, h // 3].cpu().double()
            w = torch.softmax(k @ q[b, 128 * h:128 * h + 128].cpu().double() / 128 ** 0.5, 0)
            ref = w @ v
            err = (out[b, 128 * h:128 * h + 128].cpu().double() - ref).norm() / ref.norm()
            assert err <= 2.0 ** -8, f"sequence {b}, head {h}"  # one rounding to bf16 is at most 2^-9 per element


@pytest.mark.parametrize("n_q,n_kv,batch,chunks", [(6, 2, 1, 160), (6, 2, 1, 161), (64, 4, 1, 161), (65, 5, 1, 192), (65, 5, 1, 193),
                                                   (32, 2, 8, 256), (32, 2, 8, 257), (32, 2, 9, 257)])
def test_merge_forms_against_float64(n_q, n_kv, batch, chunks):
    torch = pytest.importorskip("torch")
    from mykuiperllama_amd import capi
    positions = 128 * chunks - 5
    g = torch.Generator(device="cuda")
    g.manual_seed(chunks + n_q)
    rand = lambda *shape: torch.randn(shape, device="cuda", generator=g).bfloat16()
    q, kc, vc = rand(batch, n_q * 128), rand(batch, positions, n_kv, 128), rand(batch, positions, n_kv, 128)
    out = torch.full((batch, n_q * 128), float("nan"), dtype=torch.bfloat16, device="cuda")
    last = [positions - 1 - 1000 * b for b in range(batch)]
    ws = capi.attn_decode_batch_workspace(batch, n_q, positions)
    ws.fill_(255)  # NaN: nothing that was not written may be used
    capi.attn_decode_batch_bf16(q, kc, vc, out, n_q, n_kv, torch.tensor(last, dtype=torch.int32, device="cuda"), positions, ws)
    torch.cuda.synchronize()
    assert torch.isfinite(out).all()
    for b, h in ((0, 0), (0, n_q - 1), (batch - 1, n_q // 2)):
        k, v = kc[b, :last[b] + 1, h * n_kv // n_q].cpu().double(), vc[b, :last[b] + 1, h * n_kv // n_q].cpu().double()
        ref = torch.softmax(k @ q[b, 128 * h:128 * h + 128].cpu().double() / 128 ** 0.5, 0) @ v
        err = (out[b, 128 * h:128 * h + 128].cpu().double() - ref).norm() / ref.norm()
        assert err <= 2.0 ** -8, f"sequence {b}, head {h}"  # one rounding to bf16 is at most 2^-9 per element
