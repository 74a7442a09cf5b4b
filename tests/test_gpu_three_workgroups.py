"""Grids of 513 to 768 workgroups of four steps per wave at five and more rows, of which three fit a compute unit in some
forms of nine and more rows: against float64, the same bits in every form of a shape, and when no workgroup waits for the others."""
import pytest

from tests.test_gpu_rows_same_bits import empty, problem

pytestmark = pytest.mark.gpu

# K, N, group: 520 workgroups and the last column tile half empty; waves across groups, which stay at two; an odd number of words; 513; exactly 768 and one too many; ten K
# tiles, the last a quarter full; sixteen; two
SHAPES = [(4096, 16512, 128), (5472, 12304, 32), (5120, 13320, 128), (4608, 14592, 128), (4096, 24576, 128), (2048, 49160, 128), (4736, 15360, 128),
          (8192, 8448, 256), (1024, 65800, 128)]


@pytest.mark.parametrize("K,N,group", SHAPES)
@pytest.mark.parametrize("M", [5, 8, 9, 16])
def test_forms_of_a_shape(M, K, N, group):
    import torch
    from mykuiperllama_amd import capi
    w, rand = problem(torch, M, K, N, group)
    x, res = rand(M, K), rand(M, N)
    plain, unwaited = empty(torch, M, N), empty(torch, M, N)
    ws = capi.make_workspace(M, K, N)
    capi.gemv_awq_bf16(x, *w, plain, group, ws)
    assert capi.load().kx_gemv_awq_bf16_policy(x.data_ptr(), *(t.data_ptr() for t in w), unwaited.data_ptr(), M, K, N, group,
                                               ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream, 3) == 0
    torch.cuda.synchronize()
    assert torch.equal(plain, unwaited)
    if N % 16 == 0:
        tiles = (K + 255) // 256
        sums = torch.zeros((M, tiles, 4), dtype=torch.float32, device="cuda")
        sums[:, 0, 0] = K  # the normalised row is the row
        normed, added, out = empty(torch, M, N), empty(torch, M, N), empty(torch, M, N)
        capi.gemv_awq_chain_bf16({"in_kind": capi.IN_NORM, "norm_row": x, "norm_sumsq": sums, "norm_parts": tiles,
                                  "norm_gain": torch.ones(K, dtype=torch.bfloat16, device="cuda"), "norm_eps": 0.0, "rows": M,
                                  "out_kind": capi.OUT_ROW, "y": normed}, *w, K, N, group, ws)
        capi.add_bf16(res, plain, added)
        ssq = torch.empty((M, (N + 255) // 256, 4), dtype=torch.float32, device="cuda")
        capi.gemv_awq_chain_bf16({"in_kind": capi.IN_ROW, "x": x, "rows": M, "out_kind": capi.OUT_RESIDUAL, "residual_in": res,
                                  "residual_out": out, "sumsq_out": ssq}, *w, K, N, group, ws)
        torch.cuda.synchronize()
        assert torch.equal(plain, normed) and torch.equal(out, added)
    qw, sc, qz = w
    ref = torch.empty((M, N), dtype=torch.float64, device="cuda")
    for i, col in enumerate((0, 2, 4, 6, 1, 3, 5, 7)):  # nibble i of a word holds column col of its eight
        q, z = ((qw >> (4 * i)) & 15).double(), ((qz >> (4 * i)) & 15).double().repeat_interleave(group, 0)
        ref[:, col::8] = x.double() @ ((q - z) * sc[:, col::8].double().repeat_interleave(group, 0))
    rounded = ref.bfloat16().double()
    assert ((plain.double() - rounded).norm() / rounded.norm()).item() <= 1e-3  # as in the tests of other grids: flips of the last bit
