"""BF16 GEMV of several rows: K at the edges of the units that a wave takes (128 elements where rows start on memory lines, 128,
256 or 512 elsewhere) and of the number of waves that split it, outputs at the edges of runs of four blocks and of a round of 256, against
float64."""
import pytest

pytestmark = pytest.mark.gpu


def check(torch, capi, w, K, N, Ms):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(K * 31 + N)
    for M in Ms:
        x = torch.randn((M, K), device="cuda", generator=gen).bfloat16()
        y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
        capi.gemv_bf16(x, w, y)
        ref = (x.double() @ w.double().t().contiguous()).to(torch.bfloat16).double()
        torch.cuda.synchronize()
        # fp32 sums of bf16 products, rounded once: they differ from the rounded reference by flips of the last bit alone
        assert ((y.double() - ref).norm() / ref.norm()).item() <= 1e-3, (M, K, N)


@pytest.mark.parametrize("K", [16, 64, 128, 192, 504, 520, 896, 1032, 1088, 1536, 1544, 2048, 2056, 4032, 4088, 4104, 6144, 6152, 8184])
@pytest.mark.parametrize("N", [4099, 16399])
def test_units_and_parts(K, N):
    import torch
    from mykuiperllama_amd import capi
    w = torch.randn((N, K), device="cuda").bfloat16()
    check(torch, capi, w, K, N, (2, 3, 6, 16))


@pytest.mark.parametrize("K", [520, 1024])
@pytest.mark.parametrize("blocks", [255, 257, 1023, 1024, 1025, 1027, 2051, 2309])
def test_rounds_and_runs(K, blocks):
    import torch
    from mykuiperllama_amd import capi
    N = 16 * blocks - 5
    w = torch.randn((N, K), device="cuda").bfloat16()
    check(torch, capi, w, K, N, (3, 7))


@pytest.mark.parametrize("K,blocks", [(200, 5119), (200, 5120), (1016, 5121), (4360, 1024), (4360, 1025)])
def test_edges_of_the_forms_off_lines(K, blocks):
    import torch
    from mykuiperllama_amd import capi
    N = 16 * blocks - 7
    w = torch.randn((N, K), device="cuda").bfloat16()
    check(torch, capi, w, K, N, (3, 16))


# every form of the kernel (test_bf16_held_forms.py holds this list to it): K, blocks, and whether W starts on a memory line.
# Eight, four and two of eight waves to a block, one to eight units each, one by one and in runs, the last block beside nothing;
# off lines all of eight waves, four, two and one of four
FORMS = ([(K, 300, True) for K in (64, 1088, 2048, 2112, 3072, 3136, 5120, 5184, 7168, 8128, 8192)] +
         [(K, 2600, True) for K in (2112, 3136, 5056, 6144)] + [(1024, 2601, True)] +
         [(K, 1301, True) for K in (64, 512, 704, 1024, 1088, 1472, 2048, 2112, 2560)] +
         [(K, 2401, True) for K in (64, 512, 576, 1024, 1088, 1472, 2112, 2560)] + [(K, 3850, True) for K in (2624, 3520, 4096)] +
         [(K, 1803, True) for K in (64, 256, 448, 704, 768, 1024, 1088, 1280)] +
         [(K, 2825, True) for K in (64, 320, 576, 768, 832, 1024, 1088, 1280)] + [(768, 1999, True), (768, 2000, True)] +
         [(K, 300, False) for K in (64, 1216, 2816, 4096, 5056, 6400)] + [(K, 2401, False) for K in (1032, 2056, 2816)] +
         [(4608, 1025, False), (6080, 1029, False), (904, 5120, False), (200, 5120, False), (904, 7499, False), (904, 7500, False), (896, 7500, False),
          (1024, 5121, False)])


@pytest.mark.parametrize("K,blocks,on_lines", FORMS)
def test_every_form(K, blocks, on_lines):
    import torch
    from mykuiperllama_amd import capi
    N, shift = 16 * blocks - 5, 0 if on_lines else 8
    flat = torch.randn(N * K + shift, device="cuda").bfloat16()
    check(torch, capi, flat[shift:].view(N, K), K, N, (3, 16))


def test_weights_off_a_line():
    import torch
    from mykuiperllama_amd import capi
    K, N = 1024, 17000
    flat = torch.randn(N * K + 64, device="cuda").bfloat16()
    check(torch, capi, flat[8:8 + N * K].view(N, K), K, N, (3, 16))


@pytest.mark.parametrize("K", [136, 520, 1000, 1032, 2056, 4104, 8184])
def test_what_lies_past_a_row_takes_no_part(K):
    """The last unit of a row is read past K's end within W: an infinity there meets no zero."""
    import torch
    from mykuiperllama_amd import capi
    N, M = 40, 5
    w = torch.ones((N, K), device="cuda").bfloat16()
    w[7, K - 1] = float("inf")
    x = torch.ones((M, K), device="cuda").bfloat16()
    y = torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
    capi.gemv_bf16(x, w, y)
    torch.cuda.synchronize()
    assert torch.isinf(y[:, 7]).all() and torch.isfinite(y[:, :7]).all() and torch.isfinite(y[:, 8:]).all()
