"""The decode step in one native call: what it refuses before anything is launched (no GPU needed), and that the binding's
structures have the sizes the library was compiled with."""
import array
import ctypes
import os
import re

import pytest


@pytest.fixture(scope="module")
def capi():
    from mykuiperllama_amd import capi
    capi.load()
    return capi


def test_null_pointers_are_refused(capi):
    step = capi.load().kx_decode_step_bf16
    assert step(None, None, None) == -1
    empty = capi.StepDesc(layers=1, hidden=256)
    assert step(ctypes.addressof(empty), None, None) == -1  # a layer count without layers
    layers = array.array("q", [0] * capi.STEP_LAYER_WORDS)
    assert step(ctypes.addressof(empty), layers.buffer_info()[0], None) == -1  # the embedding table is missing


def test_structures_match_the_header(capi):
    # thirteen pointers, two workspaces with their sizes, twelve 32-bit integers, two floats
    assert ctypes.sizeof(capi.StepDesc) == 17 * 8 + 14 * 4
    assert capi.STEP_LAYER_WORDS == 4 * 3 + 4 + 2 + 1


def test_structures_match_the_library(capi):
    lib = capi.load()
    assert ctypes.sizeof(capi.StepDesc) == lib.kx_step_desc_bytes()
    assert 8 * capi.STEP_LAYER_WORDS == lib.kx_step_layer_bytes()
    # the fields in the order, and of the kind, in which the header declares them
    with open(os.path.join(os.path.dirname(capi.__file__), "csrc", "kx_internal.h")) as f:
        body = re.search(r"typedef struct kx_step_desc \{(.*?)\} kx_step_desc;", f.read(), re.S).group(1)
    kinds = {"float": ctypes.c_float, "int32_t": ctypes.c_int32, "size_t": ctypes.c_size_t}
    declared = []
    for kind, names in re.findall(r"(?:const )?(\w+)([^;]*);", re.sub(r"/\*.*?\*/", "", body)):
        declared += [(name.strip(" *"), ctypes.c_void_p if "*" in name else kinds[kind]) for name in names.split(",")]
    assert declared == list(capi.StepDesc._fields_)


def stubbed_model(monkeypatch, **changes):
    """A two-layer model on the CPU whose native call only records what it was given."""
    import torch
    from mykuiperllama_amd import capi, decode
    cfg = decode.ModelConfig(layers=2, hidden=256, intermediate=512, n_q=2, n_kv=1, vocab=64)
    row = lambda n=1: torch.zeros((1, n), dtype=torch.bfloat16)
    matrix = lambda: tuple(torch.zeros(4) for _ in range(3))
    model = decode.DecodeModel.__new__(decode.DecodeModel)
    model.__dict__.update(
        torch=torch, cfg=cfg, max_positions=8, merge_in_o=True,
        layers=[dict({m: matrix() for m in ("qkv", "o", "gateup", "down")},
                     **{n: row() for n in ("in_norm", "post_norm", "q_norm", "k_norm")}) for _ in range(2)],
        embed=row(256), lm_head=torch.zeros((64, 256)), final_norm=row(256), logits=row(64), ssq=torch.zeros((1, 4)),
        k_cache=[torch.zeros((8, 1, 128)) for _ in range(2)], v_cache=[torch.zeros((8, 1, 128)) for _ in range(2)],
        **{n: row() for n in ("x", "h", "q", "attn", "gu", "token", "pos", "next_token", "gemv_ws", "attn_ws")})
    model.__dict__.update(changes)
    calls = []
    monkeypatch.setattr(capi, "decode_step_bf16", lambda fields, words: calls.append((fields, words)))
    return model, calls


def test_a_step_without_the_head_needs_no_lm_head(monkeypatch):
    model, calls = stubbed_model(monkeypatch, lm_head=None)
    model.step(with_lm_head=False)
    (fields, _), = calls
    assert fields.get("lm_head") is None
    with pytest.raises(AttributeError):  # with the head it is asked for its shape, and nothing is launched
        model.step(with_lm_head=True)
    assert len(calls) == 1


@pytest.mark.parametrize("caches", ["k_cache", "v_cache"])
def test_a_missing_cache_is_refused(monkeypatch, caches):
    import torch
    model, calls = stubbed_model(monkeypatch, **{caches: [torch.zeros((8, 1, 128))]})  # of two layers
    with pytest.raises(IndexError):
        model.step()
    assert not calls


def test_caches_are_taken_by_layer(monkeypatch):
    import torch
    model, calls = stubbed_model(monkeypatch)
    model.step()
    by_number = {1: model.k_cache[1], 0: model.k_cache[0], 2: torch.zeros((8, 1, 128))}  # more caches than layers, in any order
    model.k_cache = by_number
    model.step()
    assert calls[0][1] == calls[1][1] and len(calls[0][1]) == 2 * 19


@pytest.mark.parametrize("matrix", ["qkv", "o", "gateup", "down"])
@pytest.mark.parametrize("parts", [2, 4])
def test_a_matrix_has_three_parts(monkeypatch, matrix, parts):
    import torch
    model, calls = stubbed_model(monkeypatch)
    model.layers[0][matrix] = tuple(torch.zeros(4) for _ in range(parts))
    with pytest.raises(ValueError):  # anything else would move every address behind it
        model.step()
    assert not calls
