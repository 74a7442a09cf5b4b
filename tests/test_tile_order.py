"""Workgroups of a grid whose column tiles share memory lines: every tile is taken once, neighbours on one XCD."""
import ctypes

import pytest

from mykuiperllama_amd.build import KX_LIB

COLTILES = [1, 2, 3, 7, 8, 15, 31, 32, 33, 36, 64, 65, 80, 95, 201, 1024]
KTILES = [1, 2, 3, 5, 8, 9, 31, 62, 200]


def tiles(lib, coltiles, ktiles):
    ct, kt = ctypes.c_int32(), ctypes.c_int32()
    out = []
    for i in range(coltiles * ktiles):
        if not lib.kx_shared_line_tile(coltiles, ktiles, i, ctypes.byref(ct), ctypes.byref(kt)):
            return None
        out.append((ct.value, kt.value))
    return out


@pytest.mark.parametrize("coltiles", COLTILES)
def test_every_tile_is_taken_once(coltiles):
    lib = ctypes.CDLL(KX_LIB)
    for ktiles in KTILES:
        got = tiles(lib, coltiles, ktiles)
        if coltiles < 2 or coltiles * ktiles < 16:
            assert got is None
            continue
        assert sorted(got) == [(c, k) for c in range(coltiles) for k in range(ktiles)], (coltiles, ktiles)
        # neighbours in a K tile lie on one XCD (workgroup i on XCD i % 8), but for the runs' and the groups' borders
        xcd = {tile: i % 8 for i, tile in enumerate(got)}
        apart = sum(xcd[c, k] != xcd[c + 1, k] for c in range(coltiles - 1) for k in range(ktiles))
        groups = -(-coltiles // 32)
        assert apart <= 7 * groups + (groups - 1) * ktiles, (coltiles, ktiles, apart)


def test_grids_past_the_reach_of_the_divisions_keep_their_numbers():
    assert not ctypes.CDLL(KX_LIB).kx_shared_line_tile(2048, 2000, 5, ctypes.byref(ctypes.c_int32()), ctypes.byref(ctypes.c_int32()))
