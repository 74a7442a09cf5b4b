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


# rows, steps per wave, N, K tiles -> whether the grid keeps the order of its numbers
@pytest.mark.parametrize("M,steps,N,ktiles,by_number", [
    # half lines, groups of eight column tiles: up to 256 workgroups, by K tiles for the rows
    (16, 4, 1920, 32, 1), (16, 4, 1920, 33, 0), (11, 4, 1920, 26, 1), (11, 4, 1920, 29, 0), (8, 2, 3968, 12, 1), (5, 2, 3968, 17, 0), (7, 2, 1920, 20, 1),
    (7, 2, 1920, 25, 0), (8, 2, 8064, 7, 1), (5, 2, 8064, 9, 0),
    # other even groups: one and two steps
    (10, 2, 2944, 16, 1), (10, 4, 2944, 16, 0), (11, 2, 1408, 22, 1), (11, 2, 1408, 23, 0), (7, 2, 1408, 22, 0), (10, 2, 13696, 8, 0),
    # odd groups, and rows on quarters of lines
    (11, 2, 1664, 13, 0), (8, 2, 3904, 17, 0),
    # as before: eight and more by rows and workgroups, two and four by K tiles
    (16, 2, 8128, 9, 1), (16, 4, 4056, 12, 1), (16, 4, 8168, 8, 0), (6, 1, 264, 12, 1), (6, 1, 264, 16, 0)])
def test_which_grids_that_finish_together_keep_their_numbers(M, steps, N, ktiles, by_number):
    assert ctypes.CDLL(KX_LIB).kx_tiles_by_number(M, steps, N, -(-N // 256), ktiles, 1) == by_number


@pytest.mark.parametrize("M,steps,coltiles,ktiles,by_number", [
    # nine and more rows: a grid just past two workgroups per compute unit, or runs that begin on the same columns
    (16, 4, 12, 44, 1), (9, 4, 16, 34, 1), (9, 4, 16, 32, 0), (10, 4, 57, 9, 1), (10, 4, 55, 10, 0), (10, 4, 19, 32, 1), (10, 4, 19, 33, 0), (16, 4, 31, 48, 1),
    (16, 4, 32, 24, 1), (16, 4, 33, 24, 0), (16, 2, 19, 32, 0),
    # five to eight: many K tiles and a little more than two per compute unit
    (8, 4, 12, 48, 1), (5, 4, 15, 36, 1), (8, 4, 16, 40, 0), (8, 4, 19, 32, 0), (8, 4, 14, 42, 0),
    (4, 4, 12, 48, 0)])
def test_which_grids_with_one_reader_keep_their_numbers(M, steps, coltiles, ktiles, by_number):
    assert ctypes.CDLL(KX_LIB).kx_tiles_by_number(M, steps, 256 * coltiles - 128, coltiles, ktiles, 0) == by_number
