"""The parity cases of the fragment-order GEMM (test_gpu_t16.py) reach every
tile that its size rule can pick, at every group size, and the row split, on a
device of 256 CUs. Host code only."""
import ctypes

import pytest

import q3vl_int8 as q
import test_gpu_t16 as cases

TILES = {(False, 32): 5, (False, 64): 5, (False, 128): 5, (True, 32): 4, (True, 64): 4, (True, 128): 2}


def plan(M, N, K, gs, swiglu=False, argmax=False):
    f = q.lib()._ZN4q3vl14gemm_t16_tilesEiiiibbiPi
    f.argtypes = [ctypes.c_int] * 4 + [ctypes.c_bool] * 2 + [ctypes.c_int, ctypes.POINTER(ctypes.c_int)]
    f.restype = None
    out = (ctypes.c_int * 3)()
    f(M, N, K, gs, swiglu, argmax, 256, out)
    return tuple(out)


def reached(shapes, gs, swiglu):
    got = set()
    for M, N, K in shapes:
        tile, rows, tile2 = plan(M, N, K, gs, swiglu)
        got.add(tile)
        if rows < M:
            got.add(tile2)
    return got


@pytest.mark.parametrize("gs", [32, 64, 128])
def test_plain_cases_reach_every_tile(gs):
    shapes = [(M, N, K) for M, N in cases.PLAIN for K in cases.plain_ks(N, gs)] + [c for c in cases.PLAIN_K if c[2] % gs == 0]
    assert reached(shapes, gs, False) == set(range(TILES[False, gs]))


@pytest.mark.parametrize("gs", [32, 64, 128])
def test_swiglu_cases_reach_every_tile(gs):
    K = 640 if gs == 128 else 320
    shapes = [(M, N, K) for M, N in cases.SWIGLU] + [(M, I, H) for M, H, I in cases.MLP if H % gs == 0 and I % gs == 0]
    assert reached(shapes, gs, True) == set(range(TILES[True, gs]))


def test_split_cases_split():
    """test_row_split's products are cut in two, with and without a tile of their own for the rest."""
    for gs in (32, 64):
        assert plan(641, 6144, 128, gs, True)[1] == plan(700, 6144, 128, gs, True)[1] == 640
    for gs in (32, 64, 128):
        for M, N, K in cases.SPLIT:
            assert plan(M, N, K, gs)[1] == 2048
