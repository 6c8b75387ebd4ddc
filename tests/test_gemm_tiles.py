"""The few-row GEMM's choice of tile against the measured times of every tile
(profiles/rows_gemm_sweep.json): host code, no GPU needed.

Bound: 15% and 0.5 us over the fastest kernel, where two launches of one kernel
differ by up to 12%.
"""
import ctypes as C
import json
import os

import pytest

import ctbind as cb
from structs import CtGemm

SWEEP = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "profiles", "rows_gemm_sweep.json")
EPI = {"store": 0, "silu": 1, "fmadd": 3, "glu": 4}


@pytest.fixture(scope="module")
def lib():
    L = C.CDLL(cb.HIP_LIB)
    L.ctk_gemm_sizeof.restype = C.c_int
    assert C.sizeof(CtGemm) == L.ctk_gemm_sizeof()
    L.ctk_gemm_tile.argtypes = [C.POINTER(CtGemm), C.c_int]
    L.ctk_gemm_tile.restype = C.c_int
    return L


def gemm(M, N, K, act="fp32", epi="store", **over):
    """A description alone: the addresses are never read."""
    g = CtGemm(lda=K, W=1 << 20, Y=1 << 20, ldy=N, M=M, N=N, K=K, epi=EPI[epi], glu_half=N // 2 if epi == "glu" else 0)
    if act == "fp32":
        g.A = 1 << 20
    else:
        g.Ahi, g.Alo = 1 << 20, 1 << 20 if act == "hilo" else None
    for k, v in over.items():
        setattr(g, k, v)
    return g


def test_choice_is_near_the_fastest(lib):
    rows = json.load(open(SWEEP))["rows"]
    assert len(rows) > 200
    slow = []
    for M, N, K, act, epi, us in rows:
        tile = lib.ctk_gemm_tile(C.byref(gemm(M, N, K, act, epi)), 1)
        mine = us[str(tile)] if tile else min(us[k] for k in ("128", "256") if k in us)
        if mine > 1.15 * min(us.values()) + 0.5:
            slow.append((M, N, K, act, epi, tile, mine, us))
    assert not slow


@pytest.mark.parametrize("act", ["fp32", "hilo", "hi"])
def test_what_the_few_row_kernel_cannot_take(lib, act):
    """An empty sum (its clamped loads would read weights that are not there),
    rows that run backwards or are further apart than 32-bit offsets reach, and
    a K outside its stages go to the general kernels, alone and in a group."""
    def tiles(**over):
        g = gemm(101, 1280, over.pop("K", 1280), act, **over)
        two = (CtGemm * 2)(g, g)
        return lib.ctk_gemm_tile(C.byref(g), 1), lib.ctk_gemm_tile(two, 2)
    alone, grouped = tiles()
    assert alone and bool(grouped) == (act == "fp32")
    for over in ({"K": 0, "lda": 1280}, {"K": 1312}, {"lda": -1280}, {"lda": 1 << 22}):
        assert tiles(**over) == (0, 0), over
