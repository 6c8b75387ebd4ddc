"""GPU checks of the few-row encoder GEMM (ctk_gemm's 16- to 128-row tiles):
every tile gives the bits of the many-row kernels (the same chain of MFMAs per
element), whatever the rows, columns and depth leave over at the tile's and the
ring's edges, and writes nothing outside the rows and columns of the launch.

The many-row kernels themselves are held to float64 by test_gpu_split_gemm.py.
ctk_gemm_tile confirms that the forced tile, or the group launch, is what runs.
Shapes: rows from 1 past each tile's edge, columns that end inside a tile (a
multiple of neither 16 nor 8 among them), K from one stage (128) over an odd
number of stages (384, 640) to one longer than the ring.
"""
import ctypes as C

import numpy as np
import pytest

import ctbind as cb
from structs import CtGemm, CtSeg
from test_gpu_gemv import Dev, f32_to_bf16, split

pytestmark = pytest.mark.gpu

EPI_STORE, EPI_SILU, EPI_RELU, EPI_FMADD, EPI_GLU = 0, 1, 2, 3, 4
OUT_SPLIT = 3
TILES = [16016, 16032, 32032, 32064, 64128, 48128, 96128, 128128]
ABSENT = {"fp32": (48128, 96128, 128128), "hi": (48128,), "hilo": ()}     # no such form
MANY_ROWS = 128              # forces the many-row kernels


@pytest.fixture(scope="module")
def lib(hip):
    L = C.CDLL(cb.HIP_LIB)
    L.ctk_gemm_sizeof.restype = C.c_int
    assert C.sizeof(CtGemm) == L.ctk_gemm_sizeof()
    L.ctk_gemm.argtypes = [C.POINTER(CtGemm), C.c_void_p]
    L.ctk_gemm_force_tile.argtypes = [C.c_int]
    L.ctk_gemm_tile.argtypes = [C.POINTER(CtGemm), C.c_int]
    L.ctk_gemm_tile.restype = C.c_int
    yield L
    L.ctk_gemm_force_tile(0)


# rows, columns (GLU: of the output), K, epilogue
SHAPES = [
    (1, 48, 128, EPI_STORE), (15, 1000, 256, EPI_RELU), (17, 44, 384, EPI_FMADD), (33, 136, 640, EPI_SILU),
    (65, 200, 1280, EPI_FMADD), (101, 1280, 1280, "split"), (64, 72, 384, EPI_GLU), (100, 640, 1280, EPI_GLU),
    (13, 1280, 5120, EPI_FMADD), (97, 264, 384, EPI_RELU), (129, 136, 256, EPI_GLU),
]


@pytest.mark.parametrize("act", ["fp32", "hilo", "hi"])
@pytest.mark.parametrize("M,N,K,epi", SHAPES, ids=[f"{m}x{n}x{k}-{e}" for m, n, k, e in SHAPES])
def test_tiles_give_the_many_row_kernels_bits(lib, hip, act, M, N, K, epi):
    dev = Dev(hip)
    rng = np.random.default_rng(M * N + K)
    glu = epi == EPI_GLU
    wrows, lda = (2 * N if glu else N), K + 8
    x = np.zeros((M, lda), np.float32)
    x[:, :K] = rng.standard_normal((M, K))
    hi, lo = split(x)
    pA, pH, pL = dev.put(x), dev.put(hi), dev.put(lo)
    pW = dev.put(f32_to_bf16(rng.standard_normal((wrows, K)).astype(np.float32) / np.sqrt(K).astype(np.float32)))
    pb = dev.put(f32_to_bf16(rng.standard_normal(wrows).astype(np.float32)))
    ldy, guard = N + 8, 3                       # columns and rows past the launch's keep their fill
    y0 = rng.standard_normal((M + guard, ldy)).astype(np.float32)
    pY, pY2 = dev.put(y0), dev.put(y0)

    def run(tile):
        g = CtGemm(lda=lda, W=pW, bias=pb if M != 33 else None, M=M, N=wrows, K=K, scale=0.5, Y=pY, ldy=ldy)
        if act == "fp32":
            g.A = pA
        else:
            g.Ahi, g.Alo = pH, pL if act == "hilo" else None
        if epi == "split":
            g.epi, g.nseg, g.seg_w = EPI_SILU, 1, N
            g.seg[0] = CtSeg(mode=OUT_SPLIT, base=pY, ld=ldy, base_lo=pY2)
        else:
            g.epi = epi
            g.glu_half = N if glu else 0
        for p in (pY, pY2):
            hip.backend_htod(p, y0.ctypes.data, y0.size)
        dev.ev.sync()
        lib.ctk_gemm_force_tile(tile)
        assert tile == 0 or lib.ctk_gemm_tile(C.byref(g), 1) == (0 if tile == MANY_ROWS else tile)
        lib.ctk_gemm(C.byref(g), None)
        return [dev.get(p, np.uint32, y0.size).reshape(y0.shape) for p in (pY, pY2)]

    want = run(MANY_ROWS)
    for tile in TILES:
        if tile in ABSENT[act] or (glu and tile in (16016, 32032)):
            continue                            # no GLU form: an odd number of column blocks per wave
        print(f"case: {act} {M}x{N}x{K} epi {epi} tile {tile}", flush=True)
        got = run(tile)
        for a, b in zip(want, got):
            assert np.array_equal(a, b), tile
    if epi != "split":
        assert np.array_equal(want[0][M:], y0[M:].view(np.uint32))
        assert np.array_equal(want[0][:, N:], y0[:, N:].view(np.uint32))
    for a, b in zip(want, run(0)):              # the tile the cost model takes
        assert np.array_equal(a, b)


# name: (columns, segment width, K, segments' modes, epilogue); the widths end
# inside tiles of 32 columns and more, on tiles' edges (640), and hold whole heads
OUTPUTS = {
    "three dense": (1920, 640, 256, "ddd", EPI_STORE),
    "dense, straddled": (600, 200, 256, "ddd", EPI_STORE),
    "split with relu": (400, 200, 384, "ss", EPI_RELU),
    "split without lo": (320, 320, 256, "h", EPI_SILU),
    "split and dense": (400, 200, 256, "sd", EPI_SILU),
    "heads fp32": (768, 384, 256, "ff", EPI_STORE),
    "heads bf16": (512, 256, 256, "bb", EPI_STORE),
    "masked residual": (200, 0, 256, "m", EPI_FMADD),
    "masked": (200, 0, 256, "m", EPI_SILU),
    "scattered rows": (200, 0, 256, "r", EPI_STORE),
    "scattered residual": (200, 0, 256, "r", EPI_FMADD),
}
HSTRIDE = 128 * 128


@pytest.mark.parametrize("act", ["fp32", "hilo", "hi"])
@pytest.mark.parametrize("name", OUTPUTS)
def test_every_output_of_every_tile(lib, hip, name, act):
    """All the places a row can go: the few-row epilogue's own and, where a tile
    straddles segments or rows are skipped or scattered, the shared one."""
    N, seg_w, K, modes, epi = OUTPUTS[name]
    dev, M = Dev(hip), 131                      # one row past a 128-row tile's and two 64-row tiles' edge
    rng = np.random.default_rng(N + K)
    x = rng.standard_normal((M, K)).astype(np.float32)
    hi, lo = split(x)
    pA, pH, pL = dev.put(x), dev.put(hi), dev.put(lo)
    pW = dev.put(f32_to_bf16(rng.standard_normal((N, K)).astype(np.float32) / np.float32(np.sqrt(K))))
    pb = dev.put(f32_to_bf16(rng.standard_normal(N).astype(np.float32)))
    m = np.arange(M)
    offs = np.where(m % 7 == 3, -1, (m % 128) * 128 + m // 128 * 6 * HSTRIDE).astype(np.int64)      # 6 heads at most
    mask, lens = (m % 5 != 2).astype(np.int32), np.where(m % 6 == 4, 0, m % 3 + 1).astype(np.int32)
    po, pm, pn = dev.put(offs), dev.put(mask), dev.put(lens)
    plane = max(12 * HSTRIDE, 3 * M * max(N, 1))                # floats: rows of three to scatter, two blocks of heads
    y0 = rng.standard_normal(plane).astype(np.float32)
    outs = [dev.put(y0) for _ in range(2 * max(1, len(modes)))]

    def run(tile):
        g = CtGemm(lda=K, W=pW, bias=pb, M=M, N=N, K=K, scale=0.5, epi=epi, Y=outs[0], ldy=N)
        if act == "fp32":
            g.A = pA
        else:
            g.Ahi, g.Alo = pH, pL if act == "hilo" else None
        if seg_w:
            g.nseg, g.seg_w = len(modes), seg_w
            for i, c in enumerate(modes):
                g.seg[i] = CtSeg(mode={"d": 0, "f": 1, "b": 2, "s": 3, "h": 3}[c], base=outs[2 * i], ld=seg_w + 8,
                                 base_lo=outs[2 * i + 1] if c == "s" else None, rowoff=po, hstride=HSTRIDE)
        elif modes == "m":
            g.row_mask = pm
        else:
            g.row_len, g.row_len_step, g.row_stride = pn, 1, 3
        for p in outs:
            hip.backend_htod(p, y0.ctypes.data, y0.size)
        dev.ev.sync()
        lib.ctk_gemm_force_tile(tile)
        assert lib.ctk_gemm_tile(C.byref(g), 1) == (0 if tile == MANY_ROWS else tile)
        lib.ctk_gemm(C.byref(g), None)
        return [dev.get(p, np.uint32, y0.size) for p in outs]

    want = run(MANY_ROWS)
    assert any((w != y0.view(np.uint32)).any() for w in want)
    for tile in TILES:
        if tile in ABSENT[act]:
            continue
        print(f"case: {name} {act} tile {tile}", flush=True)
        for a, b in zip(want, run(tile)):
            assert np.array_equal(a, b), tile


GROUP_TILES = [0] + [t for t in TILES if t not in ABSENT["fp32"]]


@pytest.mark.parametrize("tile", GROUP_TILES)
@pytest.mark.parametrize("rows,K", [((13, 13, 13, 25), 1280), ((101, 40), 1280), ((376, 376, 1), 384),
                                    ((20, 31), 1312), ((5,), 256)],
                         ids=["13", "two", "uneven", "K-not-grouped", "one"])
def test_group_gives_the_single_launches_bits(lib, hip, rows, K, tile):
    """ctk_gemm_group: the bits of each product launched alone, its rows past M
    untouched (K = 1312 has no few-row tile: the group falls back to single launches)."""
    dev = Dev(hip)
    lib.ctk_gemm_group.argtypes = [C.POINTER(CtGemm), C.c_int, C.c_void_p]
    rng = np.random.default_rng(sum(rows) + K)
    N = 328                                     # ends inside every tile
    gs, gs1 = (CtGemm * len(rows))(), (CtGemm * len(rows))()
    outs = []
    for i, M in enumerate(rows):
        px = dev.put(rng.standard_normal((M, K)).astype(np.float32))
        pW = dev.put(f32_to_bf16(rng.standard_normal((N, K)).astype(np.float32)))
        pb = dev.put(f32_to_bf16(rng.standard_normal(N).astype(np.float32)))
        y0 = rng.standard_normal((M + 2, N)).astype(np.float32)
        py = [dev.put(y0), dev.put(y0)]
        outs.append((py, y0))
        for arr, p in ((gs, py[0]), (gs1, py[1])):
            arr[i] = CtGemm(A=px, lda=K, W=pW, bias=pb if i % 2 == 0 else None, Y=p, ldy=N, M=M, N=N, K=K,
                            epi=EPI_FMADD if i % 3 == 1 else EPI_STORE, scale=0.5)
    dev.ev.sync()
    print(f"case: group of {rows} rows, K {K}, tile {tile}", flush=True)
    lib.ctk_gemm_force_tile(tile)
    took = lib.ctk_gemm_tile(gs, len(rows)) if len(rows) > 1 else 0
    assert bool(took) == (K != 1312 and len(rows) > 1) and (not took or not tile or took == tile)
    lib.ctk_gemm_group(gs, len(rows), None)
    lib.ctk_gemm_force_tile(MANY_ROWS)
    for i in range(len(rows)):
        lib.ctk_gemm(C.byref(gs1[i]), None)
    for (a, b), y0 in outs:
        got, want = dev.get(a, np.uint32, y0.size).reshape(y0.shape), dev.get(b, np.uint32, y0.size).reshape(y0.shape)
        assert np.array_equal(got, want)
        assert np.array_equal(got[-2:], y0[-2:].view(np.uint32))
