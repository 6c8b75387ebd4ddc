"""GPU checks of the decoder-class GEMM (ctk_gemm on fp32 activations, K = 1024
or 4096 -> 1024) at the sizes where its choice of tile turns: a row has the
same bits at every row count (each count takes the tile of its own), rows past
the launch and masked rows are not written, and the sums agree with float64.

Tolerance: an activation is hi + lo with a remainder of at most 2^-17 of it, and
a sum of K products in fp32 chains of K/8 adds at most K/8 2^-24 of the sum of
magnitudes: together below (2^-17 + 512 2^-24) sum |a||w| for K = 4096.
"""
import ctypes as C

import numpy as np
import pytest

import ctbind as cb
from structs import CtGemm
from test_gpu_gemv import Dev, bf16_to_f32, f32_to_bf16

pytestmark = pytest.mark.gpu

ROWS = [1, 16, 17, 33, 64, 65, 80]      # edges of 16- and 32-row tiles, one and two rounds of workgroups
TOL = 2.0 ** -17 + 512 * 2.0 ** -24


@pytest.mark.parametrize("N,K", [(1024, 1024), (4096, 1024), (16384, 1024), (1000, 1024), (1024, 4096)])
def test_rows_do_not_depend_on_the_tile(hip, N, K):
    L = C.CDLL(cb.HIP_LIB)
    L.ctk_gemm_sizeof.restype = C.c_int
    assert C.sizeof(CtGemm) == L.ctk_gemm_sizeof()
    L.ctk_gemm.argtypes = [C.POINTER(CtGemm), C.c_void_p]
    dev = Dev(hip)
    rng = np.random.default_rng(N + K)
    M = max(ROWS)
    x = rng.standard_normal((M, K)).astype(np.float32)
    W = f32_to_bf16(rng.standard_normal((N, K)).astype(np.float32) / np.float32(np.sqrt(K)))
    b = f32_to_bf16(rng.standard_normal(N).astype(np.float32))
    mask = (np.arange(M) % 5 != 3).astype(np.int32)
    px, pW, pb, pm = dev.put(x), dev.put(W), dev.put(b), dev.put(mask)
    fill = np.full((M, N), -7.0, np.float32)
    pY = dev.put(fill)

    def run(m, first=0, masked=False):
        hip.backend_htod(pY, fill.ctypes.data, fill.size)
        g = CtGemm(A=px + first * K * 4, lda=K, W=pW, bias=pb, Y=pY, ldy=N, M=m, N=N, K=K,
                   row_mask=pm if masked else None)
        dev.ev.sync()
        print(f"case: dec GEMM {m}x{N}x{K} masked={masked}", flush=True)
        L.ctk_gemm(C.byref(g), None)
        return dev.get(pY, np.float32, M * N).reshape(M, N)

    full = run(M)
    for m in ROWS[:-1]:
        got = run(m)
        assert np.array_equal(got[:m].view(np.uint32), full[:m].view(np.uint32)), m
        assert np.all(got[m:] == -7.0), m
    assert np.array_equal(run(1, first=M - 1)[0].view(np.uint32), full[M - 1].view(np.uint32))
    got = run(M, masked=True)
    assert np.array_equal(got[mask != 0].view(np.uint32), full[mask != 0].view(np.uint32))
    assert np.all(got[mask == 0] == -7.0)
    w64 = bf16_to_f32(W).astype(np.float64)
    ref = x.astype(np.float64) @ w64.T + bf16_to_f32(b)
    bound = TOL * (np.abs(x).astype(np.float64) @ np.abs(w64).T + np.abs(bf16_to_f32(b)))
    assert np.all(np.abs(full - ref) <= bound)
