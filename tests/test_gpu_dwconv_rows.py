"""GPU check of the depthwise conv + BatchNorm + SiLU at the row counts where
the launch turns from one row a thread to eight (1600 | 1601): against float64
over several sequences whose edges fall anywhere in a thread's rows, and the
same rows bit for bit on both sides of the line.

Tolerance: 9 products, a division, a square root and the hardware sigmoid, each
within a few units of 2^-24 of values whose terms are of the output's order.
"""
import ctypes as C

import numpy as np
import pytest

import ctbind as cb
from test_gpu_gemv import Dev, bf16_to_f32, f32_to_bf16

pytestmark = pytest.mark.gpu

D, TAPS = cb.ENC_D, cb.ENC_CK


def reference(x, lens, w):
    dww, dwb, bnw, bnb, bnm, bnv = [bf16_to_f32(a).astype(np.float64) for a in w]
    out, at = [], 0
    for n in lens:
        pad = np.pad(x[at:at + n].astype(np.float64), ((4, 4), (0, 0)))
        s = sum(pad[k:k + n] * dww.reshape(D, TAPS)[:, k] for k in range(TAPS)) + dwb
        v = (s - bnm) / np.sqrt(bnv + 1e-5) * bnw + bnb
        out.append(v / (1 + np.exp(-v)))
        at += n
    return np.concatenate(out)


def test_rows_per_thread_line(hip):
    L = C.CDLL(cb.HIP_LIB)
    L.ctk_dwconv_bn_silu_packed.argtypes = [C.c_void_p] * 3 + [C.c_int] + [C.c_void_p] * 9
    dev = Dev(hip)
    rng = np.random.default_rng(3)
    lens = [1, 3, 4, 13, 101, 376, 502, 600, 1]          # 1601 rows
    M = sum(lens)
    x = rng.standard_normal((M, D)).astype(np.float32)
    w = [f32_to_bf16(rng.standard_normal(n).astype(np.float32)) for n in (D * TAPS, D, D, D, D)]
    w.append(f32_to_bf16(rng.uniform(0.5, 2.0, D).astype(np.float32)))
    start = np.repeat(np.cumsum([0] + lens[:-1]), lens).astype(np.int32)
    length = np.repeat(lens, lens).astype(np.int32)
    px, ps, pl, pw = dev.put(x), dev.put(start), dev.put(length), [dev.put(a) for a in w]

    def run(m):
        ph, pg = dev.zeros(M * D * 2), dev.zeros(M * D * 2)
        dev.ev.sync()
        print(f"case: dwconv {m} rows", flush=True)
        L.ctk_dwconv_bn_silu_packed(ph, pg, px, m, ps, pl, *pw, None)
        return [dev.get(p, np.uint16, M * D).reshape(M, D) for p in (ph, pg)]

    many = run(M)                                        # eight rows a thread
    few = run(M - 1)                                     # one (the last sequence is the last row)
    for a, b in zip(many, few):
        assert np.array_equal(a[:M - 1], b[:M - 1])
        assert not b[M - 1].any()
    got = bf16_to_f32(many[0]).astype(np.float64) + bf16_to_f32(many[1])
    ref = reference(x, lens, w)
    assert np.abs(got - ref).max() <= 2e-5 * np.abs(ref).max()
