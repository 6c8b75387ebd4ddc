"""GPU check of backend_encoder_subsampling's two forms: with 16-byte aligned
scratch the convolutions run fused and every product reads bf16 planes, with
scratch off 16 bytes the fp32 stages run; both give the same bits at every edge
of the clip's length (the three stride-2 stages each end on an odd or an even
row), with a mel row stride longer than the clip.  The fused kernels are also
held to the two stages' kernels, whose taps outside the clip are skipped: a
non-finite weight there must not meet the padding.
"""
import ctypes as C

import numpy as np
import pytest

import ctbind as cb
import kernel_suite as ks
from test_gpu_gemv import Dev, f32_to_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T_mel", [1, 2, 3, 4, 5, 8, 9, 17, 31, 100, 1001])
def test_aligned_and_unaligned_scratch_give_the_same_bits(hip, kernel_model, T_mel):
    m = kernel_model
    hip.backend_weights_upload_blob(m.data_ptr, m.data_bytes)
    dev = ks.ArenaDev(hip, floats=1 << 24)
    rng = np.random.default_rng(T_mel)
    stride, T = T_mel + 3, cb.t_enc(T_mel)
    mel = np.full((cb.N_MELS, stride), np.nan, np.float32)      # nothing past a row's end is read
    mel[:, :T_mel] = rng.standard_normal((cb.N_MELS, T_mel))
    T1 = (T_mel + 1) // 2
    work = cb.SUB_CH * (T1 * 64 + (T1 + 1) // 2 * 32)
    pm, _ = dev.put(mel)
    px, _ = dev.put(np.zeros((T, cb.ENC_D), np.float32))
    pw, _ = dev.put(np.zeros(work + 4, np.float32))
    assert pw % 16 == 0
    out = []
    for off in (0, 4):
        print(f"case: subsampling T_mel={T_mel} scratch offset {off}", flush=True)
        hip.backend_encoder_subsampling(pm, T_mel, stride, px, T, pw + off, m.weights_ref())
        y = np.empty((T, cb.ENC_D), np.float32)
        hip.backend_dtoh(y.ctypes.data, px, y.nbytes)
        out.append(y)
    assert np.all(np.isfinite(out[0]))
    assert np.array_equal(out[0].view(np.uint32), out[1].view(np.uint32))


# weights at single taps that a padding tap must not meet (bf16 bits): infinities and NaN
HOSTILE = [0x7F80, 0xFF80, 0x7FC0]


def hostile(rng, n):
    """n x 9 finite bf16 weights; channel c < 27 has one non-finite tap, every
    tap with every value once."""
    w = f32_to_bf16(rng.standard_normal((n, 9)).astype(np.float32))
    for c in range(27):
        w[c, c % 9] = HOSTILE[c // 9]
    return w


def same_planes(got, want):
    """bit for bit, any NaN equal to any other"""
    for a, b in zip(got, want):
        na, nb = (a & 0x7FFF) > 0x7F80, (b & 0x7FFF) > 0x7F80
        assert np.array_equal(na, nb)
        assert np.array_equal(a[~na], b[~nb])


def conv_lib():
    L = C.CDLL(cb.HIP_LIB)
    P, I = C.c_void_p, C.c_int
    L.ctk_sub_conv0.argtypes = [P, P, I, I, P, P, P]
    L.ctk_sub_dwconv.argtypes = [P, P, I, I, P, P, P]
    L.ctk_sub_conv0_dw.argtypes = [P, P, P, I, I, P, P, P, P, P]
    L.ctk_sub_dw_split.argtypes = [P, P, P, I, I, P, P, P]
    L.ctk_split.argtypes = [P, P, P, C.c_long, P]
    return L


@pytest.mark.parametrize("T_mel", [1, 2, 3, 4, 5, 8, 9, 31])
def test_fused_convolutions_skip_padding(hip, T_mel):
    """Non-finite weights and samples, and biases of -0: the fused first two
    convolutions give the two stages' bits, whose taps outside are skipped."""
    L, dev = conv_lib(), Dev(hip)
    rng = np.random.default_rng(T_mel)
    mel = rng.standard_normal((cb.N_MELS, T_mel)).astype(np.float32)
    mel[5, T_mel - 1], mel[70, 0] = np.inf, np.nan
    b = f32_to_bf16(rng.standard_normal((2, cb.SUB_CH)).astype(np.float32))
    b[:, :40] = 0x8000
    pm, pb0, pb1 = dev.put(mel), dev.put(b[0]), dev.put(b[1])
    T1 = (T_mel + 1) // 2
    n = (T1 + 1) // 2 * 32 * cb.SUB_CH
    p0, p1, planes = dev.zeros(T1 * 64 * cb.SUB_CH * 4), dev.zeros(n * 4), [dev.zeros(n * 2) for _ in range(4)]
    plain = f32_to_bf16(rng.standard_normal((2, cb.SUB_CH, 9)).astype(np.float32))
    for w0, wd in ((hostile(rng, cb.SUB_CH), plain[1]), (plain[0], hostile(rng, cb.SUB_CH))):
        pw0, pwd = dev.put(w0.ravel()), dev.put(wd.ravel())
        dev.ev.sync()
        print(f"case: fused convolutions T_mel={T_mel}", flush=True)
        L.ctk_sub_conv0(p0, pm, T_mel, T_mel, pw0, pb0, None)
        L.ctk_sub_dwconv(p1, p0, T1, 64, pwd, pb1, None)
        L.ctk_split(planes[0], planes[1], p1, n, None)
        L.ctk_sub_conv0_dw(planes[2], planes[3], pm, T_mel, T_mel, pw0, pb0, pwd, pb1, None)
        a = [dev.get(p, np.uint16, n) for p in planes]
        same_planes(a[2:], a[:2])


@pytest.mark.parametrize("H,Wd", [(1, 32), (2, 32), (5, 32), (8, 32), (3, 33), (4, 5), (1, 1)])
def test_depthwise_skips_padding(hip, H, Wd):
    L, dev = conv_lib(), Dev(hip)
    rng = np.random.default_rng(H * 100 + Wd)
    x = np.maximum(rng.standard_normal((H, Wd, cb.SUB_CH)), 0).astype(np.float32)
    x[0, 0, 100], x[H - 1, Wd - 1, 101] = np.inf, np.nan
    w = hostile(rng, cb.SUB_CH)
    b = f32_to_bf16(rng.standard_normal(cb.SUB_CH).astype(np.float32))
    b[:40] = 0x8000
    px, pw, pb = dev.put(x), dev.put(w.ravel()), dev.put(b)
    n = (H + 1) // 2 * ((Wd + 1) // 2) * cb.SUB_CH
    p1, planes = dev.zeros(n * 4), [dev.zeros(n * 2) for _ in range(4)]
    dev.ev.sync()
    print(f"case: depthwise {H}x{Wd}", flush=True)
    L.ctk_sub_dwconv(p1, px, H, Wd, pw, pb, None)
    L.ctk_split(planes[0], planes[1], p1, n, None)
    L.ctk_sub_dw_split(planes[2], planes[3], px, H, Wd, pw, pb, None)
    a = [dev.get(p, np.uint16, n) for p in planes]
    same_planes(a[2:], a[:2])
