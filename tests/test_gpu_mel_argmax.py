"""GPU checks of the log-mel front-end's and the argmax's launch shapes: clips of
few frames (a workgroup's last wavefronts without a frame), of a whole number of
workgroups, and longer than the rows kept in registers (4096 frames); rows of
logits of whole float4 and not, with ties, NaN and infinities.

The spectrogram is held to the oracle's within the tolerance that
test_gpu_engine.py derives for it (twiddle recurrence against exact twiddles),
and to a restatement in float64.
"""
import ctypes as C
import hashlib
import threading

import numpy as np
import pytest

import ctbind as cb
import oracle_bind as ob
from test_gpu_gemv import Dev

pytestmark = pytest.mark.gpu


def test_mel_lengths(hip, kernel_model):
    hip.backend_weights_upload_blob(kernel_model.data_ptr, kernel_model.data_bytes)
    eng = cb.Engine(kernel_model, slots=1, max_requests=2, max_frames=40, kv_bf16=True)
    try:
        # short after long: the kept buffers are longer than the clip
        for n in (160, 3 * 160, 4 * 160 + 1, 4097 * 160, 1000):
            x = cb.synth_audio(n, n)
            print(f"case: mel n={n}", flush=True)
            got, ref = eng.mel(x), ob.compute_mel(x)
            assert got.shape == ref.shape
            assert np.abs(got - ref).max() < 2e-3, n
            assert np.array_equal(got, eng.mel(x))
    finally:
        eng.close()


def mel64(x):
    """The log-mel spectrogram in float64 (window and filters included)."""
    n, T = len(x), 1 + len(x) // 160
    x = x.astype(np.float64)
    e = np.concatenate([np.zeros(200), x, np.zeros(200 + 160)])
    e[1:] -= 0.97 * e[:-1].copy()
    hann = 0.5 * (1 - np.cos(2 * np.pi * np.arange(400) / 399))
    spec = np.array([np.abs(np.fft.rfft(e[160 * t:160 * t + 400] * hann, 512)) ** 2 for t in range(T)])
    def hz(m):
        return np.where(m < 15, m * 200 / 3, 1000 * np.exp((m - 15) * np.log(6.4) / 27))
    top = 15 + np.log(8.0) / (np.log(6.4) / 27)
    p = hz(np.linspace(0, top, 130))
    f = np.linspace(0, 8000, 257)
    fb = [np.maximum(0, np.minimum((f - p[i]) / (p[i + 1] - p[i]), (p[i + 2] - f) / (p[i + 2] - p[i + 1]))) * 2 / (p[i + 2] - p[i])
          for i in range(128)]
    mel = np.log(np.array(fb) @ spec.T + 2.0 ** -24)
    d = mel - mel.mean(1, keepdims=True)
    return d / np.sqrt((d ** 2).sum(1, keepdims=True) / (T - 1) + 1e-5)


@pytest.mark.parametrize("n", [3 * 160, 8000, 48000, 327680, 655520])
def test_mel_float64(hip, kernel_model, n):
    """Against float64 in the 2-norm.  Nine butterfly stages of three roundings
    of 2^-24, twice in the power and again its logarithm's absolute error: 27
    2^-23 = 3.2e-6, and a row's standard deviation here is 0.5 and more; the
    window and the filters are rounded once (2^-24)."""
    hip.backend_weights_upload_blob(kernel_model.data_ptr, kernel_model.data_bytes)
    eng = cb.Engine(kernel_model, slots=1, max_requests=2, max_frames=40, kv_bf16=True)
    try:
        x = (np.random.default_rng(n).integers(-8192, 8193, n) / np.float32(32768)).astype(np.float32)
        print(f"case: mel float64 n={n}", flush=True)
        got, ref = eng.mel(x).astype(np.float64), mel64(x)
        err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
        print(f"  relative error {err:.2e}", flush=True)
        assert err <= 7e-6
    finally:
        eng.close()


# samples: SHA-256 (first 16 digits) of the spectrogram whose rows are summed by
# 64 lanes in fp32, each lane its own frames in turn and every square fused
# into its sum, the lanes by wave_sum.  Frames a clip: few (four wavefronts a
# frame) up to 2048 = 327520 samples, one wavefront a frame from 2049 on.
MEL_BITS = {
    327520: "605bf024add393b3", 327680: "c81eeea31b284681",
    160: "b4e64e235ea18f25", 641: "247ea271ee4d5e36", 1000: "9683ffde0b0f3c68", 8000: "ae1c442037cc9fd9",
    16000: "5de6fea4e623cd40", 41000: "2260df0d47755b46", 163000: "3d027f43b70a4d6e", 164000: "4c6cf605bca0fe3d",
    320000: "7b33943304d1e715", 480000: "34f949f46aa91410", 655200: "04785f2544b22847", 655520: "8a2161bebd3f6645",
}


def test_mel_bits(hip, kernel_model):
    """The spectrogram's bits do not depend on how the launches are split: 48
    layers follow, and where their FFN rounds activations to bf16 a changed last
    bit grows to 3e-3 of the encoder's output."""
    hip.backend_weights_upload_blob(kernel_model.data_ptr, kernel_model.data_bytes)
    eng = cb.Engine(kernel_model, slots=1, max_requests=2, max_frames=40, kv_bf16=True)
    try:
        for n, want in MEL_BITS.items():
            x = (np.random.default_rng(n).integers(-8192, 8193, n) / np.float32(32768)).astype(np.float32)
            print(f"case: mel bits n={n}", flush=True)
            assert hashlib.sha256(eng.mel(x).tobytes()).hexdigest()[:16] == want, n
    finally:
        eng.close()


def test_mel_kept_buffer(hip, kernel_model):
    """Ever longer clips reuse one buffer of at most 64 MB: the device's free
    memory stays where the first of them left it, also past a clip too long for
    a kept buffer (10 M samples: 73 MB)."""
    rt = C.CDLL("libamdhip64.so")
    free, total = C.c_size_t(), C.c_size_t()

    def left():
        assert rt.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value

    hip.backend_weights_upload_blob(kernel_model.data_ptr, kernel_model.data_bytes)
    eng = cb.Engine(kernel_model, slots=1, max_requests=2, max_frames=40, kv_bf16=True)
    try:
        eng.mel(np.zeros(160, np.float32))              # the kernels are loaded before memory is counted
        before, after = left(), []
        for n in (4_800_000, 5_600_000, 6_400_000, 8_000_000, 10_000_000, 160):
            print(f"case: mel kept buffer n={n}", flush=True)
            eng.mel(np.zeros(n, np.float32))
            after.append(left())
        assert before - after[0] <= 66 << 20            # the allocator's granule is 2 MB
        assert after == after[:1] * len(after)
    finally:
        eng.close()


def test_mel_threads(hip, kernel_model):
    """Four threads on one engine, clips of all sizes at once: each gets its
    clip's bits."""
    hip.backend_weights_upload_blob(kernel_model.data_ptr, kernel_model.data_bytes)
    eng = cb.Engine(kernel_model, slots=1, max_requests=2, max_frames=40, kv_bf16=True)
    sizes = [160, 655520, 16000, 320000, 1000, 163000]
    clips = {n: (np.random.default_rng(n).integers(-8192, 8193, n) / np.float32(32768)).astype(np.float32) for n in sizes}
    wrong = []

    def work(k):
        for i in range(18):
            n = sizes[(i * (k + 1) + k) % len(sizes)]
            got = hashlib.sha256(eng.mel(clips[n]).tobytes()).hexdigest()[:16]
            if got != MEL_BITS[n]:
                wrong.append((k, i, n))

    try:
        print("case: mel on four threads", flush=True)
        threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not wrong
    finally:
        eng.close()


@pytest.mark.parametrize("n", [1, 63, 1000, 4096, 16384, 16385, 16388, 40000])
def test_argmax_rows(hip, n):
    L = C.CDLL(cb.HIP_LIB)
    L.ctk_argmax.argtypes = [C.c_void_p, C.c_void_p, C.c_int, C.c_int, C.c_void_p, C.c_void_p]
    dev = Dev(hip)
    rng = np.random.default_rng(n)
    R = 9
    x = rng.integers(-50, 50, (R, n)).astype(np.float32)     # ties: the lowest index wins
    x[1] = -np.inf
    x[2, n // 2] = np.nan                                    # NaN never wins ..
    x[3, 0] = np.nan                                         # .. but stays the answer at index 0
    x[4, n - 1] = np.inf
    x[5] = np.nan
    x[6] = np.finfo(np.float32).min
    want = []
    for row in x:
        best = 0
        if row[0] == row[0]:
            clean = np.where(np.isnan(row), -np.inf, row)
            best = int(np.argmax(clean))
        want.append(best)
    act = np.ones(R, np.int32)
    act[8] = 0
    po, px, pa = dev.put(np.full(R, -5, np.int32)), dev.put(x), dev.put(act)
    dev.ev.sync()
    print(f"case: argmax n={n}", flush=True)
    L.ctk_argmax(po, px, R, n, pa, None)
    got = dev.get(po, np.int32, R)
    assert got[8] == -5
    assert np.array_equal(got[:8], want[:8])
