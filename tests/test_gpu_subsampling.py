"""GPU check of backend_encoder_subsampling's two forms: with 16-byte aligned
scratch the convolutions run fused and every product reads bf16 planes, with
scratch off 16 bytes the fp32 stages run; both give the same bits at every edge
of the clip's length (the three stride-2 stages each end on an odd or an even
row), with a mel row stride longer than the clip.
"""
import numpy as np
import pytest

import ctbind as cb
import kernel_suite as ks

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
