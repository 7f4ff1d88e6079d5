"""The skinny kernel that holds the activations in registers (k_rows_xr) at the
edges of its range, bitwise against the register-item form (qw4_tune_decode
mode 2: the same sums in the same order): group counts around 8 and 8 x 3, 5
and 8 (the last it takes, and the first it does not), more than one unit per
workgroup with a remainder, few 16-row units, every row quarter."""
import numpy as np
import pytest

from gpu_util import dev, empty, host, repack_from_logical

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    import torch

    assert torch.cuda.is_available(), "GPU test run without a GPU"
    import w4a16_hip

    w4a16_hip.lib()
    return w4a16_hip


@pytest.fixture(scope="module")
def scratch(hip):
    s = hip.gemv_scratch_alloc(65 * 128, 40000, 128, 16)
    yield s
    hip.gemv_scratch_free(s)


def _both(hip, run):
    import torch

    hip.tune_decode(0)
    got = run()
    try:
        hip.tune_decode(2)
        want = run()
    finally:
        hip.tune_decode(0)
    torch.cuda.synchronize()
    assert torch.equal(got, want)


# 8256 rows: 129 tiles, just over half the CUs; 8320 an even tile count (swiglu
# pairs); 34816 several units a workgroup; 192 few 16-row units
@pytest.mark.parametrize("N,G", [(8320, 1), (8256, 7), (8320, 8), (8256, 9), (8320, 24), (8256, 25),
                                 (34816, 40), (8320, 41), (8256, 64), (8256, 65), (192, 3), (192, 40),
                                 (64, 64)])
def test_rows_xr_bitwise(hip, orc, scratch, N, G):
    K = 128 * G
    q, zp, s = orc.gen_weights(N, K, seed=N + G)
    w = repack_from_logical(hip, orc, q, zp, s, "awq_k")
    x16 = orc.gen_x(16, K, seed=G)
    for M in (2, 4, 5, 9, 16):
        print(f"rows_xr {N}x{K} M={M}", flush=True)
        x, h0 = dev(x16[:M]), dev(orc.gen_x(M, N, seed=M))

        def bf16():
            y = empty((M, N), np.uint16)
            hip.gemm_small_w4a16(y, w, x, M, scratch)
            return y

        def residual():
            h = h0.clone()
            hip.gemv_residual_w4a16(h, w, x, M, scratch)
            return h

        def swiglu():
            y = empty((M, N // 2), np.uint16)
            hip.gemv_swiglu_w4a16(y, w, x, M, scratch)
            return y

        def argmax():
            idx = empty((M,), np.int32)
            hip.gemv_argmax_w4a16(idx, w, x, M, scratch)
            return idx.view(dtype=h0.dtype)

        for run in (bf16, residual, argmax) + ((swiglu,) if N % 128 == 0 else ()):
            _both(hip, run)
    hip.awq_free(w)


@pytest.mark.parametrize("N,G", [(8256, 7), (8256, 40), (16448, 64), (192, 9), (20032, 20), (8256, 24), (8256, 25)])
def test_rows_xr_w8_bitwise(hip, orc, scratch, N, G):
    K = 128 * G
    src = dev(orc.gen_x(N, K, seed=N + G))
    w = hip.quantize_w8a16(src, N, K)
    for M in (2, 7, 9, 16):
        print(f"rows_xr w8 {N}x{K} M={M}", flush=True)
        x = dev(orc.gen_x(M, K, seed=M))

        def bf16():
            y = empty((M, N), np.uint16)
            hip.gemm_small_w8a16(y, w, x, M, scratch)
            return y

        def argmax():
            idx = empty((M,), np.int32)
            hip.gemv_argmax_w8a16(idx, w, x, M, scratch)
            return idx.view(dtype=x.dtype)

        for run in (bf16, argmax):
            _both(hip, run)
    hip.w8a16_free(w)
