"""qw4_linear's passes of two 16-row blocks (k_rows_xr with MB = 2): every row
count around them, a single last row left to the GEMV, group counts around 8,
24 and 40 (the last it takes, and the first it does not) -- bitwise equal to
16-row gemm_small passes."""
import numpy as np
import pytest

from gpu_util import dev, empty, repack_from_logical

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,G", [(64, 1), (192, 9), (1088, 24), (1088, 25), (8320, 40), (8320, 41)])
def test_linear_two_blocks(orc, N, G):
    import torch

    assert torch.cuda.is_available()
    import w4a16_hip as hip

    K = 128 * G
    scratch = hip.gemv_scratch_alloc(K, N, 128, 16)
    q, zp, s = orc.gen_weights(N, K, seed=N + G)
    w = repack_from_logical(hip, orc, q, zp, s, "awq_k")
    mt = hip.linear_max_t(w)
    assert mt >= 48
    x = dev(orc.gen_x(48, K, seed=G))
    for T in (16, 17, 18, 31, 32, 33, 34, 47, 48):
        print(f"linear two blocks {N}x{K} T={T}", flush=True)
        big = torch.full((T + 1, N), 0x5A5A, dtype=torch.int16, device="cuda")
        hip.linear_w4a16(big[:T], w, x[:T], T, scratch)
        want = empty((T, N), np.uint16)
        for i in range(0, T, 16):
            n = min(16, T - i)
            hip.gemm_small_w4a16(want[i:i + n], w, x[i:i + n], n, scratch)
        torch.cuda.synchronize()
        assert torch.equal(big[:T], want), T
        assert (big[T] == 0x5A5A).all()
    hip.awq_free(w)
    hip.gemv_scratch_free(scratch)
