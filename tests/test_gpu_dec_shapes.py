"""The decode kernel's launch shapes at the edges of their rules: the largest
output that takes 16 waves (CUs / 4 tiles) and the next, the outputs on either
side of one 64-row unit per workgroup, several units with a remainder, a K just
below and at 32 groups, a K whose LDS leaves no room for 64-row units, more than
eight 32- and 64-row units per workgroup (a second load of the residual). Against
the oracle; the residual and swiglu epilogues bitwise against the plain
projection followed by the separate step."""
import numpy as np
import pytest

from gpu_util import dev, empty, host, repack_from_logical

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,G", [(4096, 31), (4096, 32), (4160, 40), (64, 40), (8192, 33), (8320, 33),
                                 (16384, 8), (16512, 8), (24704, 5), (9600, 25), (8320, 200),
                                 (128, 64), (4096, 65), (83200, 2), (163840, 2), (14720, 7), (16384, 5)])
def test_dec_shapes(orc, N, G):
    import torch

    assert torch.cuda.is_available()
    import w4a16_hip as hip

    K = 128 * G
    scratch = hip.gemv_scratch_alloc(K, N, 128, 1)
    q, zp, s = orc.gen_weights(N, K, seed=N + G)
    w = repack_from_logical(hip, orc, q, zp, s, "awq_k")
    x = orc.gen_x(1, K, seed=G)
    dx = dev(x)
    ref = orc.matmul_f64(x, q, zp, s)
    print(f"dec {N}x{K}", flush=True)
    yf, y = empty((1, N), np.float32), empty((1, N), np.uint16)
    hip.gemv_w4a16_f32(yf, w, dx, scratch)
    hip.gemv_w4a16(y, w, dx, scratch)
    h = dev(orc.gen_x(1, N, seed=3))
    want = h.clone()
    hip.residual_add(want, y, N)
    hip.gemv_residual_w4a16(h, w, dx, 1, scratch)
    idx = empty((1,), np.int32)
    hip.gemv_argmax_w4a16(idx, w, dx, 1, scratch)
    torch.cuda.synchronize()
    got = host(yf, np.float32).astype(np.float64)
    assert np.max(np.abs(got - ref)) / np.max(np.abs(ref)) < 1e-5
    assert np.array_equal(host(y, np.uint16), orc.f32_to_bf16(host(yf, np.float32)))
    assert torch.equal(h, want)
    assert host(idx, np.int32)[0] == int(np.argmax(host(yf, np.float32)))
    if N % 128 == 0:
        a, b = empty((1, N // 2), np.uint16), empty((1, N // 2), np.uint16)
        hip.swiglu(a, y, 1, N // 2)
        hip.gemv_swiglu_w4a16(b, w, dx, 1, scratch)
        torch.cuda.synchronize()
        assert torch.equal(a, b)
    hip.awq_free(w)
    hip.gemv_scratch_free(scratch)
