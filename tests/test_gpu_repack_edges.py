"""Repack and row dequant at the edges of their work split: an odd group count
(two groups per wave / workgroup), one tile, parts at row offsets, and dequant
of row ranges that start and end inside tiles. Bit-exact against the oracle's
dequant of the logical weights, from every source layout."""
import numpy as np
import pytest

from gpu_util import dev, empty, host, repack_from_logical

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K", [(64, 128), (128, 384), (192, 640), (320, 1664)])
@pytest.mark.parametrize("layout", ["ct", "awq_k", "awq_n"])
def test_repack_dequant_edges(orc, N, K, layout):
    import torch

    assert torch.cuda.is_available()
    import w4a16_hip as hip

    q, zp, s = orc.gen_weights(N, K, seed=N + K)
    want = orc.dequant_bf16(q, zp, s)
    w = repack_from_logical(hip, orc, q, zp, s, layout)
    for row0, n in ((0, N), (0, 1), (N - 1, 1), (63, 2 if N > 64 else 1), (5, N - 9)):
        print(f"dequant {layout} {N}x{K} rows {row0}+{n}", flush=True)
        out = torch.full((n + 1, K), 0x5A5A, dtype=torch.int16, device="cuda")
        hip.w4a16_dequant_rows(out[:n], w, row0, n)
        torch.cuda.synchronize()
        got = host(out, np.uint16)
        assert np.array_equal(got[:n], want[row0:row0 + n])
        assert (got[n] == 0x5A5A).all()
    # the prefill GEMM reads the zero points' own array, the skinny kernels the record's copy
    x = orc.gen_x(3, K, seed=1)
    y = empty((3, N), np.uint16)
    hip.gemm_w4a16(y, w, dev(x), 3)
    torch.cuda.synchronize()
    m = orc.parity_metrics(host(y, np.uint16), orc.matmul_f64(x, q, zp, s, round_w=True))
    assert m["max_rel"] <= 1e-2 and m["mean_abs_vs_bf16_ref"] <= 1e-3, m
    hip.awq_free(w)


# the launch shapes of the row dequant: up to 160 (tile, two groups) items one round
# of rows a workgroup, up to 512 two, four beyond
@pytest.mark.parametrize("N,K", [(640, 4096), (704, 4096), (768, 3712), (2048, 4096), (2112, 4096),
                                 (2240, 3968)])
def test_dequant_launch_shapes(orc, N, K):
    import torch
    import w4a16_hip as hip

    q, zp, s = orc.gen_weights(N, K, seed=N + K)
    want = orc.dequant_bf16(q, zp, s)
    w = repack_from_logical(hip, orc, q, zp, s, "ct")
    for row0, n in ((0, N), (1, N - 2), (63, 66), (127, 1)):
        print(f"dequant {N}x{K} rows {row0}+{n}", flush=True)
        out = torch.full((n + 1, K), 0x5A5A, dtype=torch.int16, device="cuda")
        hip.w4a16_dequant_rows(out[:n], w, row0, n)
        torch.cuda.synchronize()
        got = host(out, np.uint16)
        assert np.array_equal(got[:n], want[row0:row0 + n])
        assert (got[n] == 0x5A5A).all()
    hip.awq_free(w)
