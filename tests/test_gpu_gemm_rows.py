"""The prefill GEMM's tile heights, 64 to 256 rows (the plan takes the height
that costs least): row counts at the edges of each, then each height with each
schedule that the plan pairs it with, against the oracle (weights rounded to
bf16) on sampled rows, bitwise reproducible, and nothing written outside C."""
import numpy as np
import pytest

from gpu_util import dev, host, repack_from_logical

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    import torch

    assert torch.cuda.is_available(), "GPU test run without a GPU"
    import w4a16_hip

    w4a16_hip.lib()
    return w4a16_hip


@pytest.fixture(scope="module")
def ws(hip):
    w = hip.gemm_workspace_alloc(256 << 20)
    yield w
    hip.gemm_workspace_free(w)


# one group (fewer than the buffers), a few, a long K; 70 tiles of columns with
# a ragged last one: whole tiles and split-K of the lower heights
@pytest.mark.parametrize("N,K", [(320, 128), (1024, 640), (5120, 2176), (17856, 1152)])
def test_gemm_tile_heights(hip, orc, ws, N, K):
    q, zp, s = orc.gen_weights(N, K, seed=N + K)
    w = repack_from_logical(hip, orc, q, zp, s, "awq_k")
    for M in (1, 31, 33, 64, 65, 96, 97, 128, 129, 160, 161, 192, 193, 224, 225, 257, 320, 333, 460,
              600, 1000):
        _vs_oracle(hip, orc, w, q, zp, s, M, (None, ws))
    hip.awq_free(w)


# (tile height / 32, schedule) on 256 CUs. Stream-K and hybrid: a workgroup goes
# from one tile's groups to the next one's, with the loads ahead of either.
PLANS = {
    "2 whole": (60, 33216, 384), "3 whole": (70, 33216, 384), "4 whole": (98, 33216, 384),
    "5 whole": (133, 33216, 384), "6 whole": (161, 33216, 384), "7 whole": (196, 33216, 384),
    "8 whole": (450, 22400, 384), "8 stream-K": (500, 9472, 8448), "8 hybrid": (900, 17408, 4096),
    "2 stream-K": (259, 1216, 3072), "3 stream-K": (70, 8256, 3072), "4 stream-K": (196, 8256, 4096),
    "5 stream-K": (133, 9920, 5120), "6 stream-K": (520, 5760, 8192), "7 stream-K": (400, 8256, 8192),
    "2 hybrid": (60, 70656, 2048), "3 hybrid": (257, 33024, 3072), "4 hybrid": (292, 33024, 3072), "5 hybrid": (300, 34880, 2048),
    "6 hybrid": (520, 26560, 2048), "7 hybrid": (1100, 17408, 5120),
    "2 split-K": (70, 256, 2048), "3 split-K": (133, 256, 2048), "4 split-K": (400, 256, 2048),
    "5 split-K": (259, 256, 3072), "6 split-K": (700, 2816, 3072), "7 split-K": (400, 2816, 8192),
    "8 split-K": (450, 5760, 8192),
}


@pytest.mark.parametrize("plan", PLANS)
def test_gemm_height_and_schedule(hip, orc, ws, plan):
    M, N, K = PLANS[plan]
    q, zp, s = orc.gen_weights(N, K, seed=N + K)
    w = repack_from_logical(hip, orc, q, zp, s, "awq_k")
    print(plan, flush=True)
    _vs_oracle(hip, orc, w, q, zp, s, M, (ws,))
    hip.awq_free(w)


def _vs_oracle(hip, orc, w, q, zp, s, M, spaces):
    import torch

    N, K = q.shape
    x = orc.gen_x(M, K, seed=M)
    dx = dev(x)
    rows = np.unique(np.r_[0, M - 1, M // 2, np.random.default_rng(M).integers(0, M, 3)])
    ref = orc.matmul_f64(x[rows], q, zp, s, round_w=True)
    for use in spaces:
        print(f"gemm rows {M} {N}x{K} ws={use is not None}", flush=True)
        big = torch.full((M + 2, N), 0x5A5A, dtype=torch.int16, device="cuda")
        hip.gemm_w4a16(big[1:M + 1], w, dx, M, use)
        again = torch.empty((M, N), dtype=torch.int16, device="cuda")
        hip.gemm_w4a16(again, w, dx, M, use)
        torch.cuda.synchronize()
        assert torch.equal(big[1:M + 1], again)
        assert (big[0] == 0x5A5A).all() and (big[M + 1] == 0x5A5A).all()
        m = orc.parity_metrics(host(again, np.uint16)[rows], ref)
        assert m["max_rel"] <= 1e-2 and m["mean_abs_vs_bf16_ref"] <= 1e-3, (M, m)


# split-K with other slices than 256-row tiles have, stream-K, hybrid and whole
# tiles, all below 256 rows a tile; ragged last rows and columns
@pytest.mark.parametrize("M,N,K", [(200, 1024, 2560), (200, 5120, 4096), (333, 5184, 2176),
                                   (100, 34816, 5120), (300, 34816, 5120), (300, 34816, 1024)])
def test_gemm_variants_bitwise_at_the_plan(hip, ws, M, N, K):
    """Under the cost model's own schedule (-1) too, the kernel variants cut a call
    the same way: bitwise equal, and nothing written outside C."""
    import torch

    G = K // 128
    q = torch.empty(K // 8 * N, dtype=torch.int32, device="cuda")
    s = torch.empty(G * N, dtype=torch.int16, device="cuda")
    z = torch.empty(G * N // 8, dtype=torch.int32, device="cuda")
    hip.gen_awq_k(q, s, z, N, K, N + K, 3)
    w = hip.awq_alloc_fused(N, K)
    hip.awq_repack_awq_into(w, 0, q, s, z, N, hip.LAYOUT_AWQ_K)
    x = torch.empty(M * K, dtype=torch.int16, device="cuda")
    hip.gen_bf16(x, M * K, 0, M + K, 0)
    try:
        for use in (None, ws):
            outs = []
            for variant in (0, 1, 2):
                print(f"gemm variant {variant} {M}x{N}x{K} ws={use is not None}", flush=True)
                hip.tune_gemm(-1, variant)
                big = torch.full((M + 2, N), 0x5A5A, dtype=torch.int16, device="cuda")
                hip.gemm_w4a16(big[1:M + 1], w, x, M, use)
                outs.append(big)
            torch.cuda.synchronize()
            assert (outs[0][0] == 0x5A5A).all() and (outs[0][M + 1] == 0x5A5A).all()
            for variant in (1, 2):
                assert torch.equal(outs[0], outs[variant]), variant
    finally:
        hip.tune_gemm(-1, 0)
    hip.awq_free(w)
