"""rmsnorm at the edges of its two workgroup sizes (1024 threads up to 512 rows,
256 beyond) and of the chunks a thread keeps (one, two or four rounds of 256:
rows up to 2048, 4096 and 8192 values): one chunk, a row shorter than a workgroup, exactly 8192, one chunk more, several
rounds. Rows do not depend on the workgroup size: bitwise the same row in a
call of 512 and of 513 rows."""
import numpy as np
import pytest

from gpu_util import dev, empty, host

pytestmark = pytest.mark.gpu
EPS = 1e-6


@pytest.mark.parametrize("dim", [8, 1000, 2048, 2056, 4096, 4104, 8192, 8200, 17408])
def test_rmsnorm_rows(orc, dim):
    import torch

    assert torch.cuda.is_available()
    import w4a16_hip as hip

    x, w = orc.gen_x(513, dim, seed=dim), orc.gen_x(1, dim, seed=dim + 1)[0]
    dx, dw = dev(x), dev(w)
    outs = []
    for rows in (1, 512, 513):
        print(f"rmsnorm {rows}x{dim}", flush=True)
        out = empty((rows, dim), np.uint16)
        hip.rmsnorm(out, dx, dw, rows, dim, EPS)
        outs.append(out)
    torch.cuda.synchronize()
    got = [host(o, np.uint16) for o in outs]
    assert np.array_equal(got[0], got[2][:1]) and np.array_equal(got[1], got[2][:512])
    want = orc.bf16_to_f32(orc.rmsnorm_bf16(x, w, EPS)).astype(np.float64)
    have = orc.bf16_to_f32(got[2]).astype(np.float64)
    # one bf16 ulp: the fp32 inverse differs from the oracle's in its last bits
    assert np.all(np.abs(have - want) <= np.abs(want) * 2.0 ** -7 + 1e-30)
    assert np.mean(have != want) < 0.01
