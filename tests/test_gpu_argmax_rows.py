"""argmax_rows over whole, ragged and unaligned rows: one workgroup reads a row
as the values before its first 16-byte boundary, 16-byte chunks (8192 at a
time) and the values after the last chunk. Odd row lengths put every row at
another alignment. Ties, NaN and -inf follow the reference's strict compare
from (-FLT_MAX, 0) (src/kernels/elementwise.cu:96-158)."""
import numpy as np
import pytest

from gpu_util import dev, empty, host

pytestmark = pytest.mark.gpu


def _strict_argmax(bits: np.ndarray) -> np.ndarray:
    f = (bits.astype(np.uint32) << 16).view(np.float32)
    f = np.where(np.isnan(f), -np.inf, f)
    top = f.max(axis=1, keepdims=True)
    return np.where(top[:, 0] > -np.finfo(np.float32).max, np.argmax(f == top, axis=1), 0).astype(np.int32)


@pytest.mark.parametrize("n", [1, 7, 8, 9, 63, 1025, 8191, 8200, 65541, 248320])
@pytest.mark.parametrize("kind", ["random", "ties", "special"])
def test_argmax_rows(orc, n, kind):
    import torch
    import w4a16_hip as hip

    rng = np.random.default_rng(n)
    rows = 9
    if kind == "ties":     # few distinct values: the lowest index must win
        v = rng.choice(np.array([0x0000, 0x8000, 0x3F80, 0xBF80], np.uint16), size=(rows, n))
    else:
        v = orc.gen_x(rows, n, seed=n)
    if kind == "special":
        v = v.copy()
        v[:, rng.integers(0, n, max(1, n // 4))] = 0x7FC0          # NaN
        v[1] = 0xFF80                                               # all -inf: index 0
        v[2] = 0x7FC0                                               # all NaN: index 0
        v[3, -1] = 0x7F80                                           # +inf in the last place
        v[4, 0] = 0x7F80                                            # and in the first
    out = empty((rows,), np.int32)
    print(f"argmax rows n={n} {kind}", flush=True)
    hip.argmax_rows(out, dev(v), rows, n)
    torch.cuda.synchronize()
    got = host(out, np.int32)
    assert np.array_equal(got, _strict_argmax(v))
    if kind != "special":
        assert np.array_equal(got, orc.argmax_rows_bf16(v))


# the edges of the workgroup sizes: 64 threads up to 2048 values (value by value up to
# 128), 1024 for rows of more than 24576 values in calls of at most 512 rows, 256 for the
# others
@pytest.mark.parametrize("n,rows", [(2047, 300), (2048, 3), (2049, 300), (24576, 5), (24577, 5),
                                    (24583, 512), (24583, 513), (3, 70000), (63, 7),
                                    (65, 7), (128, 40), (129, 40)])
def test_argmax_rows_workgroups(orc, n, rows):
    import torch
    import w4a16_hip as hip

    v = orc.gen_x(rows, n, seed=n + rows)
    v[0, -1] = v[rows - 1, 0] = 0x7F80          # +inf: the last and the first place
    out = empty((rows + 1,), np.int32)
    out.fill_(-7)
    print(f"argmax rows n={n} rows={rows}", flush=True)
    hip.argmax_rows(out[:rows], dev(v), rows, n)
    torch.cuda.synchronize()
    got = host(out, np.int32)
    assert np.array_equal(got[:rows], _strict_argmax(v)) and got[rows] == -7
