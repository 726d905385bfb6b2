"""The 16-byte forms of the fp32 row int8 and per-tensor fp8 quantizers, bit for
bit against the oracle (int8) and against the one-value-per-load forms, which
the same values off 16 bytes take: rows of one chunk, rows that end inside and
at the edge of each register tile, tails of 1 to 3 values, degenerate rows, NaN,
infinities, signed zeros, denormals and exact halves."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _values(rng, rows, cols):
    x = (rng.normal(0, 1, (rows, cols)) * 10.0 ** rng.integers(-6, 6, (rows, 1))).astype(np.float32)
    x[0] = np.float32(127.0)
    x[0, ::2] = rng.integers(-126, 126, x[0, ::2].shape) + np.float32(0.5)     # halves: scale 1
    if rows > 3:
        x[1] = 0.0
        x[1, 0] = -0.0
        x[2] = rng.integers(-9, 9, cols) * np.float32(1e-41)
        x[3, cols // 2] = np.nan
    return x


def _both(x):
    off = torch.empty(x.size + 1, device=DEV)
    off[1:] = torch.from_numpy(x).to(DEV).reshape(-1)
    return torch.from_numpy(x).to(DEV), off[1:].reshape(x.shape)


@pytest.mark.parametrize("rne", [False, True])
@pytest.mark.parametrize("rows,cols", [(1, 4), (5, 1024), (4, 1028), (7, 4096), (4, 4100), (4, 16384), (4, 16388)])
def test_int8_rows(lib, oracle, rows, cols, rne):
    print(f"[gpu] int8 rows f32 {rows}x{cols} rne={rne}", flush=True)
    x = _values(np.random.default_rng(rows * cols), rows, cols)
    got = []
    for xd in _both(x):
        q = torch.empty((rows, cols), dtype=torch.int8, device=DEV)
        s = torch.empty(rows, device=DEV)
        lib.dev_quantize_int8_channel(xd, q, s, half_even=rne)
        got.append((q.cpu().numpy(), s.cpu().numpy()))
    np.testing.assert_array_equal(got[0][0], got[1][0])
    np.testing.assert_array_equal(got[0][1], got[1][1])
    fin = np.isfinite(x).all(axis=1)
    ref = (oracle.quantize_int8_channel_rne if rne else oracle.quantize_int8_channel)(x)
    np.testing.assert_array_equal(got[0][0][fin], np.asarray(ref[1]).reshape(rows, cols)[fin])


@pytest.mark.parametrize("n", [1, 3, 4, 7, 1024, 4099, 300001])
def test_fp8_tensor(lib, n):
    print(f"[gpu] fp8 tensor f32 {n}", flush=True)
    x = _values(np.random.default_rng(n), 1, n).reshape(n)
    x[n // 2] = 1000.0
    x[-1] = -3000.0
    if n > 8:
        x[5], x[6] = np.nan, -0.0
    got = []
    for xd in _both(x):
        c = torch.empty(n, dtype=torch.uint8, device=DEV)
        s = torch.empty(1, device=DEV)
        lib.dev_quantize_fp8_e4m3_scaled(xd, c, s)
        got.append((c.cpu().numpy(), float(s.cpu())))
    np.testing.assert_array_equal(got[0][0], got[1][0])
    assert got[0][1] == got[1][1] == float(np.float32(3000.0) / np.float32(240.0))
