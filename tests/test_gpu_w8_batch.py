"""W8 weight-only linears with several rows (k_w8_batch: fp32 activations as
three bf16 pieces on the matrix cores): edges of the 32 and 64 row blocks and
of the 128-column tiles, widths that are no multiple of a 64-column step or of
16 bytes, one span of K and many, bias, and activations of unlike magnitude,
signed zero, infinities and NaN.

The pieces hold every bit of an fp32 activation, subnormal ones too, and an int8 is one bf16, so
only the fp32 accumulation rounds: chains of 128 columns and of K / 128 partial
sums, each rounding 2^-24 of a value a few times the result's size.  2e-6 of
the largest result is over ten times the expected random walk."""
import numpy as np
import pytest
import torch

from test_gpu_qlinear import DEV, rel_err, to_dev

pytestmark = pytest.mark.gpu


def _run(lib, x, q, s, b=None):
    y = torch.full((x.shape[0], q.shape[0]), 7.0, device=DEV)
    lib.qlinear_w8_gemv(to_dev(x), to_dev(q), to_dev(s), y, bias=None if b is None else to_dev(b))
    torch.cuda.synchronize()
    return y.cpu().numpy()


@pytest.mark.parametrize("M,N,K,bias,mean", [
    (2, 300, 6144, False, 0.0),     # the fewest rows that take it
    (5, 1, 64, False, 0.0),         # one column, one step
    (13, 130, 20, True, 0.0),       # less than a step, 4-byte aligned rows
    (7, 129, 4036, False, 1.0),     # 4036 = 63 steps and 4 columns
    (31, 128, 1040, True, 0.0),
    (32, 257, 8192, False, 0.0),    # many spans
    (33, 100, 2048, True, -3.0),    # two blocks of 32 rows
    (64, 1000, 448, False, 0.0),
    (65, 4096, 512, True, 0.0),     # blocks of 64 rows, the second with one
    (200, 4100, 320, False, 0.0),   # row and column tails
])
def test_w8_batch_matches_float64(lib, M, N, K, bias, mean):
    print(f"[gpu] w8 batch M={M} N={N} K={K} bias={bias} mean={mean}", flush=True)
    rng = np.random.default_rng(M * 7 + N + K)
    x = (rng.normal(mean, 1, (M, K)) * np.exp(rng.normal(0, 1, (M, 1)))).astype(np.float32)
    q = rng.integers(-128, 128, (N, K)).astype(np.int8)
    s = rng.uniform(1e-4, 1e-3, N).astype(np.float32)
    b = rng.normal(0, 1, N).astype(np.float32) if bias else None
    want = (x.astype(np.float64) @ q.astype(np.float64).T) * s + (0 if b is None else b)
    err = rel_err(_run(lib, x, q, s, b), want)
    assert err <= 2e-6


def test_w8_batch_every_bit_of_an_activation_counts(lib):
    """One nonzero activation per row: the product with +-1 is the fp32 value itself."""
    print("[gpu] w8 batch single activations", flush=True)
    K, M = 256, 64
    rng = np.random.default_rng(3)
    bits = rng.integers(1, 0x7F800000, M).astype(np.uint32)     # magnitudes of every size
    bits[4:24] = rng.integers(1, 1 << 25, 20)                   # subnormal and nearly so
    bits[24:48] = rng.integers(1 << 25, 1 << 28, 24)            # up to 2^-95
    vals = bits.view(np.float32)
    vals[:4] = [1.0 + 2.0**-23, -(2.0 - 2.0**-23), 3.4028234663852886e38, -0.0]
    x = np.zeros((M, K), np.float32)
    x[np.arange(M), rng.integers(0, K, M)] = vals
    q = np.where(np.arange(2)[:, None] == 0, 1, -1).astype(np.int8) * np.ones((2, K), np.int8)
    y = _run(lib, x, q, np.ones(2, np.float32))
    assert np.array_equal(y[:, 0], vals) and np.array_equal(y[:, 1], -vals)


def test_w8_batch_non_finite_activations(lib):
    print("[gpu] w8 batch non-finite", flush=True)
    rng = np.random.default_rng(5)
    x = rng.normal(0, 1, (8, 512)).astype(np.float32)
    x[1, 100], x[2, 7], x[3, 500] = np.inf, -np.inf, np.nan
    x[4, 3] = np.uint32(0x7F800001).view(np.float32)        # a NaN whose leading half is an infinity
    q = rng.integers(1, 100, (40, 512)).astype(np.int8) * np.where(rng.random((40, 1)) < 0.5, -1, 1).astype(np.int8)
    y = _run(lib, x, q, np.ones(40, np.float32))
    with np.errstate(invalid="ignore"):
        want = x.astype(np.float64) @ q.astype(np.float64).T
    assert np.array_equal(np.isnan(y), np.isnan(want))
    assert np.array_equal(np.isinf(y), np.isinf(want))
    assert np.array_equal(np.sign(y[np.isinf(y)]), np.sign(want[np.isinf(want)]))
    fine = np.isfinite(want)
    assert rel_err(y[fine], want[fine]) <= 2e-6


@pytest.mark.parametrize("size", [1e-30, 1e-34, 1e-36, 1e-38, 1e-40])
def test_w8_batch_tiny_activations(lib, size):
    """Rows of a size where bf16 has few bits or none: the error of any other rows,
    and half a unit of the smallest fp32 for results that small."""
    print(f"[gpu] w8 batch activations of {size}", flush=True)
    rng = np.random.default_rng(11)
    x = (rng.normal(0, 1, (48, 2048)) * size).astype(np.float32)
    q = rng.integers(-128, 128, (300, 2048)).astype(np.int8)
    want = x.astype(np.float64) @ q.astype(np.float64).T
    y = _run(lib, x, q, np.ones(300, np.float32))
    assert np.abs(y - want).max() <= 2e-6 * np.abs(want).max() + 2.0**-149


@pytest.mark.parametrize("M,N,K", [
    (2, 300, 4096), (2, 4096, 4096), (2, 8193, 6144), (3, 8193, 3072), (3, 8192, 2816), (4, 9000, 2048), (4, 300, 2048),
    (5, 300, 260), (5, 8193, 20), (12, 200, 20), (5, 100, 1000),
])
def test_both_sides_of_the_rows_line(lib, M, N, K):
    test_w8_batch_matches_float64(lib, M, N, K, True, 0.0)
