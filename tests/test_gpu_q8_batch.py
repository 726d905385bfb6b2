"""Low-precision linears with few rows (k_q8_batch): rows at the edges of its
32, 64 and 128 row blocks, column tails, widths that end inside a step, one
span of K and many, for int8, fp8 and the MX formats.

int8 sums are exact, so without a bias the outputs are those of the float64
product rounded where the epilogue rounds (fp32, then bf16): bit-equal to it.  fp8 and MX are
held to the tolerances of their other tests."""
import numpy as np
import pytest
import torch

from test_gpu_mx import _mfma_values
from test_gpu_qlinear import DEV, TOL_BF16, rel_err, to_dev

pytestmark = pytest.mark.gpu

SHAPES = [
    (1, 1, 128), (31, 129, 256), (33, 300, 384), (64, 128, 4096), (65, 1000, 640), (127, 130, 1024),
    (130, 257, 14336), (200, 2000, 512), (300, 640, 2048),
]


@pytest.mark.parametrize("M,N,K", SHAPES + [(5, 70, 16), (40, 200, 1040), (129, 300, 4064), (17, 513, 144)])
@pytest.mark.parametrize("bias", [False, True])
def test_int8_rows_equal_the_exact_product(lib, M, N, K, bias):
    print(f"[gpu] q8 batch int8 M={M} N={N} K={K} bias={bias}", flush=True)
    rng = np.random.default_rng(M + N + K)
    A, W = (rng.integers(-128, 128, s).astype(np.int8) for s in ((M, K), (N, K)))
    sA, sW = rng.uniform(1e-3, 1e-2, M).astype(np.float32), rng.uniform(1e-3, 1e-2, N).astype(np.float32)
    b = rng.normal(0, 5, N).astype(np.float32) if bias else None
    out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
    lib.qlinear_w8a8_i8(to_dev(A), to_dev(sA), to_dev(W), to_dev(sW), out, bias=None if b is None else to_dev(b))
    torch.cuda.synchronize()
    acc = A.astype(np.float64) @ W.astype(np.float64).T               # exact: below 2^53
    want = (acc.astype(np.float32) * sA[:, None]) * sW
    if bias:
        # the add may be fused with the last product: half a bf16 unit of the
        # result, and fp32 roundings (2^-24) of the product and of the sum
        got, size, want = out.float().cpu().numpy(), np.abs(want) + np.abs(b), want + b
        worst = float((np.abs(got - want) / (2.0 ** -8 * np.abs(want) + 2.0 ** -22 * size)).max())
        assert worst <= 1
    else:
        assert torch.equal(out.cpu(), torch.from_numpy(want).to(torch.bfloat16))


@pytest.mark.parametrize("M,N,K", SHAPES + [(40, 200, 1056), (129, 300, 4064)])
def test_fp8_rows_match_float64(lib, oracle, M, N, K):
    print(f"[gpu] q8 batch fp8 M={M} N={N} K={K}", flush=True)
    rng = np.random.default_rng(M * N + K)
    A, W = (rng.integers(0, 0x78, s).astype(np.uint8) | (rng.integers(0, 2, s).astype(np.uint8) << 7) for s in ((M, K), (N, K)))
    A[A == 0x80] = 0
    W[W == 0x80] = 0
    dec = np.array([oracle_e4m3(c) for c in range(256)])
    sA, sW = np.float32(0.01), np.float32(0.003)
    out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
    lib.qlinear_w8a8_fp8(to_dev(A), to_dev(np.array([sA])), to_dev(W), to_dev(np.array([sW])), out)
    torch.cuda.synchronize()
    want = (dec[A] @ dec[W].T) * sA * sW
    err = rel_err(out.float().cpu().numpy(), want)
    assert err <= TOL_BF16


def oracle_e4m3(c):
    """Value of an E4M3 code below the all-ones exponent (codes with exponent field
    0 are subnormals on the matrix cores)."""
    e, m = (c >> 3) & 15, c & 7
    v = m * 2.0**-9 if e == 0 else (1 + m / 8) * 2.0**(e - 7)
    return -v if c & 0x80 else v


@pytest.mark.parametrize("fmt", ["mxfp8_e4m3", "mxfp8_e5m2", "mxfp6_e3m2", "mxfp6_e2m3", "mxfp4_e2m1"])
@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("out", ["bf16", "f32"])
def test_mx_rows_match_float64(lib, fmt, M, N, K, out):
    print(f"[gpu] q8 batch {fmt} M={M} N={N} K={K} out={out}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    # block magnitudes far apart, so a block scaled by another's exponent shows
    x = torch.randn((M, K), device=DEV, generator=g) * torch.exp2(torch.randint(-6, 7, (M, K // 32), device=DEV, generator=g).float()).repeat_interleave(32, 1)
    w = torch.randn((N, K), device=DEV, generator=g) * torch.exp2(torch.randint(-6, 7, (N, K // 32), device=DEV, generator=g).float()).repeat_interleave(32, 1)
    (a, sa), (b, sb) = lib.dev_quantize_mx(x, fmt), lib.dev_quantize_mx(w, fmt)
    y = torch.full((M, N), float("nan"), dtype=torch.float32 if out == "f32" else torch.bfloat16, device=DEV)
    lib.qlinear_mx_gemm(a, sa, b, sb, fmt, y, M, N, K)
    torch.cuda.synchronize()
    va, vb = (_mfma_values(p.cpu().numpy(), s.cpu().numpy(), r, K, fmt) for p, s, r in ((a, sa, M), (b, sb, N)))
    want, size = va @ vb.T, np.abs(va) @ np.abs(vb).T
    got = y.float().cpu().numpy().astype(np.float64)
    # the matrix cores keep about 16 bits relative to the sum of |products|
    # (test_gpu_mx.py); bf16 adds half a unit of its 8 bits
    bound = 2.0 ** -13 * size + (2.0 ** -8 * np.abs(want) if out == "bf16" else 0)
    worst = float((np.abs(got - want) / np.maximum(bound, 1e-300)).max())
    assert worst <= 1
