"""W4A16 decode batches (k_w4a16_batch): rows at the edges of its 16, 32, 64
and 96 row blocks, column tails, one step to many spans of K, groups of 32 to
512, with and without zero points and bias, both output types, the SwiGLU
form and the allocation-free entry point.

The fp32 result is checked against the float64 product of the oracle's
dequantized weights.  Its sums run over at most 128 columns in one
accumulator, then over at most K / 128 scaled partial sums, each step an fp32
rounding (2^-24 of the running value, which stays below a few times the
result's size): 2e-6 of the largest result is over ten times the expected
random walk of them."""
import numpy as np
import pytest
import torch

from test_gpu_qlinear import DEV, TOL_BF16, bf16_bits, bf16_to_f32, rel_err, to_dev

pytestmark = pytest.mark.gpu


def _case(oracle, N, K, group, zeros, seed):
    """(device qweight, scales, qzeros), float64 weights."""
    rng = np.random.default_rng(seed)
    w = rng.normal(0, 0.02, (N, K)).astype(np.float32)
    rc, qw, sc, qz = oracle.w4_awq_quantize(w, group)
    assert rc == 0
    q = (qw[:, :, None] >> (4 * np.arange(8, dtype=np.uint32))) & 15
    z = ((qz[:, :, None] >> (4 * np.arange(8, dtype=np.uint32))) & 15).reshape(N, -1)[:, :K // group]
    if not zeros:
        z = np.full_like(z, 8)
    s = sc.view(np.float16).astype(np.float64)
    v = (q.reshape(N, K // group, group).astype(np.float64) - z[..., None].astype(np.float64)) * s[..., None]
    dev = (to_dev(qw.view(np.int32)), to_dev(sc.view(np.int16)), to_dev(qz.view(np.int32)) if zeros else None)
    return dev, v.reshape(N, K)


@pytest.mark.parametrize("M,N,K,group,zeros,bias,out", [
    (1, 40, 384, 128, True, False, "f32"),        # one row where the M = 1 kernels do not apply
    (1, 130, 256, 64, True, True, "bf16"),        # one row, small groups
    (2, 128, 128, 128, True, False, "f32"),       # a single step: one wave group has none
    (5, 38, 4224, 128, False, True, "f32"),       # 33 steps in spans of unlike length, column tail
    (5, 37, 4224, 128, True, False, "f32"),       # an odd number of scales
    (40, 1, 384, 128, False, False, "f32"),       # three scales
    (16, 300, 6144, 256, True, False, "bf16"),    # a full 16-row block, many spans
    (16, 65, 1152, 32, True, False, "f32"),
    (17, 129, 1152, 128, True, True, "f32"),      # one past a 16-row block
    (32, 256, 640, 64, False, False, "f32"),
    (33, 96, 2048, 128, True, False, "f32"),      # 64-row block with a tail
    (64, 1000, 512, 32, True, True, "bf16"),
    (65, 224, 4096, 512, True, False, "f32"),     # 96-row block with a tail
    (96, 136, 4096, 32, True, False, "f32"),
    (97, 200, 1536, 64, True, True, "f32"),       # two blocks
    (200, 72, 2560, 128, False, False, "bf16"),   # three blocks
    (300, 96, 1024, 128, True, False, "bf16"),    # more rows than 256, few columns
])
def test_w4_batch_matches_float64(lib, oracle, M, N, K, group, zeros, bias, out):
    print(f"[gpu] w4 batch M={M} N={N} K={K} g={group} zeros={zeros} bias={bias} out={out}", flush=True)
    (qw, sc, qz), v = _case(oracle, N, K, group, zeros, M * 131 + N)
    rng = np.random.default_rng(M + K)
    x = bf16_to_f32(bf16_bits(rng.normal(0.3, 1, (M, K)).astype(np.float32)))
    b = rng.normal(0, 1, N).astype(np.float32) if bias else None
    want = x.astype(np.float64) @ v.T + (0 if b is None else b.astype(np.float64))
    xd = to_dev(x).to(torch.bfloat16)
    bd = None if b is None else to_dev(b)
    dt = torch.float32 if out == "f32" else torch.bfloat16
    ys = []
    for call in (lib.qlinear_w4a16, lib.qlinear_w4a16, lib.qlinear_w4a16_noalloc):
        y = torch.full((M, N), float("nan"), dtype=dt, device=DEV)
        call(xd, qw, sc, qz, None, K // group, y, group, bias=bd)
        ys.append(y)
    torch.cuda.synchronize()
    err = rel_err(ys[0].float().cpu().numpy(), want)
    assert err <= (2e-6 if out == "f32" else TOL_BF16)
    # the spans' sums are added in span order, whoever arrives last
    assert torch.equal(ys[0], ys[1])
    if M < 256:
        assert torch.equal(ys[0], ys[2])


@pytest.mark.parametrize("M,F,K,group,zeros,bias", [
    (9, 64, 4096, 128, True, False),      # spans of K: gate and up meet in memory
    (16, 72, 256, 64, True, True),        # column tail of the 64-column tile
    (32, 8192, 512, 128, True, False),    # no spans: gate and up meet in LDS
    (50, 200, 1024, 32, False, True),
    (96, 136, 2048, 128, True, True),
])
def test_w4_batch_swiglu_matches_float64(lib, oracle, M, F, K, group, zeros, bias):
    print(f"[gpu] w4 batch swiglu M={M} F={F} K={K} g={group} zeros={zeros} bias={bias}", flush=True)
    (qw, sc, qz), v = _case(oracle, 2 * F, K, group, zeros, M + F)
    rng = np.random.default_rng(M * F)
    x = bf16_to_f32(bf16_bits(rng.normal(0, 1, (M, K)).astype(np.float32)))
    b = rng.normal(0, 0.5, 2 * F).astype(np.float32) if bias else None
    gu = x.astype(np.float64) @ v.T + (0 if b is None else b.astype(np.float64))
    want = gu[:, :F] / (1 + np.exp(-gu[:, :F])) * gu[:, F:]
    got = torch.full((M, F), float("nan"), dtype=torch.bfloat16, device=DEV)
    lib.qlinear_w4a16_swiglu(to_dev(x).to(torch.bfloat16), qw, sc, qz, got, group, bias=None if b is None else to_dev(b))
    torch.cuda.synchronize()
    err = rel_err(got.float().cpu().numpy(), want)
    assert err <= TOL_BF16


@pytest.mark.parametrize("M,N,K,group", [(6, 70, 512, 64), (16, 40, 2048, 32), (40, 130, 512, 32), (96, 100, 2048, 64)])
def test_w4_batch_small_groups_with_extreme_activations(lib, oracle, M, N, K, group):
    """Infinities, NaN and activations whose product with a bare code overflows: the
    result of sum x (q - z) s.  Terms are added one after the other: K roundings of
    2^-24 of the sum of their sizes."""
    print(f"[gpu] w4 batch extreme activations M={M} N={N} K={K} g={group}", flush=True)
    (qw, sc, qz), v = _case(oracle, N, K, group, True, M + group)
    x = bf16_to_f32(bf16_bits(np.random.default_rng(M).normal(0.3, 1, (M, K)).astype(np.float32)))
    x[1, 7], x[2, K - 1], x[3, 40], x[4, 9] = np.inf, -np.inf, np.nan, 2.0**127
    y = torch.full((M, N), 7.0, device=DEV)
    lib.qlinear_w4a16(to_dev(x).to(torch.bfloat16), qw, sc, qz, None, K // group, y, group)
    torch.cuda.synchronize()
    got = y.cpu().numpy().astype(np.float64)
    with np.errstate(invalid="ignore"):
        want = x.astype(np.float64) @ v.T
    assert np.isinf(want[1]).any() and np.isfinite(want[4]).all()
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isinf(got), np.isinf(want))
    assert np.array_equal(np.sign(got[np.isinf(got)]), np.sign(want[np.isinf(want)]))
    rows = np.isfinite(x).all(axis=1)
    size = np.abs(x[rows]).astype(np.float64) @ np.abs(v).T
    assert float((np.abs(got[rows] - want[rows]) / size).max()) <= K * 2.0**-24
