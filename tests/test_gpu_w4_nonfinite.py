"""W4A16 linears of several rows whose activations hold infinities, NaN and values
whose product with a bare code overflows: the results of sum x (q - z) s, as the
kernels of these shapes (groups of 128 and more with K in no whole 512s, single
rows of few columns, groups of 32 and 64) always gave them, and in bounded time.

Finite results: terms of a group and then the groups' sums are added one after the
other, K roundings of 2^-24 of the sum of the terms' sizes; bf16 adds 2^-8."""
import numpy as np
import pytest
import torch

from test_gpu_qlinear import DEV, bf16_bits, bf16_to_f32, to_dev
from test_gpu_w4_batch import _case

pytestmark = pytest.mark.gpu


def _rows(M, K, big=True):
    x = bf16_to_f32(bf16_bits(np.random.default_rng(M).normal(0.3, 1, (M, K)).astype(np.float32)))
    bad = [(0, 7, np.inf), (M // 4, K - 1, -np.inf), (M // 2, 40, np.nan), (M - 1, 9, 2.0**127 if big else np.inf)]
    for m, k, v in bad:
        x[m, k] = v
    return x


def _same(got, want, bound):
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isinf(got), np.isinf(want))
    assert np.array_equal(np.sign(got[np.isinf(got)]), np.sign(want[np.isinf(want)]))
    ok = np.isfinite(want)
    assert (np.abs(got[ok] - want[ok]) <= bound[ok]).all()


@pytest.mark.parametrize("M,N,K,group,out", [
    (1, 130, 384, 128, "f32"),
    (5, 40, 4224, 128, "f32"),        # 33 groups: the last scale by itself
    (17, 70, 1408, 128, "f32"),
    (40, 257, 11008, 128, "bf16"),    # spans of K, a column tail
    (64, 100, 1408, 128, "bf16"),     # bf16 from 64 rows on
    (96, 300, 640, 128, "f32"),
    (200, 72, 11008, 128, "bf16"),
    (250, 2000, 1408, 128, "bf16"),
    (33, 96, 768, 256, "f32"),
    (300, 40, 1408, 128, "f32"),      # more than 255 rows
    (96, 136, 2048, 64, "f32"),
    (97, 64, 1152, 32, "bf16"),
])
def test_nonfinite_activations(lib, oracle, M, N, K, group, out):
    print(f"[gpu] w4 non-finite activations M={M} N={N} K={K} g={group} {out}", flush=True)
    (qw, sc, qz), v = _case(oracle, N, K, group, True, M + group)
    if M == 1:
        x = _rows(4, K)[:1]
    else:
        x = _rows(M, K)
    xd = to_dev(x).to(torch.bfloat16)
    dt = torch.float32 if out == "f32" else torch.bfloat16
    with np.errstate(invalid="ignore"):
        want = x.astype(np.float64) @ v.T
        size = np.abs(x).astype(np.float64) @ np.abs(v).T
        bound = K * 2.0**-24 * size + (0 if out == "f32" else 2.0**-8 * np.abs(want))
    assert np.isinf(want).any()
    for call in (lib.qlinear_w4a16, lib.qlinear_w4a16_noalloc):
        y = torch.full((M, N), 7.0, dtype=dt, device=DEV)
        call(xd, qw, sc, qz, None, K // group, y, group)
        torch.cuda.synchronize()
        _same(y.float().cpu().numpy().astype(np.float64), want, bound)


@pytest.mark.parametrize("M,F,K,group", [
    (9, 64, 4224, 128),       # spans of K: gate and up meet in memory
    (32, 8192, 384, 128),     # no spans: in LDS
    (96, 136, 1408, 64),
])
def test_nonfinite_activations_swiglu(lib, oracle, M, F, K, group):
    print(f"[gpu] w4 swiglu non-finite activations M={M} F={F} K={K} g={group}", flush=True)
    (qw, sc, qz), v = _case(oracle, 2 * F, K, group, True, M + F)
    x = _rows(M, K, big=False)
    with np.errstate(invalid="ignore", over="ignore"):
        gu = x.astype(np.float64) @ v.T
        g, u = gu[:, :F], gu[:, F:]
        want = g * u / (1 + np.exp(-g))
    got = torch.full((M, F), 7.0, dtype=torch.bfloat16, device=DEV)
    lib.qlinear_w4a16_swiglu(to_dev(x).to(torch.bfloat16), qw, sc, qz, got, group)
    torch.cuda.synchronize()
    assert np.isinf(want).any()
    # g and u of K = 4096 are a few units in size: 2^-8 of the product, and of 1
    _same(got.float().cpu().numpy().astype(np.float64), want, 2.0**-7 * np.abs(np.nan_to_num(want)) + 2.0**-10)


def test_nonfinite_rows_cost_a_bounded_time(lib):
    """One row with a NaN, as an uninitialised padding row may hold, and all rows
    with an infinity: well below the generic kernel's 2.7 ms (0.3 and 0.5)."""
    M, N, K, group = 96, 6144, 4096, 64
    print(f"[gpu] w4 non-finite rows' time M={M} N={N} K={K} g={group}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(1)
    w = torch.randn((N, K), device=DEV, generator=g) * 0.02
    qw = torch.empty((N, K // 8), dtype=torch.int32, device=DEV)
    sc = torch.empty((N, K // group), dtype=torch.int16, device=DEV)
    qz = torch.empty((N, (K // group + 7) // 8), dtype=torch.int32, device=DEV)
    lib.dev_quantize_w4_awq(w, qw, sc, qz, group)
    y = torch.empty((M, N), dtype=torch.bfloat16, device=DEV)
    for rows, value in ((slice(3, 4), float("nan")), (slice(0, M), float("inf"))):
        x = torch.randn((M, K), device=DEV, generator=g)
        x[rows, 5] = value
        x = x.to(torch.bfloat16)
        ms = []
        for _ in range(4):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            lib.qlinear_w4a16(x, qw, sc, qz, None, K // group, y, group)
            b.record()
            torch.cuda.synchronize()
            ms.append(a.elapsed_time(b))
        print(f"[gpu] {value}: {min(ms):.2f} ms", flush=True)
        assert min(ms) < 2.0
