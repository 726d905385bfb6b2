"""W4A16 linears of several rows, groups of 32 and 64, whose activations hold
infinities or NaN: computed in bounded time."""
import pytest
import torch

from test_gpu_qlinear import DEV

pytestmark = pytest.mark.gpu


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
