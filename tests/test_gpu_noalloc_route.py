"""The allocation-free W4A16 entry point runs the prefill GEMM whole-K, so it takes
it only where that is the faster kernel: between the decode batches and the full
GEMM tiles it stays near the allocating entry point, which may split K (N = 4096,
K = 14336, M = 193: 66 us both; the GEMM whole-K 173)."""
import pytest
import torch

from test_zz_no_alloc import DEV, _layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(193, 4096, 14336), (255, 4096, 14336), (200, 2048, 8192)])
def test_noalloc_is_priced_whole_k(lib, M, N, K):
    print(f"[gpu] noalloc route M={M} N={N} K={K}", flush=True)
    qw, sc, qz, G = _layer(lib, N, K, 3)
    x = torch.randn((M, K), device=DEV, generator=torch.Generator(device=DEV).manual_seed(4)).to(torch.bfloat16)
    us, ys = [], []
    for call in (lib.qlinear_w4a16, lib.qlinear_w4a16_noalloc):
        y = torch.full((M, N), 7, dtype=torch.bfloat16, device=DEV)
        best = float("inf")
        for _ in range(8):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(10):
                call(x, qw, sc, qz, None, G, y, 128)
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b) * 100)
        us.append(best)
        ys.append(y.float())
    print(f"[gpu] {us[0]:.1f} us, allocation-free {us[1]:.1f} us", flush=True)
    assert float((ys[0] - ys[1]).abs().max() / ys[0].abs().max()) <= 1e-2
    assert us[1] <= 2 * us[0]
