"""SNEPPX_qlinear_noalloc_reset: ordered between two calls in K spans it changes
nothing, eagerly and in a recorded step, and it needs no call before it."""
import pytest
import torch

from test_zz_no_alloc import DEV, _layer

pytestmark = pytest.mark.gpu


def test_reset_between_calls(lib):
    M, N, K = 32, 1000, 4096
    print(f"[gpu] noalloc reset M={M} N={N} K={K}", flush=True)
    s = torch.cuda.Stream()
    st = s.cuda_stream
    qw, sc, qz, G = _layer(lib, N, K, 3)
    x = torch.randn((M, K), device=DEV, generator=torch.Generator(device=DEV).manual_seed(4)).to(torch.bfloat16)
    want = torch.empty((M, N), dtype=torch.bfloat16, device=DEV)
    ys = [torch.empty_like(want) for _ in range(2)]
    lib.qlinear_noalloc_reset()
    lib.qlinear_w4a16(x, qw, sc, qz, None, G, want, 128)
    torch.cuda.synchronize()

    def step():
        for y in ys:
            lib.qlinear_w4a16_noalloc(x, qw, sc, qz, None, G, y, 128, stream=st)
            lib.qlinear_noalloc_reset(stream=st)

    step()
    s.synchronize()
    assert all(torch.equal(y, want) for y in ys)
    graph = lib.capture(step, st)
    try:
        for _ in range(3):
            with torch.cuda.stream(s):
                for y in ys:
                    y.fill_(float("nan"))
            lib.graph_launch(graph, st)
            s.synchronize()
            assert all(torch.equal(y, want) for y in ys)
    finally:
        lib.graph_destroy(graph)
