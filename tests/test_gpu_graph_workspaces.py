"""Linears whose recorded call takes a workspace that their eager call, on the
batch kernels, does not: W4A16 split-K, the SwiGLU and MLP blocks, a prefill GEMM
in K spans, a W8A8 GEMM in K spans.  Recorded with and without an eager call
before, with an eager call and a larger one (which needs larger workspaces)
between the capture and the replays: every replay gives the same bits, and they
and the eager results are the float64 product; and eager calls go on working when
the graph is gone."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _w4(lib, N, K, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    w = torch.randn((N, K), device=DEV, generator=g) * 0.02
    G = K // 128
    qw = torch.empty((N, K // 8), dtype=torch.int32, device=DEV)
    sc = torch.empty((N, G), dtype=torch.int16, device=DEV)
    qz = torch.empty((N, (G + 7) // 8), dtype=torch.int32, device=DEV)
    lib.dev_quantize_w4_awq(w, qw, sc, qz, 128)
    sh = 4 * torch.arange(8, device=DEV, dtype=torch.int32)
    q = ((qw[..., None] >> sh) & 15).reshape(N, G, 128).double()
    z = ((qz[..., None] >> sh) & 15).reshape(N, -1)[:, :G].double()
    return (qw, sc, qz), ((q - z[..., None]) * sc.view(torch.float16).double()[..., None]).reshape(N, K)


def _x(M, K, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn((M, K), device=DEV, generator=g).to(torch.bfloat16)


def _linear(lib, M, N, K):
    w, v = _w4(lib, N, K, N)
    x, y = _x(M, K, M), torch.empty((M, N), dtype=torch.bfloat16, device=DEV)
    return y, x.double() @ v.t(), lambda st: lib.qlinear_w4a16(x, *w, None, K // 128, y, 128, stream=st)


def _silu_rows(v, x):
    gu = x.double() @ v.t()
    F = v.shape[0] // 2
    return torch.nn.functional.silu(gu[:, :F]) * gu[:, F:]


def _swiglu(lib, M, F, K):
    w, v = _w4(lib, 2 * F, K, F)
    x, y = _x(M, K, M), torch.empty((M, F), dtype=torch.bfloat16, device=DEV)
    return y, _silu_rows(v, x), lambda st: lib.qlinear_w4a16_swiglu(x, *w, y, 128, stream=st)


def _mlp(lib, M, F, K):
    (gu, v), (dn, vd) = _w4(lib, 2 * F, K, F), _w4(lib, K, F, F + 1)
    x, y = _x(M, K, M), torch.empty((M, K), dtype=torch.bfloat16, device=DEV)
    return y, _silu_rows(v, x) @ vd.t(), lambda st: lib.qlinear_w4a16_mlp(x, gu, dn, y, 128, stream=st)


def _i8(lib, M, N, K):
    g = torch.Generator(device=DEV).manual_seed(M)
    a, w = (torch.randint(-128, 128, s, device=DEV, generator=g).to(torch.int8) for s in ((M, K), (N, K)))
    sa, sw = (torch.rand(n, device=DEV, generator=g) * 1e-2 + 1e-3 for n in (M, N))
    y = torch.empty((M, N), dtype=torch.bfloat16, device=DEV)
    want = (a.double() @ w.double().t()) * sa.double()[:, None] * sw.double()
    return y, want, lambda st: lib.qlinear_w8a8_i8(a, sa, w, sw, y, stream=st)


@pytest.mark.parametrize("warmed", [False, True], ids=["cold", "warmed"])
@pytest.mark.parametrize("make,shape,larger", [
    (_linear, (16, 2048, 14336), (16, 4096, 14336)),    # split-K partials
    (_swiglu, (32, 1024, 2048), (32, 4096, 2048)),      # the projection's fp32 rows
    (_mlp, (32, 1024, 2048), (32, 4096, 2048)),
    (_linear, (512, 1024, 4096), (1024, 1024, 4096)),   # prepared activations, spans and counters
    (_i8, (2048, 1792, 4096), (2048, 3584, 4096)),      # spans and counters
], ids=lambda v: getattr(v, "__name__", None))
def test_recorded_call_with_a_workspace(lib, make, shape, larger, warmed):
    print(f"[gpu] recorded call with a workspace {make.__name__} {shape} warmed={warmed}", flush=True)
    s = torch.cuda.Stream()
    st = s.cuda_stream
    y, want, call = make(lib, *shape)
    y2, want2, call2 = make(lib, *larger)
    torch.cuda.synchronize()

    def check(got, ref):        # one bf16 rounding, in a block of the first product's too
        assert float((got.double() - ref).norm() / ref.norm()) <= 4e-3

    def eager(f, out, ref):
        with torch.cuda.stream(s):
            out.fill_(float("nan"))
        f(st)
        s.synchronize()
        check(out, ref)

    if warmed:
        eager(call, y, want)
    graph = lib.capture(lambda: call(st), st)
    bits = None
    try:
        for rep in range(4):
            if rep < 2:
                eager(call, y, want)          # also between the capture and the first replay
            if rep == 1:
                eager(call2, y2, want2)
            with torch.cuda.stream(s):
                y.fill_(float("nan"))
            lib.graph_launch(graph, st)
            s.synchronize()
            check(y, want)
            assert bits is None or torch.equal(y, bits), rep
            bits = y.clone()
    finally:
        lib.graph_destroy(graph)
    eager(call, y, want)
    eager(call2, y2, want2)
    lib.fn["SNEPPX_qlinear_release_workspaces"](st)
    s.synchronize()


def test_torch_graph_takes_its_workspaces_apart(lib):
    """The same under torch.cuda.graph, whose capture refuses allocations of every
    thread that has not relaxed its own mode, on a stream that has run nothing."""
    print("[gpu] torch graph: split-K, SwiGLU block, GEMM in spans", flush=True)
    s = torch.cuda.Stream()
    made = [_linear(lib, 16, 2048, 14336), _mlp(lib, 32, 1024, 2048), _linear(lib, 512, 1024, 4096)]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        for _, _, call in made:
            call(s.cuda_stream)
    for rep in range(3):
        with torch.cuda.stream(s):
            for y, _, _ in made:
                y.fill_(float("nan"))
            if rep == 1:
                for _, _, call in made:
                    call(s.cuda_stream)         # eagerly, in the same workspaces
            graph.replay()
        s.synchronize()
        for y, want, _ in made:
            assert float((y.double() - want).norm() / want.norm()) <= 4e-3
    del graph
    lib.fn["SNEPPX_qlinear_release_workspaces"](s.cuda_stream)
    s.synchronize()
