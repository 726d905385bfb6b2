"""Linears with several rows recorded into a graph on a stream that has not run
them: the recorded call takes no workspace (which other calls and replays would
share), before and after an eager call on the same
stream, and every replay gives the float64 product."""
import numpy as np
import pytest
import torch

from test_gpu_q8_batch import oracle_e4m3
from test_gpu_qlinear import DEV, TOL_BF16, bf16_bits, bf16_to_f32, rel_err, to_dev
from test_gpu_w4_batch import _case

pytestmark = pytest.mark.gpu


def _w4(lib, oracle, M, N, K, group):
    (qw, sc, qz), v = _case(oracle, N, K, group, True, M + N)
    x = bf16_to_f32(bf16_bits(np.random.default_rng(M).normal(0.3, 1, (M, K)).astype(np.float32)))
    y = torch.empty((M, N), dtype=torch.bfloat16, device=DEV)
    xd = to_dev(x).to(torch.bfloat16)
    return y, x.astype(np.float64) @ v.T, lambda st: lib.qlinear_w4a16(xd, qw, sc, qz, None, K // group, y, group, stream=st)


def _w8(lib, oracle, M, N, K, group):
    rng = np.random.default_rng(M)
    x, q = rng.normal(0, 1, (M, K)).astype(np.float32), rng.integers(-128, 128, (N, K)).astype(np.int8)
    s = rng.uniform(1e-4, 1e-3, N).astype(np.float32)
    xd, qd, sd = to_dev(x), to_dev(q), to_dev(s)
    y = torch.empty((M, N), device=DEV)
    return y, (x.astype(np.float64) @ q.T.astype(np.float64)) * s, lambda st: lib.qlinear_w8_gemv(xd, qd, sd, y, stream=st)


def _i8(lib, oracle, M, N, K, group):
    rng = np.random.default_rng(M)
    a, w = (rng.integers(-128, 128, s).astype(np.int8) for s in ((M, K), (N, K)))
    sa, sw = rng.uniform(1e-3, 1e-2, M).astype(np.float32), rng.uniform(1e-3, 1e-2, N).astype(np.float32)
    d = [to_dev(t) for t in (a, sa, w, sw)]
    y = torch.empty((M, N), dtype=torch.bfloat16, device=DEV)
    return y, (a.astype(np.float64) @ w.T.astype(np.float64)) * sa[:, None] * sw, lambda st: lib.qlinear_w8a8_i8(*d, y, stream=st)


def _f8(lib, oracle, M, N, K, group):
    rng = np.random.default_rng(M)
    a, w = (rng.integers(1, 0x78, s).astype(np.uint8) | (rng.integers(0, 2, s).astype(np.uint8) << 7) for s in ((M, K), (N, K)))
    dec = np.array([oracle_e4m3(c) for c in range(256)])
    s = np.array([0.01], np.float32)
    d = [to_dev(t) for t in (a, s, w, s)]
    y = torch.empty((M, N), dtype=torch.bfloat16, device=DEV)
    return y, (dec[a] @ dec[w].T) * float(s[0]) ** 2, lambda st: lib.qlinear_w8a8_fp8(*d, y, stream=st)


@pytest.mark.parametrize("make,M,N,K,group", [
    (_w4, 32, 300, 4096, 128),      # decode GEMV slices
    (_w4, 96, 200, 2048, 128),      # a smaller prefill GEMM is no choice either
    (_w4, 8, 100, 2048, 64),        # the generic kernel
    (_w4, 1, 130, 2048, 64),
    (_w8, 16, 257, 4096, 0),
    (_i8, 40, 200, 4096, 0),
    (_f8, 40, 200, 4096, 0),
], ids=lambda v: getattr(v, "__name__", str(v)))
def test_recorded_rows_take_no_workspace(lib, oracle, make, M, N, K, group):
    print(f"[gpu] recorded rows {make.__name__} M={M} N={N} K={K} g={group}", flush=True)
    s = torch.cuda.Stream()
    st = s.cuda_stream
    y, want, call = make(lib, oracle, M, N, K, group)
    torch.cuda.synchronize()
    count = lib.fn["snx_workspace_count"]
    before = count()
    graph = lib.capture(lambda: call(st), st)
    try:
        assert count() == before
        bits = None
        for _ in range(3):
            with torch.cuda.stream(s):
                y.fill_(float("nan"))
            lib.graph_launch(graph, st)
            s.synchronize()
            assert rel_err(y.float().cpu().numpy(), want) <= (2e-6 if y.dtype == torch.float32 else TOL_BF16)
            assert bits is None or torch.equal(y, bits)
            bits = y.clone()
            call(st)                # eager, the batch kernel, between the replays
            s.synchronize()
            assert rel_err(y.float().cpu().numpy(), want) <= (2e-6 if y.dtype == torch.float32 else TOL_BF16)
    finally:
        lib.graph_destroy(graph)
        lib.fn["SNEPPX_qlinear_release_workspaces"](st)
        s.synchronize()
