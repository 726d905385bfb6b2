"""k_w4_awq_quantize_v8 (groups of 32, 64 and 128, weights on 16 bytes) against
the oracle, bit for bit: one group, rows that end inside a wave and inside a
workgroup's step of 2048, odd group counts; degenerate groups, NaN first and
inner elements, infinities, signed zeros, denormals.  Weights off 16 bytes take
the general kernel and must give the same."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("group", [32, 64, 128])
@pytest.mark.parametrize("N,G", [(1, 1), (5, 3), (9, 17), (3, 33), (2, 131)])
def test_bit_exact(lib, oracle, N, G, group):
    K = G * group
    print(f"[gpu] w4 awq v8 {N}x{K} g{group}", flush=True)
    rng = np.random.default_rng(N * 1000 + K)
    w = (rng.normal(0, 1, (N, G, group)) * 10.0 ** rng.integers(-9, 5, (N, G, 1))).astype(np.float32)
    if N > 1:
        w[1, 0] = 0.125
        w[1, 1, 0] = np.nan
        w[1, 2, 5] = np.nan
        w[0, 1, 7], w[0, 2, 3] = np.inf, -np.inf
        w[0, 0, ::3], w[0, 0, 1::3] = 0.0, -0.0
        w[N - 1, G - 1] = np.float32(1e-41) * rng.integers(-9, 9, group).astype(np.float32)
    w = w.reshape(N, K)
    with np.errstate(all="ignore"):
        rc, qwo, sco, qzo = oracle.w4_awq_quantize(w, group)
    off = torch.empty(N * K + 1, device=DEV)
    off[1:] = torch.from_numpy(w).to(DEV).reshape(-1)
    for wd in (torch.from_numpy(w).to(DEV), off[1:].reshape(N, K)):
        qw = torch.empty((N, K // 8), dtype=torch.int32, device=DEV)
        sc = torch.empty((N, G), dtype=torch.int16, device=DEV)
        qz = torch.empty((N, (G + 7) // 8), dtype=torch.int32, device=DEV)
        lib.dev_quantize_w4_awq(wd, qw, sc, qz, group)
        np.testing.assert_array_equal(qw.cpu().numpy().view(np.uint32), qwo)
        np.testing.assert_array_equal(sc.cpu().numpy().view(np.uint16), sco)
        np.testing.assert_array_equal(qz.cpu().numpy().view(np.uint32), qzo)
