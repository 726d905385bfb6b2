"""W4A16 linears with little to stream, at the lines between the decode GEMV or
split-K and the batch kernel: both sides of each line give the float64 product.
The GEMVs and split-K add x (128 + q) over a group of 128 columns, take (128 + z)
times the sum of x off and add the scaled groups: at most 128 + K / 128 + 4 roundings
of 2^-24 of sums that stay below sum |x| (143 + 143) s."""
import numpy as np
import pytest
import torch

from test_gpu_qlinear import DEV, bf16_bits, bf16_to_f32, to_dev
from test_gpu_w4_batch import _case, test_w4_batch_swiglu_matches_float64 as swiglu_matches_float64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [
    (19, 10240, 512), (20, 8208, 512), (18, 8192, 1536), (32, 100, 1024), (28, 60, 2048), (29, 60, 2048), (32, 4096, 1536), (32, 4100, 1536),
    (48, 8192, 512), (49, 4096, 512), (64, 200, 512), (65, 200, 512), (48, 300, 1024), (49, 300, 1024),
    (2, 1024, 7168), (16, 2048, 7168), (16, 2049, 7168), (9, 2048, 8192), (5, 1023, 7168), (3, 1536, 8192),
])
def test_both_sides_of_the_short_lines(lib, oracle, M, N, K):
    print(f"[gpu] w4 short M={M} N={N} K={K}", flush=True)
    (qw, sc, qz), v = _case(oracle, N, K, 128, True, M + N)
    x = bf16_to_f32(bf16_bits(np.random.default_rng(M + K).normal(0.3, 1, (M, K)).astype(np.float32)))
    xd = to_dev(x).to(torch.bfloat16)
    want = x.astype(np.float64) @ v.T
    s = np.repeat(sc.cpu().numpy().view(np.float16).astype(np.float64), 128, axis=1)
    bound = (128 + K / 128 + 4) * 2.0**-24 * 286 * (np.abs(x).astype(np.float64) @ s.T)
    ys = []
    for call in (lib.qlinear_w4a16, lib.qlinear_w4a16_noalloc):
        y = torch.full((M, N), float("nan"), device=DEV)
        call(xd, qw, sc, qz, None, K // 128, y, 128)
        torch.cuda.synchronize()
        assert (np.abs(y.cpu().numpy() - want) <= bound).all()
        ys.append(y)
    assert torch.equal(*ys)


@pytest.mark.parametrize("M,N,K", [(8, 33000, 640), (16, 32768, 640), (17, 33000, 640), (1, 33000, 640)])
def test_more_columns_than_a_round_of_the_cus(lib, oracle, M, N, K):
    test_both_sides_of_the_short_lines(lib, oracle, M, N, K)


@pytest.mark.parametrize("M,F,K", [
    (9, 6144, 1024), (9, 6152, 1024), (16, 5128, 2048), (16, 5120, 2048), (12, 12296, 3072), (12, 12288, 3072),
    (16, 16392, 1024), (2, 4992, 1536), (2, 5000, 1536), (3, 4000, 2560), (4, 4000, 2560), (9, 16392, 640),
])
def test_both_sides_of_the_swiglu_lines(lib, oracle, M, F, K):
    swiglu_matches_float64(lib, oracle, M, F, K, 128, True, False)
