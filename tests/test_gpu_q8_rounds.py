"""MX linears of 33 to 127 rows on both sides of the line between the batch kernel
and the large tiles: where the large tiles are half the rounds of the CUs, and where
both are as many."""
import pytest

from test_gpu_q8_batch import test_mx_rows_match_float64 as check_rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", ["mxfp8_e4m3", "mxfp6_e2m3"])
@pytest.mark.parametrize("M,N,K", [(33, 33000, 128), (32, 33000, 128), (40, 57350, 128), (64, 32768, 128)])
def test_both_sides_of_the_rounds_line(lib, fmt, M, N, K):
    check_rows(lib, fmt, M, N, K, "bf16")
