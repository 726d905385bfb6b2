"""k_mx_quant32 (whole aligned blocks of 32) against the oracle
(oracle/mx_oracle.py), bit for bit: every binade of block peaks from the
smallest denormal to the largest finite value with the significands around the
formats' largest element, elements halfway between two codes at every distance
below the peak, zeros of both signs, non-finite blocks, and the sizes around a
workgroup's 64 blocks.  Rows that start off 16 bytes take the general kernel
and must give the same codes.  Blocks whose peak is within 2^-12 of the largest
element times a power of two are only held against that kernel: the oracle takes
numpy's float32 log2 there, whose last bits (2^-16 at |log2| = 149, a few of
them by CPU) decide the scale."""
import numpy as np
import pytest
import torch

import mx_oracle as mx

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _blocks(rng, n):
    e = np.arange(n) % 278 - 149                       # binade of the block's peak
    man = rng.choice(np.array([0, 0x400000, 0x600000, 0x700000, 0x5fffff, 0x600001, 0x6fffff, 0x700001, 0x7fffff,
                               0x3fffff, 0x400001, 0x123456], np.uint32), n)
    # element = sign, 0..23 binades below the peak, few significant bits (codes and their halves)
    down = rng.integers(0, 24, (n, 32))
    down[:, 5] = 0
    frac = 1.0 + rng.integers(0, 64, (n, 32)) / 64.0
    frac[:, 5] = 1.0 + man / 2.0 ** 23
    with np.errstate(over="ignore", under="ignore"):
        x = np.ldexp(frac, e[:, None] - down).astype(np.float32)
    x = np.where(np.isfinite(x), x, np.float32(3.4028234663852886e38))
    x *= np.where(rng.integers(0, 2, x.shape), np.float32(1), np.float32(-1))
    x[rng.random(x.shape) < 0.05] = 0.0
    x[rng.random(x.shape) < 0.02] = -0.0
    return x


@pytest.mark.parametrize("fmt", ["mxfp8_e4m3", "mxfp8_e5m2", "mxfp6_e3m2", "mxfp6_e2m3", "mxfp4_e2m1"])
@pytest.mark.parametrize("rows,cols", [(1, 32), (7, 288), (64, 32), (65, 32), (417, 96)])
def test_blocks_of_32_bit_exact(lib, fmt, rows, cols):
    print(f"[gpu] mx32 {fmt} {rows}x{cols}", flush=True)
    rng = np.random.default_rng(rows * 1000 + cols)
    x = _blocks(rng, rows * cols // 32)
    if rows > 1:
        x[1, 3], x[2, 9], x[3, 31], x[4] = np.nan, np.inf, -np.inf, 0.0
    x = x.reshape(rows, cols)
    po, so = mx.quantize(x, fmt, 32)
    po, so = po.reshape(-1, po.size // (rows * cols // 32)), so.ravel()
    with np.errstate(invalid="ignore"):
        man = np.frexp(np.abs(x.reshape(-1, 32)).max(axis=1).astype(np.float64))[0] * 2
    clear = ~(np.abs(man - (2.0 - 2.0 ** -int(fmt[-1]))) < 2.0 ** -12)   # m mantissa bits: 2 - 2^-m
    off = torch.empty(rows * cols + 1, device=DEV)
    off[1:] = torch.from_numpy(x).to(DEV).reshape(-1)
    got = []
    for xd in (torch.from_numpy(x).to(DEV), off[1:].reshape(rows, cols)):
        packed, scales = lib.dev_quantize_mx(xd, fmt, 32)
        got.append((packed.cpu().numpy().reshape(po.shape), scales.cpu().numpy().ravel()))
    for a, b in zip(*got):
        np.testing.assert_array_equal(a, b)
    np.testing.assert_array_equal(got[0][0][clear], po[clear])
    np.testing.assert_array_equal(got[0][1][clear], so[clear])
