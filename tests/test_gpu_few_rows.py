"""GPU tests of the products with at most 16 rows (gemm_rows_kernel).

Bound: a lane adds 4 products for each of its ceil(K / 256) steps at most, six
shuffle steps, three sums of waves and the bias follow, each rounding once
relative to partial sums that never exceed sum |a b|:
|got - exact| <= (4 ceil(K / 256) + 12) 2^-24 sum |a b|.
"""
from __future__ import annotations

import numpy as np
import pytest

import abi_ops as G
from cdml import synth

pytestmark = pytest.mark.gpu

# in, out: K below, at and past one step of 256, one round of four steps with KS = 1 (1024) and with KS = 4
# (4096) and their neighbours; odd output counts; more outputs than leave CUs idle (2048 and above)
SHAPES = [(4, 1), (252, 7), (256, 64), (260, 64), (516, 5), (1020, 130), (1024, 1024), (1028, 33), (3076, 50),
          (4096, 66), (4348, 31), (1024, 2048), (1276, 2051), (64, 4100)]


def bound(a, b):
    return (4 * -(-a.shape[1] // 256) + 12) * 2.0 ** -24 * (np.abs(a.astype(np.float64)) @ np.abs(b.astype(np.float64)))


@pytest.mark.parametrize("rows", [1, 2, 3, 4, 5, 8, 9, 15, 16])
@pytest.mark.parametrize("ind,out", SHAPES)
def test_forward(rows, ind, out):
    x, w, b = synth.normal(1, (rows, ind)), synth.normal(2, (out, ind)), synth.normal(3, (out,))
    want = x.astype(np.float64) @ w.T + b
    lim = bound(x, w.T) + 2.0 ** -23 * np.abs(want)
    assert np.all(np.abs(G.linear(x, w, b) - want) <= lim)
    z, y = G.linear_preact(x, w, b, 4)  # the training options
    assert np.all(np.abs(z - want) <= lim)


@pytest.mark.parametrize("rows", [1, 2, 4, 7, 16])
@pytest.mark.parametrize("dim,hd", [(64, 16), (320, 40), (512, 64), (1024, 64)])
def test_rotary_epilogue(rows, dim, hd):
    """Q and K equal the rotated products, V the product; the rotation mixes a pair's errors."""
    x = synth.normal(1, (rows, dim))
    w = [synth.normal(2 + i, (dim, dim)) for i in range(3)]
    b = [synth.normal(5 + i, (dim,)) for i in range(3)]
    got = G.project_qkv_rope(x, w[0], b[0], w[1], b[1], w[2], b[2], hd)
    for i in range(3):
        z = (x.astype(np.float64) @ w[i].T + b[i]).astype(np.float32)
        lim = bound(x, w[i].T) + 2.0 ** -22 * np.abs(z)
        if i < 2:
            z = G.rope(z, num_heads=dim // hd, head_dim=hd)
            lim = np.repeat(lim.reshape(rows, -1, 2).sum(2), 2, axis=1)
        assert np.all(np.abs(got[i].astype(np.float64) - z) <= lim), "QKV"[i]
