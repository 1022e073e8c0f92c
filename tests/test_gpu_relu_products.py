"""GPU tests of the fp32 MFMA product behind training ReLU layers (gemm_f32_kernel).

Bound: one rounding per product at most, of partial sums that never exceed
sum |a b|, and one for the bias: |z - exact| <= (K + 2) 2^-24 (sum |a b| + |b|).
"""
from __future__ import annotations

import numpy as np
import pytest

import abi_ops as G
from cdml import synth

pytestmark = pytest.mark.gpu


# rows, in, out: one k-tile, 128 x 128 tiles and their neighbours (rows and columns 127 .. 129), and 256 x 128 tiles
# (from 512 of them on) with a ragged last row and column tile
@pytest.mark.parametrize("rows,ind,out", [(17, 16, 4), (127, 48, 132), (129, 32, 127), (256, 64, 129), (1000, 16, 260),
                                          (16385, 32, 1000), (16640, 16, 1024)])
@pytest.mark.parametrize("act", [3, 4])
def test_preactivation_and_output(rows, ind, out, act):
    x, w, b = synth.normal(1, (rows, ind)), synth.normal(2, (out, ind)), synth.normal(3, (out,))
    x[::5] = 0.0
    b[::3] = 0.0  # z exactly 0 where both hold
    z, y = G.linear_preact(x, w, b, act)
    X, W = x.astype(np.float64), w.astype(np.float64)
    bound = (ind + 2) * 2.0 ** -24 * (np.abs(X) @ np.abs(W).T + np.abs(b))
    assert np.all(np.abs(z - (X @ W.T + b)) <= bound)
    assert np.array_equal(y, np.where(z > 0, z, np.float32(0) if act == 3 else np.float32(0.01) * z))
    only = G.linear_preact_output_only(x, w, b, act)
    assert np.array_equal(only, y)
    if act == 3:  # the sign of a zero output tells z < 0
        assert np.array_equal(np.signbit(only), z < 0)
