"""GPU tests of the products that run as three bf16 pieces per fp32 operand.

Bound: the kernels add eight products per rounding, so a sum over K has at most
K / 8 + a few roundings of partial sums that never exceed sum |a b|, and the
left-out products are below 2^-24 of it: |got - exact| <= (K / 8 + 8) 2^-24
sum |a b|.  A lost third piece (2^-17), a wrong index or a wrong sign is far
outside it at these K.
"""
from __future__ import annotations

import numpy as np
import pytest

import abi_ops as G
from cdml import synth

pytestmark = pytest.mark.gpu


def check(got, a, b, what, extra=0.0):
    """got against a [M, K] @ b [K, N] (+ extra) in float64."""
    with np.errstate(all="ignore"):
        A, B = a.astype(np.float64), b.astype(np.float64)
        want = A @ B + extra
        bound = (a.shape[1] / 8 + 8) * 2.0 ** -24 * (np.abs(A) @ np.abs(B) + np.abs(extra))
    fine = np.isfinite(want) & (np.abs(want) < np.finfo(np.float32).max)
    assert np.array_equal(np.isnan(got), np.isnan(want)), f"{what}: NaNs elsewhere"
    inf = ~fine & ~np.isnan(want)
    assert np.array_equal(got[inf], np.sign(want[inf]) * np.float32(np.inf)), f"{what}: infinities"
    err = np.abs(got[fine].astype(np.float64) - want[fine])
    assert np.all(err <= bound[fine]), f"{what}: {np.max(err / bound[fine]):.3g} of the bound"


# rows, in, out: one tile and its neighbours (63 .. 65, 127 .. 129), ragged k-tiles (K % 16 = 4, 8, 12; K below
# one tile), both tile sizes (128 x 128 from 192 tiles on), row counts that wgrad reads as a ragged K
SHAPES = [(17, 20, 8), (63, 64, 64), (65, 100, 36), (129, 12, 1028), (127, 136, 132), (300, 8, 200),
          (2100, 72, 1540), (2048, 64, 1536), (4099, 16, 768)]


@pytest.mark.parametrize("rows,ind,out", SHAPES)
def test_forward_and_gradients(rows, ind, out):
    # magnitudes over ten binades, so that every piece of the split carries weight
    scale = np.exp2(synth.uniform(7, rows * ind) * 10 - 5).astype(np.float32).reshape(rows, ind)
    x, w, b = synth.normal(1, (rows, ind)) * scale, synth.normal(2, (out, ind)), synth.normal(3, (out,))
    dy = synth.normal(4, (rows, out))
    check(G.linear(x, w, b), x, w.T, "forward", b.astype(np.float64))
    wg0, bg0 = synth.normal(5, (out, ind)), synth.normal(6, (out,))
    wg, bg, dx = G.linear_backward(x, dy, w, wg0, bg0)
    check(dx, dy, w, "input gradient")
    check(wg, dy.T, x, "weight gradient", wg0.astype(np.float64))
    check(bg[:, None], dy.T, np.ones((rows, 1), np.float32), "bias gradient", bg0.astype(np.float64)[:, None])


@pytest.mark.parametrize("rows,ind,out", [(70, 48, 72), (2100, 64, 1540)])
def test_values_outside_the_split(rows, ind, out):
    """Infinities, NaNs and values above the largest bf16 give what the fp32
    sum gives, and leave the other rows alone."""
    x, w = synth.normal(1, (rows, ind)), synth.normal(2, (out, ind))
    x[3, 5], x[9, 0], x[20, 7], x[41, 11] = np.inf, -np.inf, np.nan, 3.4e38
    w[:, 11] *= np.float32(1e-30)
    w[8, 5] = 0.0  # inf * 0
    check(G.linear(x, w, None), x, w.T, "forward")
    dy = synth.normal(4, (rows, out))
    dy[6, 2], dy[11, 9] = np.nan, np.inf
    wg, bg, dx = G.linear_backward(x, dy, w, np.zeros((out, ind), np.float32), np.zeros(out, np.float32))
    check(dx, dy, w, "input gradient")
    check(wg, dy.T, x, "weight gradient")
