"""The bounds of test_gpu_split_products.py see a lost third piece (no GPU: the products of two pieces are emulated)."""
from __future__ import annotations

import numpy as np
import pytest

from cdml import synth
from test_gpu_split_products import SHAPES, check


def bf16(x):
    u = x.view(np.uint32).astype(np.uint64)
    return ((u + 0x7fff + (u >> 16 & 1)) & 0xffff0000).astype(np.uint32).view(np.float32)


def two_pieces(x):
    h = bf16(x)
    return h.astype(np.float64) + bf16(x - h)


@pytest.mark.parametrize("rows,ind,out", SHAPES)
def test_a_lost_third_piece_is_seen(rows, ind, out):
    scale = np.exp2(synth.uniform(7, rows * ind) * 10 - 5).astype(np.float32).reshape(rows, ind)
    x, w, dy = synth.normal(1, (rows, ind)) * scale, synth.normal(2, (out, ind)), synth.normal(4, (rows, out))
    for a, b in ((x, w.T), (dy, w), (dy.T, x)):
        a, b = np.ascontiguousarray(a), np.ascontiguousarray(b)
        check((a.astype(np.float64) @ b.astype(np.float64)).astype(np.float32), a, b, "exact")
        with pytest.raises(AssertionError):
            check((two_pieces(a) @ two_pieces(b)).astype(np.float32), a, b, "two pieces")
