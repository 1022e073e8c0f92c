"""GPU tests of the products that run as three bf16 pieces per fp32 operand.

Bounds: the kernels add eight products per rounding, so a sum over K has n = K / 8
and a few roundings of partial sums that never exceed sum |a b|, and the left-out
products are below 2^-24 of it: |got - exact| <= (K / 8 + 8) 2^-24 sum |a b|, where
a wrong index or sign is far outside.  Of operands with independent signs the
partial sums grow like sqrt(i / n) and the roundings are independent, each at most
2^-24 / sqrt(3) of its sum in the mean square: the 2-norm of all errors is at most
2^-24 (sqrt(n / 6) + 2) of the results', which a lost third piece (2^-18) exceeds
at every shape here (test_split_bounds.py).
"""
from __future__ import annotations

import numpy as np
import pytest

import abi_ops as G
from cdml import synth

pytestmark = pytest.mark.gpu


def check(got, a, b, what, extra=0.0, floor=2.0 ** -149):
    """got against a [M, K] @ b [K, N] (+ extra) in float64; floor: what sums of subnormals may be off by."""
    with np.errstate(all="ignore"):
        A, B = a.astype(np.float64), b.astype(np.float64)
        want = A @ B + extra
        bound = (a.shape[1] / 8 + 8) * 2.0 ** -24 * (np.abs(A) @ np.abs(B) + np.abs(extra)) + floor
    fine = np.isfinite(want) & (np.abs(want) < np.finfo(np.float32).max)
    assert np.array_equal(np.isnan(got), np.isnan(want)), f"{what}: NaNs elsewhere"
    inf = ~fine & ~np.isnan(want)
    assert np.array_equal(got[inf], np.sign(want[inf]) * np.float32(np.inf)), f"{what}: infinities"
    err = np.abs(got[fine].astype(np.float64) - want[fine])
    assert np.all(err <= bound[fine]), f"{what}: {np.max(err / bound[fine]):.3g} of the bound"
    if fine.all():
        part = np.linalg.norm(err) / np.linalg.norm(want) / (2.0 ** -24 * (np.sqrt(a.shape[1] / 48) + 2))
        assert part <= 1, f"{what}: {part:.3g} of the bound on the 2-norm"


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


def test_wide_tiles():
    """512 tiles of 256 x 128, two whole rounds of 256 CUs, with ragged rows, columns and last k-tile; a few more rows
    make a short third round and leave the product to 128 x 128 tiles, which have the same bits."""
    rows, ind, out = 16300, 36, 1000
    x, w, b = synth.normal(1, (rows, ind)), synth.normal(2, (out, ind)), synth.normal(3, (out,))
    y = G.linear(x, w, b)
    check(y, x, w.T, "forward", b.astype(np.float64))
    z, h = G.linear_preact(x, w, b, 5)  # swish, with its pre-activation
    assert np.array_equal(z, y)
    more = G.linear(np.vstack([x, x[:300]]), w, b)
    assert np.array_equal(more[:rows], y)


def test_wide_tiles_rotary():
    """252 tiles of 256 x 128 (one round) against the same rows in three launches of smaller tiles."""
    rows, dim, hd, seg = 10700, 256, 32, 1070
    x = synth.normal(1, (rows, dim))
    w = [synth.normal(2 + i, (dim, dim)) for i in range(3)]
    b = [synth.normal(5 + i, (dim,)) for i in range(3)]
    args = (w[0], b[0], w[1], b[1], w[2], b[2], hd)
    got = G.project_qkv_rope(x, *args, seg_len=seg)
    check(got[2], x, w[2].T, "V", b[2].astype(np.float64))
    for i in (0, 4280, 9630):
        part = G.project_qkv_rope(x[i:i + seg], *args)
        for g, p in zip(got, part):
            assert np.array_equal(g[i:i + seg], p)


@pytest.mark.parametrize("sx,sw", [(-124, 0), (0, -124), (-60, -60), (90, -110)])
@pytest.mark.parametrize("rows,ind,out", [(70, 48, 72), (300, 100, 200), (2100, 64, 1540)])
def test_small_operands(rows, ind, out, sx, sw):
    """The split keeps all bits of operands down to the smallest normal floats."""
    x, w = synth.normal(1, (rows, ind)) * np.float32(2.0 ** sx), synth.normal(2, (out, ind)) * np.float32(2.0 ** sw)
    dy = synth.normal(4, (rows, out)) * np.float32(2.0 ** (min(sx, 0) if sw else 0))
    check(G.linear(x, w, None), x, w.T, "forward")
    wg, _, dx = G.linear_backward(x, dy, w, np.zeros((out, ind), np.float32), np.zeros(out, np.float32))
    check(dx, dy, w, "input gradient")
    check(wg, dy.T, x, "weight gradient", floor=2.0 ** -149 * 64)  # a sum of up to 64 chunks


@pytest.mark.parametrize("rows,ind,hid", [(300, 64, 256), (4099, 256, 512)])
def test_relu_block_gradients(rows, ind, hid):
    """A training ReLU block's backward against float64 with the derivatives that the kernel's own output marks, so
    that no bound has to allow for a pre-activation on either side of 0."""
    x, w1, b1 = synth.normal(1, (rows, ind)), synth.xavier_uniform(2, hid, ind), synth.normal(3, (hid,))
    dy, w2 = synth.normal(4, (rows, ind)), synth.xavier_uniform(5, ind, hid)
    z2, z1 = np.zeros((ind, hid), np.float32), np.zeros((hid, ind), np.float32)
    h = G.linear_preact_output_only(x, w1, b1, 3)
    dh, gw2, gb2 = G.linear_backward_act(h, dy, w2, z2, z2[:, 0].copy(), dz=h, act=3 | 0x100)
    check(gw2, dy.T, h, "second layer's weights")
    check(gb2[:, None], dy.T, np.ones((rows, 1), np.float32), "second layer's bias")
    on = ~np.signbit(h)
    assert not dh[~on].any()
    exact = (dy.astype(np.float64) @ w2.astype(np.float64)).astype(np.float32)
    check(np.where(on, dh, exact), dy, w2, "hidden deltas")
    dx, gw1, gb1 = G.linear_backward_act(x, dh, w1, z1, z1[:, 0].copy())
    check(dx, dh, w1, "input gradient")
    check(gw1, dh.T, x, "first layer's weights")
    check(gb1[:, None], dh.T, np.ones((rows, 1), np.float32), "first layer's bias")


# out (the product's K) with every remainder by 4 and by 16, in rows padded to the next multiple of 4
@pytest.mark.parametrize("rows,ind,out", [(17, 8, 130), (65, 64, 17), (129, 132, 19), (300, 200, 31), (4099, 1024, 45)])
def test_padded_rows_of_any_width(rows, ind, out):
    """Input gradient and matrix product of rows with an aligned stride whose width is no multiple of 4: the padding
    (NaN here) is not read into the sums."""
    ld = -(-out // 4) * 4
    dy, w = synth.normal(4, (rows, out)), synth.normal(2, (out, ind))
    padded = np.full((rows, ld), np.nan, np.float32)
    padded[:, :out] = dy
    bdy, bw, dx = G.up(padded), G.up(w), G.N.DeviceBuffer(rows * ind * 4)
    G.N.check(G.N.lib().cdml_linear_backward(None, ind, bdy.ptr, ld, bw.ptr, dx.ptr, ind, None, None, rows, ind, out, 0,
                                             None, 0, G.stream().handle))
    check(G.down(dx, (rows, ind)), dy, w, "input gradient")
    G.N.check(G.N.lib().cdml_matmul(bdy.ptr, ld, bw.ptr, ind, dx.ptr, ind, rows, out, ind, G.stream().handle))
    check(G.down(dx, (rows, ind)), dy, w, "matrix product")


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


# the K-segmented input gradient, on both tile sizes
@pytest.mark.parametrize("rows,ind,out", [(70, 48, 64), (2100, 1540, 16)])
def test_backprop_qkv_values_outside_the_split(rows, ind, out):
    d = [synth.normal(1 + i, (rows, out)) for i in range(3)]
    w = [synth.normal(4 + i, (out, ind)) for i in range(3)]
    d[0][3, 5], d[1][9, 0], d[2][20, 7], d[2][41, 11] = np.inf, -np.inf, np.nan, 3.4e38
    w[2][11] *= np.float32(1e-30)
    zeros = [t for _ in range(3) for t in (np.zeros((out, ind), np.float32), np.zeros(out, np.float32))]
    got = G.backprop_qkv(synth.normal(7, (rows, ind)), *d, *w, *zeros)[0]
    check(got, np.hstack(d), np.vstack(w), "input gradient")


@pytest.mark.parametrize("rows,dim,hd", [(70, 64, 16), (2048, 512, 64)])
def test_rotary_values_outside_the_split(rows, dim, hd):
    """Q and K are the rotation of what the fp32 sums give, infinities and NaNs included, V the sums."""
    x = synth.normal(1, (rows, dim))
    w = [synth.normal(2 + i, (dim, dim)) for i in range(3)]
    b = [synth.normal(5 + i, (dim,)) for i in range(3)]
    x[3, 5], x[9, 0], x[20, 7], x[41, 11] = np.inf, -np.inf, np.nan, 3.4e38
    for t in w:
        t[:, 11] *= np.float32(1e-30)
    got = G.project_qkv_rope(x, w[0], b[0], w[1], b[1], w[2], b[2], hd)
    check(got[2], x, w[2].T, "V", b[2].astype(np.float64))
    for i in range(2):
        with np.errstate(all="ignore"):
            X, W = x.astype(np.float64), w[i].T.astype(np.float64)
            z = X @ W + b[i]
            lim = (dim / 8 + 8) * 2.0 ** -24 * (np.abs(X) @ np.abs(W) + np.abs(b[i])) + 2.0 ** -22 * np.abs(z)
        want = G.rope(z.astype(np.float32), num_heads=dim // hd, head_dim=hd)
        lim = np.repeat(lim.reshape(rows, -1, 2).sum(2), 2, axis=1)  # the rotation mixes a pair's errors
        assert np.array_equal(np.isnan(got[i]), np.isnan(want)), "QK"[i]
        inf, fine = np.isinf(want), np.isfinite(want)
        assert np.array_equal(got[i][inf], want[inf]), "QK"[i]
        assert np.all(np.abs(got[i][fine].astype(np.float64) - want[fine]) <= lim[fine]), "QK"[i]


def attention64(q, k, v, heads, scale, causal):
    """float64 softmax attention of one sequence; (o, sum p |v|, largest sum |q| |k| of a row's scores)."""
    L, D = q.shape
    hd = D // heads
    o, w, m = (np.zeros((L, D)) for _ in range(3))
    for h in range(heads):
        c = slice(h * hd, (h + 1) * hd)
        Q, K, V = (t[:, c].astype(np.float64) for t in (q, k, v))
        with np.errstate(all="ignore"):
            s, a = Q @ K.T * scale, np.abs(Q) @ np.abs(K).T * abs(scale)
            if causal:
                s = np.where(np.tril(np.ones(s.shape, bool)), s, -np.inf)
                a = np.where(np.tril(np.ones(s.shape, bool)), a, 0)
            p = np.exp(s - s.max(1, keepdims=True))
            p /= p.sum(1, keepdims=True)
            o[:, c], w[:, c], m[:, c] = p @ V, p @ np.abs(V), a.max(1, keepdims=True)
    return o, w, m


def check_attention(got, q, k, v, heads, scale, causal, what):
    """A score's error is (hd / 8 + 8) 2^-24 sum |q| |k| scale, which moves a probability by as much
    relatively; the sums over keys add (L / 8 + 8) 2^-24, exp2 and the scaling a few 2^-23."""
    L, D = q.shape
    want, w, m = attention64(q, k, v, heads, scale, causal)
    assert np.array_equal(np.isnan(got), np.isnan(want)), f"{what}: NaNs elsewhere"
    inf = np.isinf(want)
    assert np.array_equal(got[inf], want[inf]), f"{what}: infinities"
    fine = np.isfinite(want)
    bound = (2 * (D // heads / 8 + 8) * m + L / 8 + 32) * 2.0 ** -24 * w
    with np.errstate(invalid="ignore"):
        err = np.abs(got.astype(np.float64) - want)
    assert np.all(err[fine] <= bound[fine]), f"{what}: {np.nanmax(err[fine] / bound[fine]):.3g} of the bound"


# head dims on both sides of the padded sizes 32, 64 and 128 (40 and 20 take the scalar loads), lengths around a
# 32-key tile, a wave's 32 and a workgroup's 128 queries
@pytest.mark.parametrize("L", [1, 31, 33, 127, 129, 300])
@pytest.mark.parametrize("hd", [20, 32, 40, 64, 128])
def test_attention_forward(hd, L):
    heads = 2
    q, k, v = (synth.normal(i, (L, heads * hd)) for i in (1, 2, 3))
    q = q * np.float32(3.0)  # probabilities over many binades
    for causal in (False, True):
        got = G.sdpa(q, k, v, heads, causal=causal, scale=1.0 / np.sqrt(hd))
        check_attention(got, q, k, v, heads, 1.0 / np.sqrt(hd), causal, f"hd {hd} L {L} causal {causal}")


@pytest.mark.parametrize("hd", [32, 40, 64, 128])
def test_attention_values_outside_the_split(hd):
    """Rows that an infinity, a NaN or a value above the largest bf16 reaches come out as the fp32 products give
    them; the others are untouched."""
    L, heads = 130, 2
    q, k, v = (synth.normal(i, (L, heads * hd)) for i in (4, 5, 6))
    q[7, 3], v[0, hd + 1] = np.nan, 3.4e38
    k[40, :] = 0.0
    k[40, 2] = -np.inf  # score -inf or +inf by the sign of q: weight 0, or a row of NaNs
    for causal in (False, True):
        got = G.sdpa(q, k, v, heads, causal=causal, scale=1.0 / np.sqrt(hd))
        check_attention(got, q, k, v, heads, 1.0 / np.sqrt(hd), causal, f"hd {hd} causal {causal}")
    q, k = (synth.normal(i, (L, heads * hd)) for i in (4, 5))
    v[5, 1] = np.inf  # every row sees it without the causal rule
    got = G.sdpa(q, k, v, heads, scale=1.0 / np.sqrt(hd))
    check_attention(got, q, k, v, heads, 1.0 / np.sqrt(hd), False, f"hd {hd} infinite value")


@pytest.mark.parametrize("hd", [32, 40, 64, 128])
def test_attention_small_operands(hd):
    """V of the smallest normal floats, and Q and K at opposite ends of the range."""
    L, heads, scale = 130, 2, 1.0 / np.sqrt(hd)
    q, k, v = (synth.normal(i, (L, heads * hd)) for i in (4, 5, 6))
    up, down = np.float32(2.0 ** 112), np.float32(2.0 ** -112)
    for a, b, c, what in ((q, k, v * np.float32(2.0 ** -122), "V"), (q * up, k * down, v, "K"), (q * down, k * up, v, "Q")):
        for causal in (False, True):
            check_attention(G.sdpa(a, b, c, heads, causal=causal, scale=scale), a, b, c, heads, scale, causal,
                            f"small {what}, hd {hd} causal {causal}")


def backward(q, k, v, dout, heads, scale, causal, mask=None, stored=False):
    """cdml_sdpa_bwd; stored: with the workspace that lets the dK/dV pass store dS."""
    L, D = q.shape
    bufs = [G.up(t) for t in (q, k, v, dout)]
    grads = [G.N.DeviceBuffer(L * D * 4) for _ in range(3)]
    bm = G.up(mask, np.uint8) if mask is not None else None
    n = G.C.c_size_t(0)
    if stored:
        G.N.check(G.N.lib().cdml_sdpa_bwd_stored_ds_workspace_size(1, L, L, D, heads, int(causal), G.C.byref(n)))
    else:
        G.N.check(G.N.lib().cdml_sdpa_bwd_workspace_size(1, L, L, D, heads, G.C.byref(n)))
    ws = G.N.DeviceBuffer(max(256, n.value))
    ins = [x for b in bufs for x in (b.ptr, D)]
    outs = [x for g in grads for x in (g.ptr, D)]
    G.N.check(G.N.lib().cdml_sdpa_bwd(*ins, *outs, 1, L, L, D, heads, scale, int(causal), bm.ptr if bm else None,
                                      ws.ptr, n.value, G.stream().handle))
    return [G.down(g, (L, D)) for g in grads]


def weighted(p, x):
    """p @ x in which a weight of 0 leaves a term out, an infinite one too."""
    out = p @ np.where(np.isfinite(x), x, 0.0)
    for i, c in np.argwhere(~np.isfinite(x)):
        out[p[:, i] != 0, c] += p[p[:, i] != 0, i] * x[i, c]
    return out


def backward64(q, k, v, dout, heads, scale, allowed, per=8):
    """(gradient, its error bound) of dQ, dK and dV in float64, u = 2^-24.  A probability is off by (2 (hd / 8 + 8) m +
    L / 8 + 32) u relatively (check_attention), dP by (hd / 8 + 8) u sum |dO| |V|, D by the output's error and
    its own sum's, (hd / 8 + 8) u sum |dO| |O|; products of these with the last operand add (L / 8 + 8) u.
    per: products that one rounding adds, 8 above; the fp32 MFMA adds 2."""
    L, D = q.shape
    hd, u = D // heads, 2.0 ** -24
    out = [(np.empty((L, D)), np.empty((L, D))) for _ in range(3)]
    for h in range(heads):
        c = slice(h * hd, (h + 1) * hd)
        Q, K, V, G_ = (t[:, c].astype(np.float64) for t in (q, k, v, dout))
        with np.errstate(all="ignore"):
            s = np.where(allowed, Q @ K.T * scale, -np.inf)
            m = np.max(np.where(allowed, np.abs(Q) @ np.abs(K).T * scale, 0.0), 1, keepdims=True)
            p = np.exp(s - s.max(1, keepdims=True))
            p /= p.sum(1, keepdims=True)
            o, dp = p @ V, G_ @ V.T
            d = (G_ * o).sum(1, keepdims=True)
            ds = np.where(p > 0, p * (dp - d), 0.0)
            ep = (2 * (hd / per + 8) * m + L / per + 32) * u
            edp = (hd / per + 8) * u * (np.abs(G_) @ np.abs(V).T)
            ed = (np.abs(G_) * (ep * (p @ np.abs(V)) + (hd / per + 8) * u * np.abs(o))).sum(1, keepdims=True)
            eds = np.where(p > 0, p * (ep * np.abs(dp - d) + edp + ed + 4 * u * (np.abs(dp) + np.abs(d))), 0.0)
            sum_u = (L / per + 8) * u
            out[0][0][:, c], out[0][1][:, c] = ds @ K * scale, (eds + sum_u * np.abs(ds)) @ np.abs(K) * scale
            out[1][0][:, c], out[1][1][:, c] = ds.T @ Q * scale, (eds + sum_u * np.abs(ds)).T @ np.abs(Q) * scale
            out[2][0][:, c], out[2][1][:, c] = weighted(p.T, G_), weighted((p * (ep + sum_u)).T, np.abs(G_))
    return out


def check_backward(got, want, what, floor=2.0 ** -126):
    """floor: values under the smallest normal float may be flushed."""
    for g, (w, bound), name in zip(got, want, ("dQ", "dK", "dV")):
        assert np.array_equal(np.isnan(g), np.isnan(w)), f"{what} {name}: NaNs elsewhere"
        inf = np.isinf(w)
        assert np.array_equal(g[inf], w[inf]), f"{what} {name}: infinities"
        fine = np.isfinite(w)
        with np.errstate(invalid="ignore"):
            over = np.abs(g.astype(np.float64) - np.where(fine, w, 0.0)) - bound - floor
        assert np.all(over[fine] <= 0), f"{what} {name}: {np.max(over[fine]):.3g} over the bound"


# lengths around the 32-query tiles, a wave's 32 and a workgroup's 128 keys; head dim 32 runs one wave per key block,
# 64 two, 20 and 40 their scalar loads
@pytest.mark.parametrize("L", [1, 31, 33, 97, 129, 300])
@pytest.mark.parametrize("hd", [20, 32, 40, 64])
def test_attention_backward(hd, L):
    heads, scale = 2, 1.0 / np.sqrt(hd)
    q, k, v, dout = (synth.normal(i, (L, heads * hd)) for i in (1, 2, 3, 4))
    q = q * np.float32(2.0)
    tril, full = np.tril(np.ones((L, L), bool)), np.ones((L, L), bool)
    drop = synth.uniform(9, L * L).reshape(L, L) < 0.7
    drop[:, 0] = True  # every query sees a key
    for causal, mask in ((False, None), (True, None), (False, drop), (True, drop)):
        allowed = (tril if causal else full) & (drop if mask is not None else full)
        want = backward64(q, k, v, dout, heads, scale, allowed)
        what = f"hd {hd} L {L} causal {causal} mask {mask is not None}"
        check_backward(backward(q, k, v, dout, heads, scale, causal, mask), want, what)
        if causal and mask is None:
            check_backward(backward(q, k, v, dout, heads, scale, causal, stored=True), want, what + " stored dS")


# head dims 20 and 40: scalar loads, the last column beside those that count as zero
@pytest.mark.parametrize("hd,col", [(32, 3), (64, 3), (20, 19), (40, 39)])
def test_attention_backward_values_outside_the_split(hd, col):
    """An infinite and a huge output gradient: the keys they reach get what the fp32 products give, the others
    their values."""
    L, heads, scale = 130, 2, 1.0 / np.sqrt(hd)
    q, k, v, dout = (synth.normal(i, (L, heads * hd)) for i in (1, 2, 3, 4))
    # Query 31 sees all of the first 32 keys, in the first head.  (A masked pair of the same 32 x 32 block has weight
    # 0, and 0 * inf is a NaN in fp32 too.)
    dout[31, col] = np.inf
    dout[70, hd + 5] = 3.4e38  # above the largest bf16
    v[:, hd + 5] *= np.float32(1e-30)
    tril, full = np.tril(np.ones((L, L), bool)), np.ones((L, L), bool)
    drop = synth.uniform(9, L * L).reshape(L, L) < 0.7
    drop[:, 0] = drop[31] = True  # every query sees a key, and query 31 all that it may
    for causal, mask in ((True, None), (False, None), (False, drop), (True, drop)):
        allowed = (tril if causal else full) & (drop if mask is not None else full)
        # what they reach is summed on the fp32 MFMA
        want = backward64(q, k, v, dout, heads, scale, allowed, per=2)
        for stored in (False, True):
            check_backward(backward(q, k, v, dout, heads, scale, causal, mask, stored=stored and mask is None), want,
                           f"hd {hd} causal {causal} mask {mask is not None} stored {stored}")


@pytest.mark.parametrize("hd", [20, 32, 40, 64])
def test_attention_backward_small_operands(hd):
    """Gradients of the smallest normal floats, and V, Q and K of such, keep all their bits."""
    L, heads, scale = 130, 2, 1.0 / np.sqrt(hd)
    t = [synth.normal(i, (L, heads * hd)) for i in (1, 2, 3, 4)]
    tril = np.tril(np.ones((L, L), bool))
    for small in ((3,), (2,), (0,), (1,)):
        q, k, v, dout = (x * np.float32(2.0 ** -120) if i in small else x for i, x in enumerate(t))
        want = backward64(q, k, v, dout, heads, scale, tril)
        for stored in (False, True):
            check_backward(backward(q, k, v, dout, heads, scale, True, stored=stored), want,
                           f"hd {hd} small {'QKVG'[small[0]]} stored {stored}", floor=2.0 ** -149 * L)


def backward_saved(q, k, v, dout, batch, heads, rope):
    """Causal cdml_sdpa_bwd_saved(_rope) of `batch` sequences, with room for the stored dS -> dQ, dK, dV."""
    R, D = q.shape
    L, hd, C = R // batch, D // heads, G.C
    lib, st, scale = G.N.lib(), G.stream().handle, 1.0 / np.sqrt(D // heads)
    bufs = [G.up(t) for t in (q, k, v, dout)]
    o, lse, cs = G.N.DeviceBuffer(R * D * 4), G.N.DeviceBuffer(batch * heads * L * 4), G.N.DeviceBuffer(L * hd * 4)
    grads = [G.N.DeviceBuffer(R * D * 4) for _ in range(3)]
    qkv = [x for b in bufs[:3] for x in (b.ptr, D)]
    outs = [x for g in grads for x in (g.ptr, D)]
    G.N.check(lib.cdml_sdpa_fwd_lse(*qkv, o.ptr, D, lse.ptr, batch, L, L, D, heads, scale, 1, None, st))
    G.N.check(lib.cdml_rope_table(cs.ptr, L, hd, 10000.0, st))
    n = C.c_size_t(0)
    G.N.check(lib.cdml_sdpa_bwd_saved_workspace_size(batch, L, L, D, heads, 1, C.byref(n)))
    ws = G.N.DeviceBuffer(n.value)
    args = [*qkv, o.ptr, D, lse.ptr, bufs[3].ptr, D, *outs, batch, L, L, D, heads, scale, 1, None]
    if rope:
        G.N.check(lib.cdml_sdpa_bwd_saved_rope(*args, cs.ptr, L, ws.ptr, n.value, st))
    else:
        G.N.check(lib.cdml_sdpa_bwd_saved(*args, ws.ptr, n.value, st))
    return [G.down(g, (R, D)) for g in grads]


# 13 to 16 query blocks, whole and ragged, of at least 512 (sequence, head) pairs take the kernel that stages a
# head's whole K; a few sequences take the tiled one, which test_attention_backward checks
@pytest.mark.parametrize("L", [385, 416, 447, 512])
@pytest.mark.parametrize("rope", [False, True])
def test_short_dq_has_the_bits_of_the_tiled_one(L, rope):
    heads, few, copies = 4, 4, 32
    q, k, v, dout = (synth.normal(i, (few * L, heads * 32)) for i in (1, 2, 3, 4))
    dout[L + 5, 40] = np.inf  # one head's dQ is recomputed on the fp32 MFMA
    want = backward_saved(q, k, v, dout, few, heads, rope)
    got = backward_saved(*(np.tile(t, (copies, 1)) for t in (q, k, v, dout)), few * copies, heads, rope)
    for g, w, name in zip(got, want, ("dQ", "dK", "dV")):
        assert np.array_equal(g.view(np.uint32), np.tile(w, (copies, 1)).view(np.uint32)), name


def drift(err, sign):
    """Mean of sign * err over the errors' root mean square, in units of what independent errors give."""
    return abs((err * sign).mean()) / np.sqrt((err ** 2).mean()) * np.sqrt(err.size)


def test_errors_do_not_add_up_over_rows():
    """The bf16 MFMA rounds down; the kernels alternate the signs of rows and columns so that its drift does not
    collect in sums over rows (bias gradients).  Independent errors give a normal deviate; without the alternation
    along the rows the drift of dQ is 10 and that of O, alternating with the column, 11."""
    rows, ind, out = 32768, 64, 64
    x, w = synth.normal(1, (rows, ind)), synth.normal(2, (out, ind))
    err = G.linear(x, w, None) - x.astype(np.float64) @ w.astype(np.float64).T
    alternating = np.where(np.arange(out) % 2, -1.0, 1.0)
    assert drift(err, 1.0) < 5 and drift(err, alternating) < 5
    batch, heads, hd, L = 256, 4, 32, 128
    D, scale = heads * hd, 1.0 / np.sqrt(hd)
    q, k, v, dout = (synth.normal(i, (batch * L, D)) for i in (1, 2, 3, 4))
    dq, dk, _ = backward_saved(q, k, v, dout, batch, heads, False)
    o = G.sdpa(q, k, v, heads, causal=True, scale=scale, batch=batch)
    Q, K, V, W = (t.reshape(batch, L, heads, hd).transpose(0, 2, 1, 3).astype(np.float64) for t in (q, k, v, dout))
    s = np.where(np.tril(np.ones((L, L), bool)), Q @ K.swapaxes(2, 3) * scale, -np.inf)
    p = np.exp(s - s.max(3, keepdims=True))
    p /= p.sum(3, keepdims=True)
    O = p @ V
    ds = p * (W @ V.swapaxes(2, 3) - (W * O).sum(3, keepdims=True))
    flat = lambda t: t.transpose(0, 2, 1, 3).reshape(-1, D)
    alternating = np.where(np.arange(D) % 2, -1.0, 1.0)
    for got, want, name in ((dq, ds @ K * scale, "dQ"), (dk, ds.swapaxes(2, 3) @ Q * scale, "dK"), (o, O, "O")):
        err = got - flat(want)
        assert drift(err, 1.0) < 5 and drift(err, alternating) < 5, name
