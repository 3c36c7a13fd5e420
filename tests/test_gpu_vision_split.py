"""The vision tower's kernels on fp16 parts one at a time against float64: the product on every tile
and output that the tower runs, LayerNorm over a split product's parts, the heads and attention at
one and two query blocks a wave, the weights' spreads.  The operands' layouts are restated here in
numpy.  Needs an MI355X."""
import math
import sys

import numpy as np
import pytest

import exn_hip as X
from oracle import exn_oracle as xo
from oracle import exn_vision_oracle as vo
from vision_split_cases import CASES, padded

pytestmark = pytest.mark.gpu
ULP = 2.0 ** -24      # half a unit in fp32's last place, relative


def say(*a):
    print("[gpu]", *a, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def ctx():
    c = X.Context(0)
    yield c
    c.close()


def dev(ctx, a):
    return X.DevBuf.of(ctx, np.ascontiguousarray(a))


def split_rows(x, kp, scale):
    """X (M x K) as split rows of KP: 32 hi and 32 lo halves for every 32 columns."""
    v = np.zeros((len(x), kp), np.float32)
    v[:, :x.shape[1]] = x * np.float32(scale)
    hi = v.astype(np.float16)
    lo = (v - hi.astype(np.float32)).astype(np.float16)
    return np.stack([hi.reshape(len(x), -1, 32), lo.reshape(len(x), -1, 32)], 2).reshape(len(x), 2 * kp).view(np.uint16)


def joined(rows, scale):
    """The values of split rows."""
    h = rows.view(np.float16).astype(np.float64).reshape(len(rows), -1, 2, 32)
    return (h[:, :, 0] + h[:, :, 1]).reshape(len(rows), -1) / scale


def packed(w, kp):
    """W (N x K), fp16 values, in KP / 32 runs of N rounded up to 64 rows of 32."""
    a = np.zeros(((len(w) + 63) // 64 * 64, kp), np.float16)
    a[:len(w), :w.shape[1]] = w
    return a.reshape(len(a), -1, 32).transpose(1, 0, 2).copy().view(np.uint16)


@pytest.mark.parametrize("kind,tile,m,n,parts", CASES)
def test_split_product(ctx, kind, tile, m, n, parts):
    """K ends 42 columns before its padding; rows of 1 and of 2^-9 times their size.  A sum of K
    products in steps of 32 and two parts rounds K / 16 times, and a few more in what follows (bias,
    residual, GELU's exp2, reciprocal and products), each at most ULP of the products' absolute sum;
    the input's parts keep 2^-23 of a row and 2^-40 of the bound (8)."""
    say("vis_gemm_s", kind, tile, m, n, parts)
    kp = padded(parts)
    k = kp - 42
    x = np.clip(xo.normal(1, 7101, m * k).reshape(m, k), -8, 8)
    x[1::3] *= np.float32(2.0 ** -9)
    w = (xo.normal(1, 7102, n * k).reshape(n, k) / np.float32(math.sqrt(k))).astype(np.float16)
    b = xo.normal(1, 7103, n) * np.float32(0.1)
    sx, so, ldy = 2.0 ** 12, 2.0 ** 10, (n + 63) // 64 * 64
    dx, dw, db = dev(ctx, split_rows(x, kp, sx)), dev(ctx, packed(w, kp)), dev(ctx, b)
    want = x.astype(np.float64) @ w.astype(np.float64).T
    scale = np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64).T + 2.0 ** -40 * 8 * 2 ** 24 * np.abs(w).sum(1, dtype=np.float64)
    args = (m, n, kp, 1 / sx)
    if kind == "f32":
        r = xo.normal(1, 7104, m * n).reshape(m, n)
        for res in (False, True):
            y = dev(ctx, r)                   # with a residual the output is written over it
            X.call("exn_vis_gemm_s", ctx.h, dx.h, dw.h, db.h, y.h if res else None, y.h, None, *args, 0.0, 0, 0, 1)
            exact = want + b + (r if res else 0)
            err = np.abs(y.get() - exact) / (scale + np.abs(b) + np.abs(exact))
            assert err.max() < (kp / 16 + 8) * ULP, err.max()
    elif kind == "part":
        y = dev(ctx, np.full((parts, m, n), np.nan, np.float32))
        X.call("exn_vis_gemm_s", ctx.h, dx.h, dw.h, None, None, y.h, None, *args, 0.0, 0, 0, parts)
        err = np.abs(y.get().astype(np.float64).sum(0) - want) / scale
        assert err.max() < (kp / 16 + 8) * ULP, err.max()
    else:
        y = dev(ctx, np.full((m, 2 * ldy), 0xFFFF, np.uint16))
        X.call("exn_vis_gemm_s", ctx.h, dx.h, dw.h, db.h, None, None, y.h, *args, so, ldy, 1 if kind == "tanh" else 2, 1)
        v = want + b
        if kind == "tanh":
            exact = 0.5 * v * (1 + np.tanh(math.sqrt(2 / math.pi) * (v + 0.044715 * v ** 3)))
        else:
            from scipy.special import erf
            exact = 0.5 * v * (1 + erf(v / math.sqrt(2)))
        got = joined(y.get(), so)
        assert not got[:, n:].any()           # the next product reads zeros there
        # GELU's slope is at most 1.13; its own steps round values up to |v| (1 + 2 |v|) deep
        err = np.abs(got[:, :n] - exact) / (scale + np.abs(b) + np.abs(v) * (1 + 2 * np.abs(v)) + 2.0 ** -10)
        assert err.max() < (kp / 16 + 8) * ULP, err.max()


@pytest.mark.parametrize("k", [1152, 4304])
def test_split_product_is_no_further_off_than_the_fp32_one(ctx, k):
    """The tower's products at 320 patches: relative distance from 64 bits, on fp16 parts and on fp32
    MFMAs, the same inputs."""
    m, n, kp = 320, 1152, (k + 63) // 64 * 64
    x = xo.normal(1, 7105, m * k).reshape(m, k)
    w = (xo.normal(1, 7106, n * k).reshape(n, k) / np.float32(math.sqrt(k))).astype(np.float16)
    b = np.zeros(n, np.float32)
    y, yf = X.DevBuf(ctx, (m, n), np.float32), X.DevBuf(ctx, (m, n), np.float32)
    dx, dw, db = dev(ctx, split_rows(x, kp, 2.0 ** 12)), dev(ctx, packed(w, kp)), dev(ctx, b)
    X.call("exn_vis_gemm_s", ctx.h, dx.h, dw.h, db.h, None, y.h, None, m, n, kp, 2.0 ** -12, 0.0, 0, 0, 1)
    fx, fw = dev(ctx, x), dev(ctx, w.astype(np.float32))
    X.call("exn_vis_gemm", ctx.h, fx.h, fw.h, db.h, None, yf.h, m, n, k, 0)
    want = x.astype(np.float64) @ w.astype(np.float64).T
    e, ef = xo.rel_l2(y.get(), want), xo.rel_l2(yf.get(), want)
    say("vis_gemm_s K", k, "relative distance", e, "fp32", ef)
    assert e < ef < 2e-6


@pytest.mark.parametrize("rows,width,parts", [(37, 1152, 0), (1, 1152, 1), (40, 1152, 3), (9, 1152, 8), (9, 4608, 0)])
def test_split_layernorm(ctx, rows, width, parts):
    """X += bias + the parts in order (float32, bit for bit), then LayerNorm as fp32 rows and as
    split rows, both within 1e-5 of float64 (as the fp32 kernel's test)."""
    say("vis_ln_s", rows, width, parts)
    x = xo.normal(3, 7120, rows * width).reshape(rows, width) * np.float32(3.0) + np.float32(1.5)
    w = np.float32(1) + np.float32(0.1) * xo.normal(3, 7121, width)
    b, bias = np.float32(0.02) * xo.normal(3, 7122, width), xo.normal(3, 7123, width)
    part = xo.normal(3, 7124, max(parts, 1) * rows * width).reshape(-1, rows, width)
    new = x
    if parts:
        a = np.broadcast_to(bias, x.shape)
        for p in part:
            a = (a + p).astype(np.float32)
        new = (a + x).astype(np.float32)
    x64 = new.astype(np.float64)
    c = x64 - x64.mean(1, keepdims=True)
    want = c / np.sqrt((c ** 2).mean(1, keepdims=True) + 1e-6) * w + b
    dp, dbias, dw, db = dev(ctx, part), dev(ctx, bias), dev(ctx, w), dev(ctx, b)
    for split in (False, True):
        dx = dev(ctx, x)
        y = X.DevBuf(ctx, (rows, 2 * width) if split else (rows, width), np.uint16 if split else np.float32)
        X.call("exn_vis_ln_s", ctx.h, rows, width, dx.h, parts, dp.h if parts else None, dbias.h if parts else None,
               dw.h, db.h, 2.0 ** 8, y.h if split else None, None if split else y.h)
        assert np.array_equal(dx.get(), new)
        got = joined(y.get(), 2.0 ** 8) if split else y.get()
        assert np.abs(got - want).max() < 1e-5


# queries a workgroup: 64, or 128 where those make over 384 workgroups (the last two)
@pytest.mark.parametrize("n,heads", [(4, 16), (68, 16), (132, 3), (320, 16), (1000, 2), (260, 160), (4096, 16)])
def test_split_heads_and_attention(ctx, n, heads):
    """QKV rows through the split heads and attention into fp32 and split rows: against softmax
    attention in float64 (three heads), within 2e-5 (the fp32 kernel's bar) and, over the heads, no
    further off than the fp32 kernel on the same heads."""
    say("vis_attend_s", n, heads)
    D = 72 * heads
    qkv = xo.normal(4, 7130, n * 3 * D).reshape(n, 3, heads, 72)
    qkv[:, :2] *= np.float32(2.0)
    cos, sin = vo.rotary(*vo.merge_order(n // 2, 2), 72)
    cs = np.concatenate([cos, sin], 1).astype(np.float32)
    qscale, np_ = 1.4426950408889634 / math.sqrt(72), (n + 63) // 64 * 64
    # bounds: |q|, |k| at most 2 x 6 sqrt(2), |v| at most 6
    eq, ek, ev = 2.0 ** 13, 2.0 ** 10, 2.0 ** 12
    dq, dk = X.DevBuf(ctx, (heads, n, 152), np.uint16), X.DevBuf(ctx, (heads, n, 152), np.uint16)
    dvt = X.DevBuf(ctx, (2, heads, 72, np_), np.uint16)
    dqkv, dcs = dev(ctx, qkv), dev(ctx, cs)
    X.call("exn_vis_heads_s", ctx.h, n, heads, dqkv.h, dcs.h, qscale * eq, ek, ev, dq.h, dk.h, dvt.h)
    yf = X.DevBuf(ctx, (n, D), np.float32)
    X.call("exn_vis_attend_s", ctx.h, n, heads, dq.h, dk.h, dvt.h, 1 / (eq * ek), 1 / ev, None, yf.h)
    got = yf.get()
    if D % 64 == 0:
        ys = X.DevBuf(ctx, (n, 2 * D), np.uint16)
        X.call("exn_vis_attend_s", ctx.h, n, heads, dq.h, dk.h, dvt.h, 1 / (eq * ek), 1 / ev, ys.h, None)
        assert np.abs(joined(ys.get(), ev) - got).max() < 2 ** -22 * np.abs(got).max()   # the same in two parts
    q, k = (vo.rope(qkv[:, i].astype(np.float64), cs[:, :72].astype(np.float64), cs[:, 72:].astype(np.float64)) for i in (0, 1))
    some = sorted({0, heads // 2, heads - 1})
    want = vo_attention64(q[:, some], k[:, some], qkv[:, 2, some].astype(np.float64))
    mine = got.reshape(n, heads, 72)[:, some]
    assert np.abs(mine - want).max() < 2e-5
    f32 = [dev(ctx, np.ascontiguousarray(a, np.float32)) for a in (
        (q[:, some] * qscale).transpose(1, 0, 2), k[:, some].transpose(1, 0, 2), qkv[:, 2, some].transpose(1, 2, 0))]
    ref = X.DevBuf(ctx, (n, len(some) * 72), np.float32)
    X.call("exn_vis_attend", ctx.h, n, len(some), f32[0].h, f32[1].h, f32[2].h, ref.h)
    e, ef = xo.rel_l2(mine, want), xo.rel_l2(ref.get().reshape(n, -1, 72), want)
    say("vis_attend_s", n, heads, "relative distance", e, "fp32", ef)
    assert e < 1.05 * ef


def vo_attention64(q, k, v):
    out = np.empty_like(v)
    for h in range(q.shape[1]):
        s = q[:, h] @ k[:, h].T / math.sqrt(72)
        p = np.exp(s - s.max(1, keepdims=True))
        out[:, h] = p @ v[:, h] / p.sum(1, keepdims=True)
    return out


@pytest.mark.parametrize("rows,cols,period,gelu", [(100, 1152, 1152, 0), (67, 4608, 1152, 1), (3, 72, 36, 1)])
def test_spreads(ctx, rows, cols, period, gelu):
    """The outputs' mean squares and the largest row norm over deviation, sums in double; a row of
    zeros counts for nothing, one whose columns all meet zero gains makes it infinite."""
    rng = np.random.default_rng(rows)
    w = rng.standard_normal((rows, cols)).astype(np.float32)
    g, b = rng.standard_normal(period).astype(np.float32), (0.1 * rng.standard_normal(period)).astype(np.float32)
    bias = rng.standard_normal(rows).astype(np.float32)
    w[1] = 0
    w[2] *= np.float32(2.0 ** -80)
    g[5] = b[5] = 0
    for lost in (False, True):
        if lost:
            w[0] = 0
            w[0, 5] = 1
        a2, t2, sp = (X.DevBuf(ctx, (k,), np.float64) for k in (period, rows, 2))
        dw, dg, db, dbias = dev(ctx, w), dev(ctx, g), dev(ctx, b), dev(ctx, bias)
        X.call("exn_vis_spread", ctx.h, rows, cols, dw.h, dg.h, db.h, period, dbias.h, gelu, a2.h, t2.h, sp.h)
        wa2 = g.astype(np.float64) ** 2 + b.astype(np.float64) ** 2
        w2 = w.astype(np.float64) ** 2
        t, q = w2 @ np.tile(wa2, cols // period), w2.sum(1)
        want = t + bias.astype(np.float64) ** 2
        if gelu:
            from scipy.special import erf
            f = lambda v: (0.5 * v * (1 + erf(v / math.sqrt(2)))) ** 2
            d = np.sqrt(3 * t)
            want = (f(bias - d) + 4 * f(bias.astype(np.float64)) + f(bias + d)) / 6
        assert np.abs(a2.get() - wa2).max() < 1e-15 * wa2.max()
        assert (np.abs(t2.get() - want) < 1e-11 * (want + 1e-12)).all()
        live = q > 0
        top = math.inf if lost else (q[live] / t[live]).max()
        assert sp.get()[0] == top or abs(sp.get()[0] / top - 1) < 1e-12
