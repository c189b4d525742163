"""The U-Net layers at every width of channel access (16 bytes per thread, or
one channel where the counts, offsets or addresses do not allow it), odd
rows and remainders, against the float64 reference or exactly."""
import ctypes

import numpy as np
import pytest

from oracle import unet_oracle as U

pytestmark = pytest.mark.gpu


def bits(a):
    return (np.ascontiguousarray(a, np.float32).view(np.uint32) >> 16).astype(np.uint16)


def unbits(a):
    return (a.astype(np.uint32) << 16).view(np.float32)


def at(a, nbytes):
    return ctypes.c_void_p(a.ptr.value + nbytes)


def rel(a, b):
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-30)


@pytest.mark.parametrize("C,Ct,c0", [(8, 24, 16), (8, 12, 4), (4, 8, 4), (3, 7, 2), (16, 16, 0), (40, 48, 8), (264, 264, 0)])
@pytest.mark.parametrize("shape", [(1, 1, 1, 1), (2, 1, 3, 5), (1, 2, 9, 33)], ids=str)
def test_layers(gpu, shape, C, Ct, c0):
    st = gpu
    from thesis_amd import nn
    print("[case] layers", shape, C, Ct, c0, flush=True)
    D = st.DeviceArray.from_numpy
    N, d, h, w = shape
    big, P = (N, 2 * d, 2 * h, 2 * w), N * d * h * w
    rng = np.random.default_rng(C + w)
    x = U.bf16_round(rng.standard_normal(big + (C,))).astype(np.float32)
    out = st.DeviceArray((P, C), np.uint16)
    nn.pool_fwd(D(bits(x)), out, shape, C)
    assert np.array_equal(out.numpy(), bits(U.bf16_round(U.pool(x.astype(np.float64)))).reshape(P, C))
    g = rng.standard_normal(shape + (C,)).astype(np.float32)
    g0 = rng.standard_normal(big + (C,)).astype(np.float32)
    gin = D(g0)
    nn.pool_bwd(D(g), gin, shape, C)
    assert rel(gin.numpy(), g0 + U.pool_bwd(g.astype(np.float64))) < 1e-6
    xs = U.bf16_round(rng.standard_normal(shape + (C,))).astype(np.float32)
    keep = rng.integers(0, 1 << 15, (8 * P, Ct)).astype(np.uint16)
    up = D(keep)
    nn.up_fwd(D(bits(xs)), up, shape, C, Ct, c0)
    keep[:, c0:c0 + C] = bits(U.up(xs)).reshape(8 * P, C)
    assert np.array_equal(up.numpy(), keep)
    gw = rng.standard_normal(big + (Ct,)).astype(np.float32)
    gs = st.DeviceArray(shape + (C,), np.float32)
    nn.up_bwd(D(gw), gs, shape, C, Ct, c0)
    assert rel(gs.numpy(), U.up_bwd(gw[..., c0:c0 + C].astype(np.float64))) < 1e-6
    # channel copies: bf16, float, float added
    for f32, acc in ((0, 0), (1, 0), (1, 1)):
        src = rng.standard_normal((P, C)).astype(np.float32)
        dst = rng.standard_normal((P, Ct)).astype(np.float32)
        ds, dd = (D(src), D(dst)) if f32 else (D(bits(src)), D(bits(dst)))
        nn.chan_copy(ds, dd, P, C, C, 0, Ct, c0, f32, bool(acc))
        want = dst if f32 else bits(dst)
        want[:, c0:c0 + C] = (want[:, c0:c0 + C] + src if acc else src) if f32 else bits(src)
        assert np.array_equal(dd.numpy(), want), (f32, acc)
    # relu backward with remainders, NaN and both zeros; from aligned and odd addresses
    n = P * C + 5
    y = rng.standard_normal(n + 1).astype(np.float32)
    y[::7], y[3::11], y[4::13] = 0.0, -0.0, np.nan
    yb, gv = bits(y), rng.standard_normal(n + 1).astype(np.float32)
    for off in (0, 1):
        o = D(np.full(n + 1, 7, np.uint16))
        dy, dg = D(yb), D(gv)
        nn.relu_bwd(at(dg, 4 * off), at(dy, 2 * off), at(o, 2 * off), n)
        want = np.full(n + 1, 7, np.uint16)
        want[off:off + n] = np.where(unbits(yb[off:off + n]) > 0, bits(U.bf16_round(gv[off:off + n])), 0)
        assert np.array_equal(o.numpy(), want), off


@pytest.mark.parametrize("C", [1, 2, 4, 8, 32, 64, 128, 256])
@pytest.mark.parametrize("P", [1, 77, 40009])
def test_bias_and_head(gpu, P, C):
    st = gpu
    from thesis_amd import nn
    print("[case] bias", P, C, flush=True)
    D = st.DeviceArray.from_numpy
    rng = np.random.default_rng(P + C)
    # one spare element in front, so that an odd address can be given
    x = U.bf16_round(rng.standard_normal(P * C + 1)).astype(np.float32)
    db0 = rng.standard_normal(C).astype(np.float32)
    dx = D(bits(x))
    for off in (0, 1):
        v = x[off:off + P * C].reshape(P, C).astype(np.float64)
        db = D(db0)
        nn.bias_grad(at(dx, 2 * off), db, P, C)
        # float sums of P terms over at least 64 partial sums
        bound = 1e-6 * np.abs(v).sum(0) + 1e-6
        assert (np.abs(db.numpy() - (db0 + v.sum(0))) <= bound).all(), off
        w = rng.standard_normal(C).astype(np.float32)
        y = st.DeviceArray((P,), np.float32)
        nn.head_fwd(at(dx, 2 * off), D(w), D(np.array([0.5], np.float32)), y, P, C)
        assert (np.abs(y.numpy() - (0.5 + v @ w)) <= 3e-5 * (1 + np.abs(v) @ np.abs(w))).all()
    P16 = P * C // 16
    if not P16:
        return
    for off in (0, 1):
        v = x[off:off + P16 * 16].reshape(P16, 16).astype(np.float64)
        w = rng.standard_normal(16).astype(np.float32)
        gy = rng.standard_normal(P16).astype(np.float32)
        gx, dw, db = D(np.zeros(P16 * 16, np.float32)), D(np.zeros(16, np.float32)), D(np.zeros(1, np.float32))
        nn.head_bwd(at(dx, 2 * off), D(w), D(gy), gx, dw, db, P16, 16)
        assert np.array_equal(gx.numpy().reshape(P16, 16), gy[:, None] * w)
        g64 = gy.astype(np.float64)
        assert (np.abs(dw.numpy() - g64 @ v) <= 1e-6 * (np.abs(g64) @ np.abs(v)) + 1e-6).all()
        assert abs(db.numpy()[0] - g64.sum()) <= 1e-6 * np.abs(g64).sum() + 1e-6
