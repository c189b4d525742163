"""The tiled convolution kernels (forward, backward data, weight gradient) at
the edges of their 16 x 4 x 2/4 tiles and channel blocks, against the FP64
restatement: relative L2 error 1e-5 per layer, as for the other layers (FP32
accumulation of at most 27*128 products: sqrt(3456) * 2^-24 = 3.5e-6 of the
products' norm)."""
import numpy as np
import pytest

from oracle import unet_oracle as U
from test_gpu_unet import _conv_case, bits, rel

pytestmark = pytest.mark.gpu

SHAPES = [(1, 4, 4, 16), (1, 5, 5, 17), (2, 3, 7, 33), (1, 1, 1, 1), (1, 9, 2, 15)]
CHANNELS = [(8, 4), (16, 16), (24, 20), (32, 64), (40, 12), (48, 16), (16, 48), (96, 32), (32, 96), (128, 36)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("ci,co", CHANNELS)
def test_conv_tiles(gpu, shape, ci, co):
    st = gpu
    from thesis_amd import nn
    print("[case] conv tiles", shape, ci, co, flush=True)
    rng = np.random.default_rng(ci * 1000 + co)
    N, D, H, W = shape
    P = N * D * H * W
    x, w, f32, b16, want = _conv_case(st, nn, rng, shape, ci, co, True)
    assert rel(f32, want) < 1e-5
    assert np.all(np.abs(b16 - f32) <= np.abs(f32) * 2 ** -8 + 1e-30)
    gy = U.bf16_round(rng.standard_normal(shape + (co,)))
    _, gw_ref, _ = U.conv3_bwd(x, w[:, :27 * ci], gy)
    dx = st.DeviceArray.from_numpy(bits(x).reshape(P, ci))
    dg = st.DeviceArray.from_numpy(bits(gy).reshape(P, co))
    before = np.zeros((co, nn.kpad(ci)), np.float32)
    before[:, 27 * ci:] = 3.0  # padding columns are not touched
    gw = st.DeviceArray.from_numpy(before)
    nn.conv3_wgrad(dx, dg, gw, shape, ci, co)
    nn.conv3_wgrad(dx, dg, gw, shape, ci, co)  # accumulates
    g = gw.numpy()
    assert rel(g[:, :27 * ci], 2 * gw_ref) < 1e-5
    assert np.all(g[:, 27 * ci:] == 3.0)


def test_conv_tiles_infinite_neighbour(gpu):
    """An infinity at the sample's edge reaches only the taps that see it:
    positions of a tile outside the sample add nothing to the weight
    gradient (0 * inf)."""
    st = gpu
    from thesis_amd import nn
    shape, ci, co = (1, 2, 3, 18), 8, 16
    rng = np.random.default_rng(3)
    x = U.bf16_round(rng.standard_normal(shape + (ci,)))
    gy = U.bf16_round(np.abs(rng.standard_normal(shape + (co,))) + 0.5)
    x[0, 1, 2, 17, 0] = np.inf
    xb = bits(np.where(np.isinf(x), 0, x)).reshape(-1, ci)
    xb[-1, 0] = 0x7F80
    dx = st.DeviceArray.from_numpy(xb)
    dg = st.DeviceArray.from_numpy(bits(gy).reshape(-1, co))
    gw = st.DeviceArray((co, nn.kpad(ci)), np.float32)
    gw.fill_zero()
    nn.conv3_wgrad(dx, dg, gw, shape, ci, co)
    g = gw.numpy()[:, :27 * ci].reshape(co, 27, ci)
    sees = np.zeros(27, bool)
    for t in range(27):
        dz, dy, dq = t // 9 - 1, t // 3 % 3 - 1, t % 3 - 1
        # position p with p + tap = the corner (1, 2, 17)
        sees[t] = 0 <= 1 - dz < 2 and 0 <= 2 - dy < 3 and 0 <= 17 - dq < 18
    assert np.all(np.isposinf(g[:, sees, 0])) and np.all(np.isfinite(g[:, ~sees, 0]))
    assert np.all(np.isfinite(g[:, :, 1:]))


def test_wgrad_streams_share_a_gradient(gpu):
    """Weight gradients on several streams add up in one array: whole numbers,
    so every order gives the same sums."""
    st = gpu
    from thesis_amd import nn
    shape, ci, co = (1, 8, 8, 16), 16, 16
    rng = np.random.default_rng(11)
    x = rng.integers(-3, 4, shape + (ci,)).astype(np.float64)
    gy = rng.integers(-3, 4, shape + (co,)).astype(np.float64)
    _, want, _ = U.conv3_bwd(x, np.zeros((co, 27 * ci)), gy)
    dx = st.DeviceArray.from_numpy(bits(x).reshape(-1, ci))
    dg = st.DeviceArray.from_numpy(bits(gy).reshape(-1, co))
    gw = st.DeviceArray((co, nn.kpad(ci)), np.float32)
    gw.fill_zero()
    streams = [st.Stream() for _ in range(4)]
    st.synchronize()
    print("[case] wgrad streams", flush=True)
    for _ in range(32):
        for s in streams:
            nn.conv3_wgrad(dx, dg, gw, shape, ci, co, stream=s)
    for s in streams:
        s.sync()
    assert np.array_equal(gw.numpy()[:, :27 * ci], 128 * want)
