"""The resident form (every sweep of a dispatch in one launch, the field in
registers; AUTO's choice for small 3D grids of radius 1, and the persistent
batch mode's for equal grids) against the oracle, both buffers bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _fields(nx, ny, nz, dt, equal, seed):
    rng = np.random.default_rng(seed)
    u1 = rng.random((nz, ny, nx)).astype(dt)
    return u1, (u1.copy() if equal else rng.random((nz, ny, nx)).astype(dt))


def _params(st, nx, ny, nz, its, op, dt):
    return st.StencilParams.make(nx=nx, ny=ny, nz=nz, radius=1, iterations=its, op=op,
                                 dtype=st.F64 if dt == np.float64 else st.F32, variant="auto", heuristic=1)


# one and several blocks along y and z, partial last blocks of one row and one
# plane, rows that end in the middle of a lane's columns, each number of
# columns per lane, planes per block and rows per block
SHAPES = [(64, 8, 6), (40, 9, 7), (63, 17, 33), (65, 33, 18), (128, 40, 130), (127, 70, 66), (130, 24, 50),
          (255, 33, 40), (61, 140, 125), (96, 96, 96)]


@pytest.mark.parametrize("nx,ny,nz", SHAPES)
@pytest.mark.parametrize("dt", [np.float32, np.float64], ids=["f32", "f64"])
def test_resident_form_matches_oracle(gpu, oracle, nx, ny, nz, dt):
    st = gpu
    for op, equal, its in ((1, True, 24), (1, False, 25), (0, False, 27)):
        p = _params(st, nx, ny, nz, its, op, dt)
        cfg = st.launch_config(p)
        assert cfg["launches"] == 1 and cfg["temporal_steps"] == its
        print("[case] resident", nx, ny, nz, dt.__name__, op, equal, its, flush=True)
        u1, u2 = _fields(nx, ny, nz, dt, equal, nx + ny + nz)
        a, b = u1.copy(), u2.copy()
        oracle.run(a, b, 3, 1, op, its)
        d1, d2 = st.DeviceArray.from_numpy(u1), st.DeviceArray.from_numpy(u2)
        in_u2, _ = st.dispatch_kernels(p, d1, d2)
        assert in_u2 == bool(its % 2)
        assert np.array_equal(d1.numpy().view(np.uint8), a.view(np.uint8))
        assert np.array_equal(d2.numpy().view(np.uint8), b.view(np.uint8))


def test_resident_batch_matches_oracle(gpu, oracle):
    st = gpu
    nx, ny, nz, n = 64, 40, 33, 8
    s = st.Stream()
    for its in (24, 33):
        us = [_fields(nx, ny, nz, np.float32, i % 2 == 0, 100 + i) for i in range(n)]
        dev = [(st.DeviceArray.from_numpy(a), st.DeviceArray.from_numpy(b)) for a, b in us]
        probs = [dict(nx=nx, ny=ny, nz=nz, radius=1, iterations=its, op=1, u1=d1, u2=d2) for d1, d2 in dev]
        print("[case] resident batch", its, flush=True)
        st.dispatch_batched(probs, (), st.BATCH_PERSISTENT, stream=s, timed=True)
        s.sync()
        for (a, b), (d1, d2) in zip(us, dev):
            oracle.run(a, b, 3, 1, 1, its)
            assert np.array_equal(d1.numpy().view(np.uint32), a.view(np.uint32))
            assert np.array_equal(d2.numpy().view(np.uint32), b.view(np.uint32))


def test_resident_dispatches_on_two_streams(gpu, oracle):
    """Back to back on two streams, each filling the card by itself, with
    changing shapes on one stream (the exchange buffers and tags go on)."""
    st = gpu
    sa, sb = st.Stream(), st.Stream()
    runs = []
    for k, (nx, ny, nz) in enumerate([(128, 128, 128), (64, 64, 64), (128, 128, 128), (200, 60, 50)]):
        for s in (sa, sb):
            u1, u2 = _fields(nx, ny, nz, np.float32, False, 7 * k + (s is sa))
            runs.append((s, _params(st, nx, ny, nz, 26, 1, np.float32), u1, u2,
                         st.DeviceArray.from_numpy(u1), st.DeviceArray.from_numpy(u2)))
    st.synchronize()
    print("[case] resident two streams", flush=True)
    for s, p, _, _, d1, d2 in runs:
        st.dispatch_kernels(p, d1, d2, stream=s)
    sa.sync()
    sb.sync()
    for _, p, u1, u2, d1, d2 in runs:
        oracle.run(u1, u2, 3, 1, 1, 26)
        assert np.array_equal(d1.numpy().view(np.uint32), u1.view(np.uint32))
        assert np.array_equal(d2.numpy().view(np.uint32), u2.view(np.uint32))
