"""The block form (several sweeps of a 2D block in registers per launch,
AUTO's choice for radius 1) against the oracle, both buffers bit for bit: at
the edges of its 64 x 32 blocks, with equal and different shells, and with
values whose quotient by the neighbour count is subnormal, infinite or NaN."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(st, p, u1, u2):
    d1, d2 = st.DeviceArray.from_numpy(u1), st.DeviceArray.from_numpy(u2)
    in_u2, _ = st.dispatch_kernels(p, d1, d2)
    st.synchronize()
    return (d1.numpy(), d2.numpy()), in_u2


def _same(got, want):
    w = got.dtype.itemsize
    it = np.uint32 if w == 4 else np.uint64
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan)
    assert np.array_equal(got.view(it)[~nan], want.view(it)[~nan])


@pytest.mark.parametrize("nx,ny", [(8, 8), (63, 31), (64, 32), (65, 33), (110, 46), (111, 47), (300, 71)])
@pytest.mark.parametrize("dt", ["f32", "f64"])
@pytest.mark.parametrize("op,equal", [(1, True), (1, False), (0, False)])
def test_block_form_matches_oracle(gpu, oracle, nx, ny, dt, op, equal):
    st = gpu
    rng = np.random.default_rng(nx * 1000 + ny)
    npdt = np.float32 if dt == "f32" else np.float64
    u1 = rng.random((1, ny, nx)).astype(npdt)
    u2 = u1.copy() if equal else rng.random((1, ny, nx)).astype(npdt)
    for its in (4, 5, 11, 24):
        print("[case] block", nx, ny, dt, op, equal, its, flush=True)
        p = st.StencilParams.make(nx=nx, ny=ny, nz=1, dimensions=2, radius=1, iterations=its, op=op,
                                  dtype=st.F64 if dt == "f64" else st.F32, variant="auto", heuristic=1)
        assert st.launch_config(p)["temporal_steps"] == 9
        a, b = u1.copy().reshape(ny, nx), u2.copy().reshape(ny, nx)
        oracle.run(a, b, 2, 1, op, its)
        (g1, g2), in_u2 = _run(st, p, u1, u2)
        assert in_u2 == bool(its % 2)
        _same(g1.reshape(ny, nx), a)
        _same(g2.reshape(ny, nx), b)


@pytest.mark.parametrize("dt", ["f32", "f64"])
@pytest.mark.parametrize("scale", ["tiny", "huge", "mixed"])
def test_block_form_quotient_at_the_limits(gpu, oracle, dt, scale):
    st = gpu
    npdt = np.float32 if dt == "f32" else np.float64
    fi = np.finfo(npdt)
    rng = np.random.default_rng(11)
    nx, ny, its = 97, 53, 5
    u = rng.standard_normal((ny, nx)).astype(npdt)
    with np.errstate(all="ignore"):
        if scale == "tiny":
            u = (u * npdt(6) * fi.smallest_subnormal).astype(npdt)
        elif scale == "huge":
            u = (u * fi.max / npdt(4)).astype(npdt)
        else:
            u = np.ldexp(u, rng.integers(fi.minexp - 20, fi.maxexp - 2, u.shape)).astype(npdt)
            u[rng.random(u.shape) < 0.2] = npdt(-0.0)
            u[17, 40] = np.inf
            u[30, 60] = np.nan
    p = st.StencilParams.make(nx=nx, ny=ny, nz=1, dimensions=2, radius=1, iterations=its, op=0,
                              dtype=st.F64 if dt == "f64" else st.F32, variant="auto", heuristic=1)
    print("[case] block quotient", dt, scale, flush=True)
    a, b = u.copy(), np.zeros_like(u)
    oracle.run(a, b, 2, 1, 0, its)
    (g1, g2), _ = _run(st, p, u, np.zeros_like(u))
    _same(g1, a)
    _same(g2, b)


@pytest.mark.parametrize("op", [0, 1])
@pytest.mark.parametrize("its", [8, 9, 24])
def test_block_form_without_last_single_pass(gpu, oracle, op, its):
    """Planes whose family is the streaming form: the result, and the shell
    of the other buffer, whose interior is then unspecified."""
    st = gpu
    nx, ny = 2056, 2049
    print("[case] block, no single pass", op, its, flush=True)
    rng = np.random.default_rng(its)
    u1, u2 = (rng.random((1, ny, nx)).astype(np.float32) for _ in range(2))
    p = st.StencilParams.make(nx=nx, ny=ny, nz=1, dimensions=2, radius=1, iterations=its, op=op, variant="auto",
                              heuristic=1)
    cfg = st.launch_config(p)
    assert cfg["temporal_steps"] in (5, 7, 9) and cfg["launches"] * cfg["temporal_steps"] < its + 2 * cfg["temporal_steps"]
    a, b = u1.copy().reshape(ny, nx), u2.copy().reshape(ny, nx)
    oracle.run(a, b, 2, 1, op, its)
    got, in_u2 = _run(st, p, u1, u2)
    assert in_u2 == bool(its % 2)
    _same(got[its % 2].reshape(ny, nx), (a, b)[its % 2])
    other, want = got[1 - its % 2].reshape(ny, nx), (a, b)[1 - its % 2]
    for cut in (np.s_[0], np.s_[-1], np.s_[:, 0], np.s_[:, -1]):
        _same(other[cut], want[cut])
