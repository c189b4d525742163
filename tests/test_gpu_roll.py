"""The rolling form (AUTO's choice for 2D grids of radius 2 to 16) against the
oracle, both buffers bit for bit: widths around the segments of 256 (FP32) and
128 (FP64) columns and their stored parts, odd heights, a single segment,
passes of three sweeps and of one, equal and different shells."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (nx, ny): at least 2^20 cells; from 2^22 where the rule asks for them
SMALL = [(19, 60001), (255, 4133), (257, 4111), (1031, 1021), (4099, 259)]
LARGE = [(130, 32771), (2051, 2053)]
CASES = [(s, r, "f32") for s in SMALL for r in (2, 3, 5, 6, 7)] + [(s, r, "f32") for s in LARGE for r in (4, 8, 9, 12, 16)]
CASES += [(s, r, "f64") for s in SMALL[1:] for r in (2, 3, 5, 8, 16)] + [(s, 4, "f64") for s in LARGE]
CASES += [((2900, 2897), r, "f32") for r in (4, 5)]


@pytest.mark.parametrize("shape,r,dt", CASES, ids=str)
def test_roll_form_matches_oracle(gpu, oracle, shape, r, dt):
    st = gpu
    nx, ny = shape
    npdt = np.float32 if dt == "f32" else np.float64
    for op, equal, its in ((1, True, 4), (0, False, 5)):
        print("[case] roll", nx, ny, r, dt, op, equal, its, flush=True)
        rng = np.random.default_rng(nx + r)
        u1 = rng.random((ny, nx)).astype(npdt)
        u2 = u1.copy() if equal else rng.random((ny, nx)).astype(npdt)
        p = st.StencilParams.make(nx=nx, ny=ny, nz=1, dimensions=2, radius=r, iterations=its, op=op,
                                  dtype=st.F64 if dt == "f64" else st.F32, variant="auto", heuristic=1)
        cfg = st.launch_config(p)
        deep = r <= 3 or u1.nbytes >= 2 ** 25 * 2 ** (r - 4) and r <= (6 if dt == "f32" else 5)
        # one pass of three sweeps, then single ones
        assert (cfg["temporal_steps"], cfg["launches"]) == ((3, its - 2) if deep else (1, its)), cfg
        d1, d2 = st.DeviceArray.from_numpy(u1), st.DeviceArray.from_numpy(u2)
        in_u2, _ = st.dispatch_kernels(p, d1, d2)
        assert in_u2 == bool(its % 2)
        oracle.run(u1, u2, 2, r, op, its)
        it = np.uint32 if dt == "f32" else np.uint64
        assert np.array_equal(d1.numpy().reshape(ny, nx).view(it), u1.view(it)), (op, its)
        assert np.array_equal(d2.numpy().reshape(ny, nx).view(it), u2.view(it)), (op, its)
        d1.free()
        d2.free()
