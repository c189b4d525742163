"""THESIS sweeps whose quotient by the neighbour count is subnormal, a tie,
infinite or NaN, in the kernels that multiply by the reciprocal and correct:
row forms (consecutive and quad layout), streaming forms in 3D and 2D."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FORMS = [("smem_register", (256, 20, 19), 1), ("smem_register", (384, 18, 21), 4), ("smem_register", (128, 20, 19), 1),
         ("smem_register", (128, 21, 20), 3), ("coop", (512, 24, 20), 1), ("coop", (256, 37, 1), 1)]


@pytest.mark.parametrize("dt", ["f32", "f64"])
@pytest.mark.parametrize("scale", ["tiny", "huge", "mixed"])
@pytest.mark.parametrize("variant,shape,r", FORMS)
def test_quotient_ranges(gpu, oracle, variant, shape, r, scale, dt):
    st = gpu
    if variant == "coop" and dt == "f64":
        pytest.skip("the streaming forms are FP32")
    nx, ny, nz = shape
    dims = 3 if nz > 1 else 2
    print("[case] quotient", variant, shape, r, scale, dt, flush=True)
    npdt = np.float32 if dt == "f32" else np.float64
    fi = np.finfo(npdt)
    rng = np.random.default_rng(nx + ny + r)
    u = rng.standard_normal((nz, ny, nx)).astype(npdt)
    if scale == "tiny":
        u = (u * fi.smallest_subnormal * 50).astype(npdt)
    elif scale == "huge":
        u = np.ldexp(u, fi.maxexp - 4).astype(npdt)
    else:
        u = np.ldexp(u, rng.integers(fi.minexp - 20, fi.maxexp - 2, u.shape)).astype(npdt)
        u[rng.random(u.shape) < 0.1] = npdt(-0.0)
        u[rng.random(u.shape) < 1e-3] = npdt(np.inf)
    for its in (2, 8):
        a, b = u.copy(), u.copy()
        d1, d2 = st.DeviceArray.from_numpy(u), st.DeviceArray.from_numpy(u)
        p = st.StencilParams.make(nx=nx, ny=ny, nz=nz, dimensions=dims, radius=r, iterations=its, op=0,
                                  dtype=st.F64 if dt == "f64" else st.F32, variant=variant, heuristic=1)
        st.dispatch_kernels(p, d1, d2)
        with np.errstate(all="ignore"):
            oracle.run(*((a, b) if dims == 3 else (a.reshape(ny, nx), b.reshape(ny, nx))), dims, r, 0, its)
        got, it = d1.numpy().reshape(a.shape), np.uint32 if dt == "f32" else np.uint64
        nan = np.isnan(a)
        assert np.array_equal(np.isnan(got), nan), its
        assert np.array_equal(got.view(it)[~nan], a.view(it)[~nan]), its
        d1.free()
        d2.free()
