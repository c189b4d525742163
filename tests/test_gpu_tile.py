"""The tile form of SMEM_REGISTER (the library's choice for row widths and
radii the row form does not serve as well) against the oracle, both buffers
bit for bit: widths around the 64-column tiles, heights around its 32 and 64
rows, every number of quads of x halo, equal and different shells."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (nx, ny, nz), radii; more than 2^20 cells (2^21 or 2^22 for the widest)
F32 = [((65, 129, 130), (1, 2, 3, 4)), ((130, 97, 90), (1, 4, 5)), ((63, 130, 131), (2, 5)), ((191, 66, 95), (3,)),
       ((192, 64, 96), (1, 4)), ((200, 161, 133), (6, 8)), ((129, 191, 172), (7, 9)), ((260, 130, 126), (10, 11, 12)),
       ((101, 105, 103), (6, 8, 12, 13)), ((129, 163, 200), (13, 14, 15, 16)), ((513, 129, 70), (16,))]
F64 = [((65, 129, 130), (1, 2, 3)), ((130, 97, 90), (4, 5)), ((194, 65, 90), (3, 4)), ((201, 161, 131), (6,)),
       ((101, 105, 103), (5, 6, 8)), ((129, 131, 127), (7, 9, 10)), ((194, 65, 170), (10,))]


@pytest.mark.parametrize("shape,radii,dt", [(s, r, np.float32) for s, r in F32] + [(s, r, np.float64) for s, r in F64],
                         ids=str)
def test_tile_form_matches_oracle(gpu, oracle, shape, radii, dt):
    st = gpu
    nx, ny, nz = shape
    for r in radii:
        for op, equal, its in ((1, True, 3), (0, False, 2)):
            print("[case] tile", shape, r, dt.__name__, op, equal, flush=True)
            rng = np.random.default_rng(nx + r)
            u1 = rng.random((nz, ny, nx)).astype(dt)
            u2 = u1.copy() if equal else rng.random((nz, ny, nx)).astype(dt)
            p = st.StencilParams.make(nx=nx, ny=ny, nz=nz, radius=r, iterations=its, op=op,
                                      dtype=st.F64 if dt == np.float64 else st.F32, variant="smem_register", heuristic=1)
            cfg = st.launch_config(p)
            assert cfg["block_x"] == 64 and cfg["block_y"] in (32, 64) and cfg["coarsen_x"] in (2, 4), cfg
            d1, d2 = st.DeviceArray.from_numpy(u1), st.DeviceArray.from_numpy(u2)
            in_u2, _ = st.dispatch_kernels(p, d1, d2)
            assert in_u2 == bool(its % 2)
            oracle.run(u1, u2, 3, r, op, its)
            assert np.array_equal(d1.numpy().view(np.uint8), u1.view(np.uint8)), (shape, r, op)
            assert np.array_equal(d2.numpy().view(np.uint8), u2.view(np.uint8)), (shape, r, op)
            d1.free()
            d2.free()
