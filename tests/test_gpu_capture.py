"""Dispatches in AUTO's newer forms, and the weight gradient, on a stream under
capture (first use of the stream's workspace included) and through the
no-alloc entry point: bit for bit what they give eagerly, also on replays with
other fields between which the program goes on with its own work."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (nx, ny, nz), radius, sweeps: resident (run by another form here), block, rolling, tile with
# and without the shell comparison
CASES = [((64, 64, 64), 1, 24), ((128, 128, 128), 1, 25), ((300, 200), 1, 24), ((1031, 1021), 3, 7), ((2051, 2053), 8, 4),
         ((130, 97, 90), 4, 9), ((130, 97, 90), 4, 2), ((129, 131, 127), 12, 5)]


def _params(st, shape, r, its, op):
    return st.StencilParams.make(nx=shape[0], ny=shape[1], nz=shape[2] if len(shape) == 3 else 1, dimensions=len(shape),
                                 radius=r, iterations=its, op=op, variant="auto", heuristic=1)


def _fields(shape, seed, equal):
    rng = np.random.default_rng(seed)
    a = rng.random(shape[::-1]).astype(np.float32)
    return a, (a.copy() if equal else rng.random(shape[::-1]).astype(np.float32))


class _Capture:
    def __init__(self, stream):
        self.hip, self.s, self.exec = C.CDLL("libamdhip64.so.7"), stream, C.c_void_p()

    def _ok(self, rc):
        assert rc == 0, rc

    def begin(self):
        self._ok(self.hip.hipStreamBeginCapture(self.s.handle, 0))  # global mode

    def end(self):
        graph = C.c_void_p()
        self._ok(self.hip.hipStreamEndCapture(self.s.handle, C.byref(graph)))
        self._ok(self.hip.hipGraphInstantiate(C.byref(self.exec), graph, None, None, C.c_size_t(0)))
        self._ok(self.hip.hipGraphDestroy(graph))

    def replay(self):
        self._ok(self.hip.hipGraphLaunch(self.exec, self.s.handle))
        self.s.sync()

    def close(self):
        self._ok(self.hip.hipGraphExecDestroy(self.exec))


@pytest.mark.parametrize("shape,r,its", CASES, ids=str)
def test_captured_dispatch(gpu, shape, r, its):
    st = gpu
    for op, equal in ((1, True), (0, False)):
        print("[case] captured", shape, r, its, op, equal, flush=True)
        p = _params(st, shape, r, its, op)
        want = []
        for seed in (1, 2):
            d1, d2 = (st.DeviceArray.from_numpy(a) for a in _fields(shape, seed, equal))
            in_u2, _ = st.dispatch_kernels(p, d1, d2)
            want.append((d2 if in_u2 else d1).numpy())
        s = st.Stream()
        cap = _Capture(s)
        d1, d2 = (st.DeviceArray.from_numpy(a) for a in _fields(shape, 0, equal))
        st.synchronize()
        cap.begin()
        in_u2, _ = st.dispatch_kernels(p, d1, d2, stream=s)
        cap.end()
        for seed, w in ((1, want[0]), (2, want[1]), (1, want[0])):
            a, b = _fields(shape, seed, equal)
            d1.copy_from(st.DeviceArray.from_numpy(a), s)
            d2.copy_from(st.DeviceArray.from_numpy(b), s)
            s.sync()
            cap.replay()
            assert np.array_equal((d2 if in_u2 else d1).numpy().view(np.uint32), w.view(np.uint32)), seed
            st.dispatch_kernels(_params(st, (333, 251, 207), 2, 4, 1), *(st.DeviceArray.from_numpy(x) for x in _fields((333, 251, 207), 9, True)),
                                stream=s)  # the program's own work on the stream
            s.sync()
        cap.close()


@pytest.mark.parametrize("shape,r,its", CASES, ids=str)
def test_noalloc_dispatch(gpu, shape, r, its):
    st = gpu
    f = st.lib().stencil_dispatch_noalloc
    f.argtypes = [C.POINTER(st.StencilParams), C.c_void_p, C.c_void_p, C.c_void_p, C.POINTER(C.c_int)]
    for op, equal in ((1, True), (0, False)):
        p = _params(st, shape, r, its, op)
        out = []
        for noalloc in (False, True):
            print("[case] noalloc", noalloc, shape, r, its, op, equal, flush=True)
            d1, d2 = (st.DeviceArray.from_numpy(a) for a in _fields(shape, 3, equal))
            flag = C.c_int(-1)
            if noalloc:
                assert f(C.byref(p), d1.ptr, d2.ptr, None, C.byref(flag)) == 0
                st.synchronize()
                in_u2 = bool(flag.value)
            else:
                in_u2, _ = st.dispatch_kernels(p, d1, d2)
            assert in_u2 == bool(its % 2)
            out.append((d2 if in_u2 else d1).numpy())
        assert np.array_equal(out[0].view(np.uint32), out[1].view(np.uint32))


def test_workspace_beside_a_capture(gpu):
    """A workspace that grows on one stream while another is under capture, and
    one that grows after a graph was captured with it."""
    st = gpu
    from thesis_amd import nn
    rng = np.random.default_rng(5)
    s, t = st.Stream(), st.Stream()

    def layer(n, ci, co):
        x, g = (st.DeviceArray.from_numpy((rng.standard_normal((n * 4096, c)).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16))
                for c in (ci, co))
        gw = st.DeviceArray((co, nn.kpad(ci)), np.float32)
        gw.fill_zero()
        return lambda stream: nn.conv3_wgrad(x, g, gw, (n, 16, 16, 16), ci, co, stream=stream), gw

    small, gs = layer(1, 16, 16)
    large, gl = layer(8, 64, 64)
    other, go = layer(8, 48, 16)
    st.synchronize()
    print("[case] workspace beside a capture", flush=True)
    cap = _Capture(t)
    small(s)
    cap.begin()
    other(t)   # recorded; first use of t's workspace
    large(s)   # s's workspace grows meanwhile
    cap.end()
    cap.replay()
    s.sync()
    a, b = go.numpy(), gl.numpy()
    assert a.any() and b.any()
    large(t)   # t's workspace grows; the graph keeps its block
    t.sync()
    cap.replay()
    assert np.array_equal(go.numpy(), 2 * a)   # accumulates: the same sums again
    assert np.array_equal(gl.numpy(), 2 * b)
    cap.close()
