"""The library's host side where there is no GPU: which kernels a call
launches, what it does when the runtime refuses something, under capture and
from several threads.  Each case runs in its own process on a stand-in for the
HIP runtime (tests/hostsim/hip_standin.cpp), whose kernels do nothing."""
import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import ctypes as C, re, sys, threading, time
sys.path.insert(0, {root!r})
R = C.CDLL({lib!r}, mode=C.RTLD_GLOBAL)
log, answer = [], {{}}   # (event, handle, size, thread); event -> result or function
@C.CFUNCTYPE(C.c_int, C.c_char_p, C.c_void_p, C.c_size_t, C.POINTER(C.c_void_p))
def hook(event, handle, size, args):
    event = event.decode()
    m = re.search(r"k_[a-z0-9_]+", event)
    name = m.group(0).rstrip("0123456789") if m else event
    if m: name = re.match(r"\\d+(k_\\w+)", event[re.search(r"\\d+k_", event).start():]).group(1)[:int(re.search(r"(\\d+)k_", event).group(1))]
    log.append((name, handle, size, threading.get_ident()))
    a = answer.get(name, 0)
    return a(handle, size, args) if callable(a) else a
R.standin_hook(hook)
def kernels(): return [e[0] for e in log if e[0].startswith("k_")]
import thesis_amd as st
from thesis_amd import nn
def auto(nx, ny, nz=None, **kw):
    kw = dict(dict(op=1, variant="auto", heuristic=1, iterations=4), **kw)
    return st.StencilParams.make(nx=nx, ny=ny, nz=nz or 1, dimensions=3 if nz else 2, **kw)
A, B = 1 << 20, 1 << 40  # addresses of buffers that no kernel touches
"""


@pytest.fixture(scope="session")
def host(tmp_path_factory, st):
    lib = str(tmp_path_factory.mktemp("standin") / "libamdhip64.so.7")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-std=c++17", "-Wl,-soname,libamdhip64.so.7", "-o", lib,
                    os.path.join(HERE, "hostsim", "hip_standin.cpp")], check=True)

    def run(body):
        script = PRELUDE.format(root=ROOT, lib=lib) + textwrap.dedent(body)
        r = subprocess.run([sys.executable, "-c", script], capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stdout + r.stderr
    return run


def test_wgrad_forms(host):
    """Wide inputs and channel counts that are no multiple of 4 stay on the
    tiled weight gradient; tiles that are mostly padding and a handful of
    positions go to the kernels without tiles."""
    host("""
    def route(shape, ci, co):
        log.clear()
        nn.conv3_wgrad(A, A, A, shape, ci, co)
        return kernels()
    TILE, ROWS, GATHER = ["k_conv3_wgrad_tile", "k_wgrad_reduce"], ["k_pc_transpose"] * 2 + ["k_conv3_wgrad_t"], ["k_conv3_wgrad"]
    for ci, co in ((96, 32), (104, 16), (112, 64), (128, 36), (128, 128), (176, 32), (16, 6), (32, 1), (24, 18)):
        for shape in ((8, 16, 16, 16), (8, 8, 8, 8), (2, 33, 33, 33)):
            assert route(shape, ci, co) == TILE, (shape, ci, co, route(shape, ci, co))
    assert route((1, 1, 1, 100000), 64, 64) == ROWS       # 1 of 16 rows of a tile, whole octets of positions
    assert route((1, 20000, 1, 1), 64, 64) == GATHER      # 1 of 64 positions
    assert route((1, 20000, 1, 1), 16, 16) == TILE
    assert route((1, 2, 2, 8), 64, 64) == GATHER and route((8, 4, 4, 1), 152, 120) == GATHER
    assert route((1, 4, 4, 4), 16, 16) == TILE and route((4, 4, 4, 4), 64, 64) == TILE
    assert route((1, 1, 1, 1000), 64, 64) == TILE
    assert route((8, 16, 16, 16), 192, 32) == GATHER      # no tile fits
    """)


def test_conv_forms(host):
    """The tiled convolution where its tiles are filled and fill the card, the
    kernel without tiles elsewhere."""
    host("""
    def route(shape, ci, co):
        log.clear()
        nn.conv3(A, A, A, A, None, shape, ci, co)
        return kernels()
    for shape, ci, co in (((8, 64, 64, 64), 48, 16), ((8, 64, 64, 64), 16, 48), ((8, 16, 16, 16), 64, 64),
                          ((8, 32, 32, 32), 96, 32), ((8, 32, 32, 32), 64, 64), ((4, 4, 4, 4), 16, 16), ((1, 2, 2, 2), 8, 16),
                          ((8, 8, 1, 60), 40, 40), ((6, 9, 1, 21), 32, 52)):
        assert route(shape, ci, co) == ["k_conv3_tile"], (shape, ci, co)
    for shape, ci, co in (((1, 1, 1, 100000), 16, 16), ((1, 300, 300, 3), 64, 64), ((4, 20, 20, 20), 128, 128),
                          ((1, 40, 40, 40), 64, 80), ((8, 32, 32, 32), 64, 80), ((64, 8, 8, 8), 64, 256),
                          ((4000, 2, 2, 2), 8, 16), ((1, 1, 300, 301), 32, 32), ((7, 13, 34, 63), 80, 96)):
        assert route(shape, ci, co) == ["k_conv3"], (shape, ci, co)
    """)


def test_mixed_small_kernels(host):
    """The 16-bit modes off the row kernels: one flat kernel per pass."""
    host("""
    p = auto(17, 300, 300, radius=4, dtype=st.BF16, iterations=3, restart=10)
    sizes = []
    answer["k_mx_sweep"] = lambda stream, size, args: sizes.append(size) or 0
    st.dispatch_mixed(p, A, A, A, A, A)
    cells = 9 * 292 * 292
    assert kernels().count("k_mx_defect") == 1 and sizes == [-(-cells // 256)] * 3, (kernels(), sizes)
    """)


def test_mixed_lane_kernels(host):
    """64 x 4 threads per workgroup where the grid is small or its rows fill the
    wavefronts, the flat kernels elsewhere."""
    host("""
    def route(dims, nx, ny, nz, radius):
        log.clear()
        p = st.StencilParams.make(nx=nx, ny=ny, nz=nz, dimensions=dims, radius=radius, op=1, dtype=st.BF16,
                                  iterations=3, restart=10)
        st.dispatch_mixed(p, A, A, A, A, A)
        return [k.split("<")[0] for k in kernels() if "sweep" in k or "defect" in k]
    for call in ((3, 256, 256, 256, 8), (3, 123, 284, 71, 1), (3, 123, 284, 71, 2), (2, 2048, 2048, 1, 16),
                 (3, 41, 41, 41, 5), (2, 88, 2912, 1, 8), (2, 59, 202, 1, 14), (3, 114, 99, 104, 10)):
        assert route(*call) == ["k_mx_defect_rows"] + ["k_mx_sweep_rows"] * 3, (call, kernels())
    for call in ((3, 123, 284, 71, 3), (3, 333, 251, 207, 6), (3, 70, 70, 70, 2), (3, 67, 123, 194, 1), (3, 97, 50, 351, 14),
                 (2, 11, 100000, 1, 4), (2, 41, 3001, 1, 5), (2, 2048, 2048, 1, 5)):
        assert route(*call) == ["k_mx_defect"] + ["k_mx_sweep"] * 3, (call, kernels())
    """)


def test_layer_grids(host):
    """Workgroups of the layers that move bytes follow the groups of channels,
    whatever the shape; a loss over many values takes more blocks."""
    host("""
    def grid(name, call):
        got = []
        answer[name] = lambda stream, size, args: got.append(size) or 0
        call()
        return got[0]
    for n, d, h, w in ((8, 32, 32, 32), (1, 50000, 1, 1), (64, 2, 2, 2)):
        for c, v in ((16, 8), (20, 1), (3, 1)):
            assert grid("k_pool_fwd", lambda: nn.pool_fwd(A, A, (n, d, h, w), c)) == -(-n * d * h * w * c // v // 256)
    assert grid("k_chan_copy", lambda: nn.chan_copy(A, A, 1 << 21, 64, 76, 4, 140, 0, 0)) == 65536
    assert grid("k_sumsq", lambda: nn.sumsq(A, A, A, 1 << 21, 1.0)) == 512
    assert grid("k_sumsq", lambda: nn.sumsq(A, A, A, 1 << 25, 1.0)) == 2048
    """)


def test_roll_plan(host):
    """The rolling form's chunks are the best of every chunk count, found
    without trying them all."""
    host("""
    import ctypes, math, random
    def exhaustive(nx, ny, r, es, steps):
        cx = 16 // es; ln = 64 * cx; h = (r * steps + cx - 1) // cx * cx
        nseg = 1 if nx <= ln else -(-(nx - ln) // (ln - 2 * h)) + 1
        occ = min(8, 512 // (8 * r * steps + (84 if es == 8 else 72)))
        share = lambda k: (0.0, 1.7, 2.26)[k] if k < 3 else float(k)
        best = None
        for nch in range(1, ny + 1):
            rows = -(-ny // nch)
            if nch > 1 and rows < 8: break
            waves = nseg * -(-ny // rows); per = -(-waves // 1024)
            cost = (per // occ * share(occ) + share(per % occ)) * (rows + 2 * steps * r)
            if best is None or cost < best[0]: best = (cost, rows, waves)
        return best[1:]
    rng = random.Random(7)
    got = []
    answer["k_roll"] = lambda stream, size, args: got.append(tuple(ctypes.cast(args[2], ctypes.POINTER(ctypes.c_int))[3:5])) or 0
    shapes = [(8192, 8192, 4, 0), (19, 60001, 2, 0), (4099, 259, 7, 0), (2051, 2053, 16, 1)]
    for _ in range(40):
        nx = int(2 ** rng.uniform(5, 13)); shapes.append((nx, int(2 ** 22.1 / nx * rng.uniform(1, 8)), rng.randint(2, 12), rng.randint(0, 1)))
    taken = 0
    for nx, ny, r, f64 in shapes:
        if min(nx, ny) <= 2 * r: continue
        p = auto(nx, ny, radius=r, dtype=st.F64 if f64 else st.F32, iterations=4)
        got.clear()
        try: st.dispatch_kernels(p, A, B)
        except st.StencilError: continue  # beyond the launch limits of the family that AUTO names
        if not got: continue
        taken += 1
        steps = st.launch_config(p)["temporal_steps"]
        rows, waves = exhaustive(nx, ny, r, 8 if f64 else 4, steps)
        assert got[0] == (waves, rows), (nx, ny, r, f64, got[0], (waves, rows))
    assert taken > 25
    p = auto(5, 20000000, radius=2, iterations=4)
    best = 1e9
    for _ in range(5):
        t0 = time.perf_counter(); st.dispatch_kernels(p, A, B); best = min(best, time.perf_counter() - t0)
    assert best < 2e-3, best
    """)


def test_tile_plan(host):
    """The tile form's rows and z chunk are the best of every chunk count,
    found without trying them all."""
    host("""
    import random
    def exhaustive(nx, ny, nz, r, es):
        cx = 2 if r > (5 if es == 8 else 12) else 4
        best = None
        for ry in (1, 2):
            words = 2 * r * ry * cx * es // 4
            if ry == 2 and cx == 2 or cx == 4 and words > (112 if ry == 2 else 96): continue
            lds = 2 * (32 * ry + 2 * r) * ((64 + 2 * ((r + 3) // 4 * 4)) * es // 16) * 16
            two = words <= 40 and lds <= 80 * 1024
            xy = -(-nx // 64) * -(-ny // (32 * ry)); room = 512 if two else 256
            for nch in range(1, nz + 1):
                ch = -(-nz // nch)
                if nch > 1 and ch < 3: break
                n = xy * -(-nz // ch)
                light, full = 1.15 * (ch + 0.3 * 2 * r), ch + 2.0 * r
                cost = -(-n // room) * (light if cx == 2 or light < full else full) * (ry + 0.6) * (1.6 if two else 1.0)
                if best is None or cost < best[0]: best = (cost, 32 * ry, ch, n)
        return best[1:]
    rng = random.Random(11)
    taken = 0
    for _ in range(300):
        nx, ny = (int(2 ** rng.uniform(4, 10)) for _ in "xy")
        nz = int(2 ** 20 / nx / ny * 2 ** rng.uniform(0.5, 6)); r = rng.randint(1, 16); f64 = rng.random() < 0.4
        if not 2 * r < min(nx, ny, nz) or nz > 60000: continue
        p = auto(nx, ny, nz, radius=r, dtype=st.F64 if f64 else st.F32, variant="smem_register")
        try: c = st.launch_config(p)
        except st.StencilError: continue
        if c["block_x"] != 64 or c["block_y"] not in (32, 64) or c["grid_y"] != 1 or c["zchunk"] != c["block_z"]: continue
        want = exhaustive(nx, ny, nz, r, 8 if f64 else 4)
        if (c["block_y"], c["zchunk"], c["grid_x"]) != want:
            # another form's numbers, or a plan of the same cost
            raise AssertionError((nx, ny, nz, r, f64, c, want))
        taken += 1
    assert taken > 60, taken
    p = auto(40, 40, 1000000, radius=3, variant="smem_register")
    best = 1e9
    for _ in range(5):
        t0 = time.perf_counter(); st.sweep(p, A, B); best = min(best, time.perf_counter() - t0)
    assert kernels()[-1] == "k_tile" and best < 1e-3, (kernels()[-1], best)
    """)


def test_small_interiors(host):
    """Grids whose interior is a small part of their tiles stay with the kernels
    they had: the register march or the plain kernel."""
    host("""
    def route(nx, ny, nz, r, dt=st.F32):
        log.clear()
        st.dispatch_kernels(auto(nx, ny, nz, radius=r, dtype=dt, iterations=2), A, B)
        return kernels()[-1]
    march = {(1000, 33, 33): (6, 8), (4000, 20, 20): (6, 8), (40, 4000, 20): (8,), (90, 548, 34): (8,), (9, 9, 100000): (1,)}
    plain = {(1000, 33, 33): (10, 12), (104, 104, 104): (10, 12), (33, 33, 2000): (12,), (33, 33, 5000): (16,)}
    plain64 = {(1000, 33, 33): (5, 6, 8), (4000, 20, 20): (5, 6, 8), (33, 33, 2000): (10,), (12000, 12000, 11): (5,)}
    tile = {(1000, 33, 33): (2, 4), (1000, 1000, 20): (6, 8), (2000, 500, 24): (10,), (104, 104, 104): (6, 8), (64, 64, 400): (12,),
            (128, 128, 128): (6, 8, 10, 12), (333, 251, 207): (1, 2, 6, 12, 16), (20, 20, 40000): (2, 8)}
    tile64 = {(128, 128, 128): (3, 5, 8, 10), (104, 104, 104): (5, 6, 8), (40, 4000, 20): (6, 8), (2000, 500, 24): (10,)}
    for want, dt, cases in (("k_march", st.F32, march), ("k_base", st.F32, plain), ("k_base", st.F64, plain64),
                            ("k_tile", st.F32, tile), ("k_tile", st.F64, tile64), ("k_rowc", st.F64, {(256, 256, 256): (3,)})):
        for shape, radii in cases.items():
            for r in radii: assert route(*shape, r, dt).startswith(want), (shape, r, dt, route(*shape, r, dt))
    """)


def test_tile_shell_comparison(host):
    """A short run in the tile form does not pay for comparing the shells."""
    host("""
    def compared(n, r, its):
        log.clear()
        st.dispatch_kernels(auto(n, n, n, radius=r, iterations=its), A, B)
        assert kernels()[-1] == "k_tile"
        return "k_grid_shell_eq" in kernels()
    assert not compared(128, 6, 2) and compared(128, 6, 8) and not compared(320, 2, 1) and compared(320, 2, 2)
    """)


def test_roll_small_planes(host):
    """Planes that are mostly shell rows, and few sweeps of radius 2 over small
    planes of whole quads, stay with the kernels they had."""
    host("""
    def rolls(nx, ny, r, its=16, dt=st.F32, op=1):
        log.clear()
        st.dispatch_kernels(auto(nx, ny, radius=r, dtype=dt, iterations=its, op=op), A, B)
        return kernels()[-1] == "k_roll"
    assert not rolls(100000, 40, 16, dt=st.F64) and rolls(100000, 40, 12, dt=st.F64)
    assert not rolls(300000, 9, 4, dt=st.F64) and rolls(300000, 9, 3, dt=st.F64)
    assert not rolls(1024, 1024, 2, 7, op=0) and not rolls(1024, 1024, 2, 3) and rolls(1024, 1024, 2, 16)
    assert rolls(1031, 1021, 2, 4) and rolls(2048, 2048, 2, 3) and not rolls(64, 60000, 2, 7, op=0) and rolls(1024, 1024, 3, 3)
    assert not rolls(1024, 1024, 2, 3, dt=st.F64) and rolls(1024, 1024, 2, 4, dt=st.F64) and rolls(64, 60000, 2, 3, dt=st.F64)
    """)


def test_workspace_growth_and_capture(host):
    """Growing the workspace neither ends a capture on another stream nor takes
    a block away from a captured graph; a block that cannot be freed is kept."""
    host("""
    mode, capturing, freed, blocks = [0], set(), [], []
    answer["mode"] = lambda h, n, a: mode.__setitem__(0, n) or 0
    answer["capturing"] = lambda h, n, a: int(h in capturing)
    def guarded(h, n, a): return 900 if capturing and mode[0] != 2 else 0    # stream capture would be ended
    def free(h, n, a):
        if not guarded(h, n, a): freed.append(h)
        return guarded(h, n, a)
    answer["malloc"], answer["free"] = guarded, free
    answer["sync"] = lambda h, n, a: 900 if h in capturing else 0
    answer["k_pc_transpose"] = lambda h, n, a: blocks.append(C.cast(a[1], C.POINTER(C.c_void_p))[0]) or 0
    def call(stream, pos):  # 128 + 64 channel-major words of 2 bytes a position in the workspace
        log.clear(); blocks.clear()
        nn.conv3_wgrad(A, A, A, (1, 1, 1, pos), 64, 64, stream=stream)
        assert kernels()[-1] == "k_conv3_wgrad_t"
        return blocks[0]
    S, T = 0x5000, 0x6000
    a = call(S, 1 << 18)
    capturing.add(T)
    b = call(S, 1 << 19)                       # grows while T is under capture
    assert freed == [a] and b != a
    c = call(T, 1 << 18)                       # first use, under capture
    d = call(T, 1 << 19)                       # grows under capture: nothing waited for, nothing freed
    assert freed == [a] and d != c
    capturing.clear()
    call(T, 1 << 22)                           # grows outside: c and d belong to the captured graph
    assert freed == [a]
    answer["free"] = 1
    try: call(S, 1 << 22); raise SystemExit("growth without its free")
    except st.StencilError: pass
    answer["free"] = free
    e = call(S, 1 << 22)
    assert freed == [a, b] and e not in (a, b)
    """)


def test_threads_on_one_stream(host):
    """Each call's launches on a stream come in one piece, also the first ones,
    which allocate: what they leave in the stream's workspace is theirs."""
    host("""
    def pause(h, n, a): time.sleep(0.0005); return 0
    for k in ("k_flag_one", "k_grid_shell_eq", "k_tile", "k_resident_clear", "k_resident", "k_conv3_wgrad_tile", "k_wgrad_reduce",
              "capturing", "malloc", "mode"): answer[k] = pause
    def calls(stream):
        for _ in range(3):
            st.dispatch_kernels(auto(96, 96, 96, iterations=24), A, B, stream=stream)
            st.dispatch_kernels(auto(200, 200, 100, radius=2, iterations=4), A, B, stream=stream)
            nn.conv3_wgrad(A, A, A, (8, 16, 16, 16), 16, 16, stream=stream)
    want = [["k_resident"], ["k_flag_one", "k_grid_shell_eq"] + ["k_tile"] * 4, ["k_conv3_wgrad_tile", "k_wgrad_reduce"]] * 3
    for stream in (0x5000, 0x6000):
        log.clear()
        ts = [threading.Thread(target=calls, args=(stream,)) for _ in range(4)]
        [t.start() for t in ts]; [t.join() for t in ts]
        got = [(e[0], e[3]) for e in log if e[0].startswith("k_") and e[0] != "k_resident_clear"]
        first = [e[0] for e in log if e[0].startswith("k_resident")]
        assert first[0] == "k_resident_clear" and first.count("k_resident_clear") == 1, first
        runs = []  # launches of one thread in a row
        for name, t in got:
            if runs and runs[-1][1] == t: runs[-1][0].append(name)
            else: runs.append(([name], t))
        flat = {}
        for names, t in runs:
            seq = flat.setdefault(t, [])
            seq += names
            done = [n for w in want for n in w][:len(seq)]
            ends = [sum(map(len, want[:i])) for i in range(len(want) + 1)]
            assert seq == done and len(seq) in ends, (names, seq)
    """)


def test_per_thread_stream(host):
    """hipStreamPerThread is another stream on each thread, with a workspace
    of its own."""
    host("""
    blocks = set()
    answer["k_flag_one"] = lambda h, n, a: blocks.add((threading.get_ident(), C.cast(a[0], C.POINTER(C.c_void_p))[0])) or 0
    barrier = threading.Barrier(3)
    def call():
        barrier.wait()
        for _ in range(3): st.dispatch_kernels(auto(200, 200, 100, radius=2, iterations=4), A, B, stream=2)
        barrier.wait()
    ts = [threading.Thread(target=call) for _ in range(3)]
    [t.start() for t in ts]; [t.join() for t in ts]
    assert len(blocks) == 3 and len({b for _, b in blocks}) == 3, blocks
    """)


def test_no_room_for_workspace(host):
    """Calls that ran without a workspace before they were given a faster form
    still run where there is no room for one."""
    host("""
    answer["malloc"] = 2  # hipErrorOutOfMemory
    def route(call):
        log.clear(); call()
        return kernels()
    run = lambda *a, **kw: st.dispatch_kernels(auto(*a, **kw), A, B)
    assert route(lambda: run(64, 64, 64, iterations=24))[0].startswith("k_base")
    assert route(lambda: run(128, 128, 128, iterations=24)) == ["k_tile"] * 24
    assert route(lambda: run(333, 251, 207, radius=2)) == ["k_tile"] * 4
    assert route(lambda: nn.conv3_wgrad(A, A, A, (2, 33, 33, 33), 16, 16)) == ["k_conv3_wgrad"]
    problems = [dict(nx=64, ny=40, nz=33, radius=1, iterations=24, op=1, u1=A, u2=B)] * 4
    try: st.dispatch_batched(problems, (), st.BATCH_PERSISTENT, stream=0x5000)
    except st.StencilError as e: assert e.status == 4  # its own table needs memory, as before
    """)


def test_resident_poll_that_gives_up(host):
    """A launch whose workgroups waited in vain for each other is an error of
    the call that waits for it, or of the next one on its stream."""
    host("""
    def in_vain(h, n, args):  # what the kernel does: sets the word at the head of its arguments
        word = C.cast(args[0], C.POINTER(C.POINTER(C.c_uint)))[0]
        assert word[0] == 0
        word[0] = 1
        return 0
    p = auto(64, 64, 64, iterations=24)
    call = lambda stream, timed=False: st.dispatch_kernels(p, A, B, stream=stream, timed=timed)
    def fails(f):
        try: f()
        except st.StencilError as e: return e.status == 3
        return False
    call(0x5000); call(0x6000)
    answer["k_resident"] = in_vain
    assert fails(lambda: call(0x5000, True))
    call(0x5000)
    answer["k_resident"] = 0
    log.clear()
    call(0x6000)                                     # another stream: not its failure
    assert kernels() == ["k_resident"]
    assert fails(lambda: call(0x5000)) and kernels() == ["k_resident"]
    call(0x5000)                                     # reported once
    answer["k_resident"] = in_vain
    problems = [dict(nx=64, ny=40, nz=33, radius=1, iterations=24, op=1, u1=A, u2=B)] * 4
    assert fails(lambda: st.dispatch_batched(problems, (), st.BATCH_PERSISTENT, stream=0x5000, timed=True))
    """)
