"""The host side of liblbm_hip.so on the CPU, over a stand-in for the HIP
runtime (hip_stand_in.c): which launches a call makes, and what is left of a
handle when an allocation or a launch fails.  Each test runs in a process of
its own, where the stand-in takes the runtime's place."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

SETUP = """
import ctypes as ct, sys
import numpy as np
si = ct.CDLL(sys.argv[1], mode=ct.RTLD_GLOBAL)
from lbm_amd import capi, poisson

def flag(name, kind=ct.c_int):
    return kind.in_dll(si, name)

class Multi2dArgs(ct.Structure):  # lbm_multi2d.h
    _fields_ = [("src", ct.c_void_p), ("dst", ct.c_void_p), ("steps", ct.c_int), ("ntiles", ct.c_int),
                ("plane", ct.c_longlong), ("nx", ct.c_int), ("ny", ct.c_int), ("px", ct.c_int), ("per", ct.c_int * 2),
                ("face", ct.c_void_p), ("links", ct.c_void_p), ("omega", ct.c_double), ("F", ct.c_double * 3),
                ("ntx", ct.c_int), ("tw", ct.c_int), ("th", ct.c_int), ("tiles", ct.c_void_p), ("doms", ct.c_void_p),
                ("active", ct.c_void_p)]

def launches(what, since=0):
    names = (ct.c_char * 64 * 4096).in_dll(si, "si_name")
    args = (ct.c_ubyte * 512 * 4096).in_dll(si, "si_args")
    n = flag("si_launches").value
    return [(names[k].value.decode(), bytes(args[k])) for k in range(since, min(n, 4096)) if what in names[k].value.decode()]

def count():
    return flag("si_launches").value

def fail_launch(name, after=0):
    (ct.c_char * 64).in_dll(si, "si_fail_launch").value = name.encode()
    flag("si_fail_after").value = after

def multi2d(since=0):
    return [Multi2dArgs.from_buffer_copy(a) for _, a in launches("k_multi2d", since)]
"""


@pytest.fixture(scope="session")
def stand_in(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("hip") / "hip_stand_in.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", out, os.path.join(HERE, "hip_stand_in.c")], check=True)
    return out


def run(stand_in, body):
    env = dict(os.environ, PYTHONPATH=ROOT)
    r = subprocess.run([sys.executable, "-c", SETUP + body, stand_in], env=env, cwd=ROOT, capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.parametrize("fails", range(4))  # each allocation of the rebuild
def test_failed_batch_rebuild_keeps_tiles_and_steps_together(stand_in, fails):
    """Domains retire, the shorter list of tiles gets another plan (more steps
    per launch on smaller tiles), and there is no memory for it: the next run
    goes on with the old tiles, on which the new number of steps does not fit
    the LDS."""
    run(stand_in, f"""
n = 8 * 160 * 128
b = capi.Batch([{{"shape": (160, 128), "omega": 1.2, "faces": {{}}}}] * 8, storage="f32")
b.init(np.ones(n), np.zeros((n, 2)))
def launches_of_a_run():
    since = count()
    b.run(50, 0.0, 50)
    return [(a.steps, a.ntiles, a.tiles) for a in multi2d(since)]
before = launches_of_a_run()
flag("si_retire").value = 4
flag("si_fail_malloc").value = {fails}
try:
    b.run(50, 0.0, 50)
    assert False
except capi.LBMError as e:
    assert e.code == capi.LBM_ENOMEM
flag("si_fail_malloc").value = -1
assert launches_of_a_run() == before
b.set_tiling(64, 0)  # succeeds
assert launches_of_a_run()[0][0] > before[0][0]
""")


@pytest.mark.parametrize("call", ["set_storage", "set_faces"])
def test_without_block_flags_steps_run_one_per_launch(stand_in, call):
    """The launch that marks the two-step kernel's blocks that meet a solid
    fails: the call succeeds, the marks of the old storage form's tiles (or
    none) are not used with the new tiles, and a later call makes them."""
    run(stand_in, f"""
wall = ("wall", None, 1.0)
faces = {{"-y": wall, "+y": wall, "-z": wall, "+z": wall}}
solid = np.zeros((64, 100, 128), np.uint8)
solid[20:30, 20:30, 20:30] = 1
lat = capi.Lattice((128, 100, 64), storage="f64", omega=1.2, faces=faces, solid=solid)
def kernels_of_two_steps():
    since = count()
    lat.step(2)
    return [n for n, _ in launches("", since)]
assert len(launches("k_multi3d_solid")) == 2 and ["k_multi3d" in n for n in kernels_of_two_steps()] == [True]
def change(k):
    if "{call}" == "set_storage":
        lat.set_storage("f32" if k else "f64")
    else:
        lat.set_faces(dict(faces, **{{"+z": ("wall", (0.01 * k, 0.0, 0.0), 1.0)}}))
fail_launch("k_multi3d_solid")
change(1)
assert ["k_multi3d" in n for n in kernels_of_two_steps()] == [False, False]
fail_launch("")
change(0)
assert ["k_multi3d" in n for n in kernels_of_two_steps()] == [True]
""")


def test_as_many_steps_as_the_argument_holds(stand_in):
    """2^31 - 1 steps are launched (until the stand-in lets a launch fail)."""
    run(stand_in, """
def fails_on_the_way(step, kernel):
    since = count()
    fail_launch(kernel, after=5)
    try:
        step(2 ** 31 - 1)
        assert False
    except RuntimeError:
        pass
    fail_launch("")
    assert len(launches(kernel, since)) == 5
lat = capi.Lattice((64, 32), omega=1.2)
fails_on_the_way(lat.step, "k_multi2d")
assert multi2d()[0].steps == 8
p = poisson.Poisson(5, 64, 32, 1.0, 0.0)
p.set_faces({f: ("neumann", None, k) for k, f in enumerate(("-x", "+x", "-y", "+y"))})
p.init(np.zeros(64 * 32))
fails_on_the_way(p.step, "k_poisson_multi")
""")


def test_a_failed_launch_leaves_the_state_current(stand_in):
    """The next launch reads the state that the failed one would have read."""
    run(stand_in, """
lat = capi.Lattice((64, 32), omega=1.2)
lat.step(8)
fail_launch("k_multi2d")
try:
    lat.step(8)
    assert False
except capi.LBMError as e:
    assert e.code == capi.LBM_EHIP
fail_launch("")
lat.step(8)
first, after = multi2d()
assert after.src == first.dst and after.dst == first.src
""")


TILES = """
def extent(b, e, back, n, periodic):
    if periodic:
        return b - back, e + back
    if back:
        b, e = min(b, n - 2), max(e, 1)
    return max(b - back, 0), min(e + back, n - 1)

def slots(x0, x1, y0, y1, nx, ny, T, perx, pery, open_faces):
    '''LDS slots per direction of a tile (k_multi2d): its region and what the
    in-place steps, each a line or two further down, need in front'''
    rx, ry = extent(x0, x1, T, nx, perx), extent(y0, y1, T, ny, pery)
    pitch, rows = rx[1] - rx[0] + 1, ry[1] - ry[0] + 1
    columns = not perx and (rx[0] == 0 and open_faces or rx[1] == nx - 1 and open_faces)
    sx, sy = (rows, 1) if columns else (1, pitch)
    pad = down = 0
    for s in range(1, T):
        ex, ey = extent(x0, x1, T - s, nx, perx), extent(y0, y1, T - s, ny, pery)
        down += ((2 if ex[1] == nx - 1 else 1) * rows if columns else pitch) + 2
        pad = max(pad, down - (ey[0] - ry[0]) * sy - (ex[0] - rx[0]) * sx)
    assert pitch * rows * max(pitch, rows) < 1 << 20  # the kernel's division by a line
    return pad + pitch * rows

def updates(a, pery):
    '''cells updated per cell kept and step'''
    return sum((a.tw + 2 * s) * (a.th + 2 * s if pery else min(a.th + 2 * s, a.ny)) for s in range(a.steps)) / \\
        (a.steps * a.tw * min(a.th, a.ny))
"""


@pytest.mark.parametrize("storage,esize", [("f32", 4), ("f64", 8), ("f16", 2)])
@pytest.mark.parametrize("faces", ["periodic", "walls", "neem"])
def test_low_domains(stand_in, storage, esize, faces):
    """Domains of few rows: every tile fits the LDS, rows of a periodic axis are
    not updated several times over, and where tiles of so few rows take longer
    than one step per launch there are none."""
    run(stand_in, TILES + f"""
wall = ("wall", None, 1.0)
kinds = {{"periodic": {{}}, "walls": {{"-y": wall, "+y": wall}},
         "neem": {{"-y": wall, "+y": wall, "-x": ("velocity_neem", (0.01, 0.0), 1.0), "+x": ("pressure_neem", None, 1.0)}}}}
box = "{faces}" == "periodic"
cap = (80 * 1024 - 256) // (9 * {esize} + (0 if box else 2)) // 16 * 16
for ny in list(range(3, 34)) + [48, 63]:
    for cells in (100, 3000, 30000, 400000, 1500000):
        nx = max(3, cells // ny)
        lat = capi.Lattice((nx, ny), storage="{storage}", omega=1.2, faces=kinds["{faces}"])
        since = count()
        lat.step(24)
        lat.close()
        plans = multi2d(since)
        assert plans or (ny < 64 and cells >= 30000), (nx, ny)
        if not plans:
            assert len(launches("k_step", since)) == 24
            continue
        a = plans[0]
        if cells >= 400000 and ny < 32:
            # (FP64: the step that it replaces moves twice the bytes)
            assert updates(a, box) < (3.0 if {esize} == 8 else 2.0), (nx, ny, a.tw, a.th, a.steps)
        edge = lambda n, w: sorted({{0, w, n // w // 2 * w, (n - 1) // w * w - w, (n - 1) // w * w}} & set(range(0, n, w)))
        for x0 in edge(nx, a.tw):
            for y0 in edge(ny, a.th):
                n = slots(x0, min(x0 + a.tw, nx) - 1, y0, min(y0 + a.th, ny) - 1, nx, ny, a.steps, "{faces}" != "neem", box,
                          "{faces}" == "neem")
                assert n <= cap, (nx, ny, a.tw, a.th, a.steps, x0, y0, n)
for shape, force in (((1 << 20, 3), (0.0, 0.0, 0.0)), ((20000, 50), (1e-6, 1e-6, 0.0))):
    lat = capi.Lattice(shape, storage="f16", omega=1.2, force=force)
    since = count()
    lat.step(24)
    assert len(launches("k_step", since)) == 24, shape
""")


@pytest.mark.parametrize("storage,esize", [("f32", 4), ("f64", 8), ("f16", 2)])
@pytest.mark.parametrize("periodic", [False, True])
def test_low_domains_in_a_batch(stand_in, storage, esize, periodic):
    """Domains of few rows beside one of many: their tiles are as large as the
    others (not as wide), every tile fits the LDS, and all cells are covered."""
    run(stand_in, TILES + f"""
class MultiTile(ct.Structure):
    _fields_ = [(n, ct.c_int) for n in ("d", "x0", "y0", "w", "h")]
wall = ("wall", None, 1.0)
faces = {{}} if {periodic} else {{"-x": ("velocity_zh", (0.01, 0.0), 1.0), "+x": ("pressure_abb", None, 1.0), "-y": wall, "+y": wall}}
rng = np.random.default_rng(0)
shapes = [(int(rng.integers(500, 1500)), int(rng.integers(3, 9))) for _ in range(200)] + [(300, 200), (3, 3), (40, 500)]
b = capi.Batch([{{"shape": s, "omega": 1.2, "faces": faces}} for s in shapes], storage="{storage}")
b.run(50, 0.0, 50)
a = multi2d()[0]
cap = (80 * 1024 - 256) // (9 * {esize} + 2) // 16 * 16
assert a.steps <= 3 or not {periodic}
tiles = (MultiTile * a.ntiles).from_address(a.tiles)
seen = [np.zeros(s[::-1], int) for s in shapes]
most = max(t.w * t.h for t in tiles)
for t in tiles:
    nx, ny = shapes[t.d]
    seen[t.d][t.y0:t.y0 + t.h, t.x0:t.x0 + t.w] += 1
    assert slots(t.x0, t.x0 + t.w - 1, t.y0, t.y0 + t.h - 1, nx, ny, a.steps, {periodic}, {periodic}, not {periodic}) <= cap
    if ny < 9 and nx > 500 and t.x0 + t.w < nx:  # twice as wide: larger than the largest, the LDS or the kernel's division allow
        w = 2 << (t.w - 1).bit_length()  # (the domain is cut evenly into widths of up to a power of two)
        n = (w + 2 * a.steps) * (ny + 2 * a.steps) + 4 * a.steps
        assert w * ny > most or n > cap or n * (w + 2 * a.steps) >= 1 << 20, (nx, ny, t.w)
assert all((s == 1).all() for s in seen)
""")


@pytest.mark.parametrize("q", [5, 9])
def test_low_poisson_windows(stand_in, q):
    """Windows of few rows: every tile's region fits the LDS and its lines the
    first-layer arrays, and where there are cells enough a tile holds at least
    half as many as that of a square window."""
    run(stand_in, f"""
class PMulti(ct.Structure):  # lbm_poisson.hip
    _fields_ = [(n, ct.c_int) for n in ("steps", "tw", "th", "ntx", "ntiles")] + [("phi_prev", ct.c_void_p), ("write_phi", ct.c_int)]
args = (ct.c_ubyte * 64 * 4096).in_dll(si, "si_args2")
def extent(b, e, back, n):
    return max(min(b, n - 3) - back, 0), min(max(e, 2) + back, n - 1)
def plan(nx, ny):
    p = poisson.Poisson({q}, nx, ny, 1.0, 0.0)
    p.set_faces({{f: ("neumann", None, k) for k, f in enumerate(("-x", "+x", "-y", "+y"))}})
    p.init(np.zeros(nx * ny))
    since = count()
    p.step(48)
    p.close()
    return PMulti.from_buffer_copy(bytes(args[since])[:40])
for cells in (400, 20000, 100000, 400000, 2000000):
    side = int(cells ** 0.5)
    square = plan(side, side)
    for ny in list(range(5, 27)) + [40]:
        nx = max(5, cells // ny)
        m = plan(nx, ny)
        assert m.ntx == -(-nx // m.tw) and m.ntiles == m.ntx * -(-ny // m.th)
        for x0 in {{0, m.tw if m.tw < nx else 0, (nx - 1) // m.tw * m.tw}}:
            for y0 in range(0, ny, m.th):
                x = extent(x0, min(x0 + m.tw, nx) - 1, m.steps, nx)
                y = extent(y0, min(y0 + m.th, ny) - 1, m.steps, ny)
                pitch, rows = x[1] - x[0] + 1, y[1] - y[0] + 1
                assert pitch * rows <= 1024 and pitch <= 128 and rows <= 128, (nx, ny, m.tw, m.th, m.steps)
        if cells >= 100000:
            assert 2 * m.tw * m.th > square.tw * square.th or m.th < ny or 2 * (m.tw + m.steps) > 128, (nx, ny, m.tw, m.th)
""")


# domains whose two steps in one pass were timed above or below two launches
TWO_STEP_ROUTES = """
wall = ("wall", None, 1.0)
moving = ("wall", (0.01, 0.02, 0.01), 1.0)
channel = {"-y": wall, "+y": wall, "-z": wall, "+z": wall}
box = dict(channel, **{"-x": wall, "+x": wall})
def two_steps(shape, storage, faces, force=(0.0, 0.0, 0.0), solids=0.0):
    solid = (np.random.default_rng(0).random(np.prod(shape)) < solids).astype(np.uint8) if solids else None
    lat = capi.Lattice(shape, storage=storage, omega=1.2, faces=faces, force=force, solid=solid)
    since = count()
    lat.step(2)
    lat.close()
    names = [n for n, _ in launches("", since)]
    assert len(names) in (1, 2) and ("k_multi3d" in names[0]) == (len(names) == 1), names
    return len(names) == 1
x, xy = (1e-6, 0.0, 0.0), (1e-6, 1e-6, 0.0)
"""


def test_two_steps_only_where_they_are_faster(stand_in):
    run(stand_in, TWO_STEP_ROUTES + """
for shape, storage, faces, force, solids, two in (
        ((160, 96, 96), "f32", channel, x, 0.0, True), ((100, 100, 100), "f32", channel, x, 0.0, False),
        ((130, 101, 99), "f32", box, xy, 0.0, True), ((128, 96, 96), "f32", channel, xy, 0.0, False),
        ((128, 96, 96), "f32", dict(box, **{"+y": moving}), (0.0,) * 3, 0.0, True),
        ((128, 96, 96), "f32", dict(box, **{"+x": moving, "+y": moving, "+z": moving}), (0.0,) * 3, 0.0, False),
        ((100, 100, 100), "f32", channel, x, 0.2, True),
        ((128, 128, 128), "f32", {}, xy, 0.0, True), ((128, 64, 66), "f32", {}, (0.0,) * 3, 0.0, False),
        ((512, 3, 400), "f32", {}, (0.0,) * 3, 0.0, False), ((512, 3, 400), "f64", {}, (0.0,) * 3, 0.0, True),
        ((256, 128, 100), "f16", {}, (0.0,) * 3, 0.0, True), ((256, 128, 100), "f16", {}, xy, 0.0, False),
        ((512, 6, 1100), "f16", {}, (0.0,) * 3, 0.0, False), ((512, 5, 400), "f64", channel, (0.0,) * 3, 0.0, False),
        ((97, 61, 45), "f64", box, (0.0,) * 3, 0.0, True)):
    assert two_steps(shape, storage, faces, force, solids) == two, (shape, storage, faces, force, solids)
""")


def test_least_cells_of_two_steps_in_fp64(stand_in):
    run(stand_in, TWO_STEP_ROUTES + """
for shape, two in (((64, 64, 48), False), ((64, 64, 49), True), ((700, 20, 18), True), ((128, 38, 36), False)):
    for faces in (channel, box):
        assert two_steps(shape, "f64", faces) == two, shape
""")


def test_steps_per_launch(stand_in):
    """lbm_steps_per_launch against the launches that lbm_step makes."""
    run(stand_in, """
wall = ("wall", None, 1.0)
for shape, storage, faces in (((64, 32), "f64", {}), ((333333, 3), "f16", {}), ((400, 300), "f32", {"-y": wall, "+y": wall}),
                              ((64, 32), "f32", {"-y": ("wall_eq", None, 1.0), "+y": ("wall_eq", None, 1.0)}),
                              ((128, 128, 64), "f32", {}), ((40, 40, 40), "f32", {})):
    lat = capi.Lattice(shape, storage=storage, omega=1.2, faces=faces)
    for n in (1, 2, 3, 9, 24, 25):
        since = count()
        lat.step(n)
        multi = multi2d(since)
        most = max(a.steps for a in multi) if multi else 2 if launches("k_multi3d", since) else 1
        assert lat.steps_per_launch(n) == most, (shape, storage, n, most)
    lat.close()
""")


def test_large_readback_with_another_device_current(stand_in):
    """A handle's read-backs go on its own device, whichever the caller has
    current (a read-back of 18 MB goes through events)."""
    run(stand_in, """
si.hipSetDevice(1)
lat = capi.Lattice((1000, 750), storage="f64", omega=1.2)
b = capi.Batch([{"shape": (1000, 750), "omega": 1.2}], storage="f64")
p = poisson.Poisson(5, 1600, 1400, 1.0, 0.0)
p.set_faces({f: ("neumann", None, k) for k, f in enumerate(("-x", "+x", "-y", "+y"))})
p.init(np.zeros(1600 * 1400))
si.hipSetDevice(0)
lat.macros()
lat.populations()
b.macros(0)
p.phi()
current = ct.c_int()
si.hipGetDevice(ct.byref(current))
assert current.value == 0
""")
