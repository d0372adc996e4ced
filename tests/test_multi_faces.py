"""Faces and solids of the launches that take several steps, each case checked
to be one: open x faces of every kind with walls or periodic y faces beside
them, corners where priorities decide, solids in the face columns and next to
them (a NEEM cell whose inward neighbour is solid keeps its bounce-back
values).  Against single steps, equal bit for bit."""
import numpy as np
import pytest

WALL = ("wall", None, 1.0)
Y_WALLS = {"-y": WALL, "+y": WALL}
Y_MOVING = {"-y": ("wall", (0.02, 0.0), 1.0, 3), "+y": ("wall", (-0.01, 0.0), 1.0, 0)}


def x_faces(low, high, prio=1):
    value = {"velocity": (0.03, 0.0), "pressure": None}
    spec = [(k, value[k.split("_")[0]], 1.002 if s else 0.999, prio) for s, k in enumerate((low, high))]
    return {"-x": spec[0], "+x": spec[1]}


FACES2 = {
    "zh_zh": {**x_faces("velocity_zh", "pressure_zh"), **Y_WALLS},
    "zh_zh_periodic": x_faces("pressure_zh", "velocity_zh"),
    "abb_abb_periodic": x_faces("pressure_abb", "pressure_abb"),
    "abb_zh_moving": {**x_faces("pressure_abb", "velocity_zh", 2), **Y_MOVING},
    "neem_neem_periodic": x_faces("pressure_neem", "velocity_neem"),
    "neem_moving": {**x_faces("velocity_neem", "pressure_neem", 1), **Y_MOVING},
    "neem_wall": {"-x": ("velocity_neem", (0.03, 0.0), 1.0), "+x": ("wall", (0.0, 0.02), 1.0), **Y_WALLS},
    "wall_neem": {"-x": WALL, "+x": ("pressure_neem", None, 1.001), **Y_WALLS},
    "corners": {"-x": ("wall", (0.0, 0.03), 1.0, 2), "+x": ("wall", (0.0, -0.02), 1.0, 0), "-y": ("wall", (0.02, 0.0), 1.0, 1),
                "+y": ("wall", (0.04, 0.0), 1.0, 2)},
}
SINGLE2 = {  # faces that the kernel has no rule for
    "neem_y": {"-y": ("pressure_neem", None, 1.0), "+y": ("velocity_neem", (0.0, -0.02), 1.0)},
    "abb_y": {"-y": ("pressure_abb", None, 1.0), "+y": ("pressure_abb", None, 0.999)},
    "wet_eq": {"-y": ("wall_eq", None, 1.0), "+y": ("wall_eq", (0.02, 0.0), 1.0)},
    "periodic_pressure": {"-x": ("periodic_pressure", None, 1.001), "+x": ("periodic_pressure", None, 1.0), **Y_WALLS},
}


def scattered(shape, seed):
    """A tenth of the cells, in the face columns and rows too; a solid column
    next to each x face on some rows."""
    rng = np.random.default_rng(seed)
    s = rng.random(shape[::-1]) < 0.1
    s[..., ::5, 1] = True
    s[..., 2::7, -2] = True
    s[..., 3::5, 0] = True
    s[..., 1::4, -1] = True
    return s.reshape(-1).astype(np.uint8)


def both(shape, storage, faces, calls, solid=None, launch=True):
    from lbm_amd import capi

    rng = np.random.default_rng(3)
    n, dim = int(np.prod(shape)), len(shape)
    rho, u = 1 + 1e-3 * rng.standard_normal(n), 0.01 + 2e-3 * rng.standard_normal((n, dim))
    out = []
    for many in (True, False):
        lat = capi.Lattice(shape, storage=storage, omega=1.1, faces=faces, solid=solid)
        assert (lat.steps_per_launch(max(calls)) > 1) == launch
        lat.init(rho, u)
        for k in calls if many else (1,) * sum(calls):
            lat.step(k)
        out.append(lat.populations())
        lat.close()
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("storage", ["f32", "f64", "bf16"])
@pytest.mark.parametrize("faces", list(FACES2))
def test_d2q9_faces_and_solids(storage, faces):
    for shape in ((3, 3), (5, 40), (33, 18), (131, 70), (640, 410)):
        for solid in (None, scattered(shape, 5)):
            a, b = both(shape, storage, FACES2[faces], (2, 9, 13), solid)
            assert np.array_equal(a, b, equal_nan=True), shape
            assert solid is not None or np.isfinite(a).all()


@pytest.mark.parametrize("storage", ["f32", "f64"])
@pytest.mark.parametrize("faces", list(SINGLE2))
@pytest.mark.gpu
def test_d2q9_faces_without_a_rule_run_one_step_per_launch(storage, faces):
    a, b = both((131, 70), storage, SINGLE2[faces], (2, 9), launch=False)
    assert np.isfinite(a).all() and np.array_equal(a, b)


Z_WALLS = {"-y": WALL, "+y": ("wall", (0.02, 0.0, 0.01), 1.0, 3), "-z": WALL, "+z": ("wall", (0.0, 0.01, 0.0), 1.0, 1)}
FACES3 = {
    "neem": {"-x": ("velocity_neem", (0.03, 0.0, 0.0), 1.0), "+x": ("pressure_neem", None, 1.0), **Z_WALLS},
    "neem_wall": {"-x": ("pressure_neem", None, 1.001), "+x": ("wall", (0.0, 0.01, 0.02), 1.0, 2), **Z_WALLS},
    "neem_periodic": {"-x": ("pressure_neem", None, 1.001), "+x": ("velocity_neem", (0.03, 0.0, 0.0), 1.0)},
    "walls": {"-x": ("wall", (0.0, 0.01, 0.02), 1.0, 1), "+x": WALL, **Z_WALLS},
}


@pytest.mark.gpu
@pytest.mark.parametrize("faces", list(FACES3))
@pytest.mark.parametrize("shape", [(67, 66, 64), (3, 300, 221), (4, 5, 10001), (10001, 7, 3), (700, 3, 96), (41, 240, 20)])
def test_d3q19_faces_and_solids(faces, shape):
    for solid in (None, scattered(shape, 7)):
        a, b = both(shape, "f64", FACES3[faces], (2, 5), solid)
        assert np.array_equal(a, b, equal_nan=True)
        assert solid is not None or np.isfinite(a).all()


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(150, 101, 99), (3, 800, 380), (40, 800, 30), (300, 52, 60)])
def test_d3q19_fp32_walls_and_solids(shape):
    solid = scattered(shape, 9)
    a, b = both(shape, "f32", {"-z": WALL, "+z": ("wall", (0.02, 0.01, 0.0), 1.0)}, (2, 3), solid)
    assert np.isfinite(a).all() and np.array_equal(a, b)


LID3 = {"-x": WALL, "+x": ("wall", (0.0, 0.0, 0.02), 1.0), **Z_WALLS}


@pytest.mark.gpu
@pytest.mark.parametrize("storage,shape,faces,force", [
    ("f32", (5, 5, 31500), {}, (0.0, 0.0, 0.0)), ("f32", (33, 31, 770), {}, (1e-5, 0.0, 0.0)),
    ("f32", (100, 98, 81), {}, (0.0, 0.0, 0.0)), ("f32", (4, 1020, 200), {}, (1e-5, 2e-6, 0.0)),
    ("f32", (4, 1020, 200), Z_WALLS, (1e-5, 0.0, 0.0)), ("f32", (5, 5, 31500), LID3, (0.0, 0.0, 0.0)),
    ("f32", (150, 143, 149), LID3, (0.0, 0.0, 0.0)), ("f32", (8800, 30, 3), {**Y_WALLS, "-z": WALL, "+z": WALL}, (0.0, 0.0, 0.0)),
    ("f16", (150, 143, 149), {}, (1e-5, 0.0, 0.0)), ("bf16", (3, 1300, 810), {}, (0.0, 0.0, 0.0))])
def test_d3q19_smaller_storage_forms(storage, shape, faces, force):
    from lbm_amd import capi

    n, rng, out = int(np.prod(shape)), np.random.default_rng(4), []
    rho, u = 1 + 1e-3 * rng.standard_normal(n), 0.01 + 2e-3 * rng.standard_normal((n, 3))
    for calls in ((4, 3), (1,) * 7):
        lat = capi.Lattice(shape, storage=storage, omega=1.1, faces=faces, force=force)
        assert lat.steps_per_launch(2) == 2
        lat.init(rho, u)
        for k in calls:
            lat.step(k)
        out.append(lat.populations())
        lat.close()
    assert np.isfinite(out[0]).all() and np.array_equal(*out)
