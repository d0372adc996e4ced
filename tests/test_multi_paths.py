"""Calls whose steps go several per launch, in the forms that choose between
that and one step per launch, against single steps: the populations are equal
bit for bit."""
import numpy as np
import pytest

WALL = ("wall", None, 1.0)


def start(shape, seed):
    rng = np.random.default_rng(seed)
    n = int(np.prod(shape))
    return 1 + 1e-3 * rng.standard_normal(n), 0.02 + 2e-3 * rng.standard_normal((n, len(shape)))


@pytest.mark.gpu
@pytest.mark.parametrize("storage", ["f32", "f64"])
def test_batch_goes_on_after_domains_retire(storage):
    """Half of the domains are at rest and retire at the first check; the
    others go on with tiles and steps per launch of the shorter list."""
    from lbm_amd import capi

    shape, box = (160, 128), {"-x": WALL, "+x": WALL, "-y": WALL, "+y": WALL}
    fields = [start(shape, k) if k % 2 else (np.ones(160 * 128), np.zeros((160 * 128, 2))) for k in range(8)]
    b = capi.Batch([{"shape": shape, "omega": 1.0 + 0.05 * k, "faces": box} for k in range(8)], storage=storage)
    b.init(np.concatenate([f[0] for f in fields]), np.concatenate([f[1] for f in fields]))
    steps = b.run(26, 1e-300, 78)[0]
    assert [int(s) for s in steps] == [-1 if k % 2 else 26 for k in range(8)]
    for k in range(8):
        lat = capi.Lattice(shape, storage=storage, omega=1.0 + 0.05 * k, faces=box)
        lat.init(*fields[k])
        for _ in range(78 if k % 2 else 26):
            lat.step(1)
        assert np.array_equal(b.populations(k), lat.populations()), k
        lat.close()
    b.close()


@pytest.mark.gpu
@pytest.mark.parametrize("storage", ["f32", "f64", "f16"])
@pytest.mark.parametrize("faces", ["periodic", "walls", "neem"])
def test_low_domains_equal_single_steps(storage, faces):
    """Few rows: wide tiles, two to eight steps per launch, or one."""
    from lbm_amd import capi

    walls = {"-y": WALL, "+y": ("wall", (0.02, 0.0), 1.0)}
    kinds = {"periodic": {}, "walls": walls,
             "neem": dict(walls, **{"-x": ("velocity_neem", (0.03, 0.0), 1.0), "+x": ("pressure_neem", None, 1.0)})}
    for nx, ny in ((701, 3), (40000, 3), (300000, 3), (30011, 5), (250007, 6), (33, 12), (20001, 17), (60000, 31), (30003, 45), (9001, 62)):
        solid = (np.random.default_rng(ny).random(nx * ny) < 0.05).astype(np.uint8) if ny > 5 else None
        out = []
        for calls in ((17, 2, 5), (1,) * 24):
            lat = capi.Lattice((nx, ny), storage=storage, omega=1.2, faces=kinds[faces], solid=solid)
            lat.init(*start((nx, ny), ny))
            for n in calls:
                lat.step(n)
            out.append(lat.populations())
            lat.close()
        assert np.isfinite(out[0]).all() and np.array_equal(*out), (nx, ny)


@pytest.mark.gpu
@pytest.mark.parametrize("storage", ["f32", "f64", "f16"])
@pytest.mark.parametrize("periodic", [False, True])
def test_batch_of_low_domains_equals_domains_alone(storage, periodic):
    """Wide tiles in domains of few rows, beside one of many rows."""
    from lbm_amd import capi

    faces = {} if periodic else {"-x": ("velocity_zh", (0.03, 0.0), 1.0), "+x": ("pressure_abb", None, 1.0), "-y": WALL, "+y": WALL}
    rng = np.random.default_rng(1)
    shapes = [(int(rng.integers(500, 1500)), int(rng.integers(3, 9))) for _ in range(30)] + [(300, 200), (3, 3)]
    fields = [start(s, k) for k, s in enumerate(shapes)]
    b = capi.Batch([{"shape": s, "omega": 1.1, "faces": faces} for s in shapes], storage=storage)
    b.init(np.concatenate([f[0] for f in fields]), np.concatenate([f[1] for f in fields]))
    b.run(20, 0.0, 40)
    for k in (0, 1, 5, 17, 29, 30, 31):
        lat = capi.Lattice(shapes[k], storage=storage, omega=1.1, faces=faces)
        lat.init(*fields[k])
        for _ in range(40):
            lat.step(1)
        assert np.array_equal(b.populations(k), lat.populations()), shapes[k]
        lat.close()
    b.close()


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["dirichlet", "neumann"])
@pytest.mark.parametrize("Q,nx,ny", [(5, 100003, 5), (9, 66661, 6), (5, 60011, 8), (9, 50001, 13), (5, 900001, 5), (9, 31, 5)])
def test_low_poisson_windows_equal_single_steps(Q, nx, ny, kind):
    from lbm_amd import poisson

    rng = np.random.default_rng(ny)
    faces = {f: (kind if f[1] == "y" else "dirichlet", rng.random(ny if f[1] == "x" else nx), k)
             for k, f in enumerate(("-x", "+x", "-y", "+y"))}
    phi0, out = rng.random(nx * ny), []
    for calls in ((13, 2, 9), (1,) * 24):
        p = poisson.Poisson(Q, nx, ny, 1.3, -0.003)
        p.set_faces(faces)
        p.init(phi0)
        for n in calls:
            p.step(n)
        out.append((p.phi(), p.step_check()[0]))
        p.close()
    assert np.isfinite(out[0][0]).all() and np.array_equal(out[0][0], out[1][0]) and out[0][1] == out[1][1]
