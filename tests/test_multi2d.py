"""Several D2Q9 steps per launch (k_multi2d) against as many single steps:
the same cell update on a tile in LDS, so the populations are equal bit for
bit.  Sizes around the tile edges, domains smaller than a tile and its halo,
every face kind next to every tile edge, solids, all storage forms."""
import numpy as np
import pytest

FACES = {
    "periodic": {},
    "walls": {"-y": ("wall", None, 1.0), "+y": ("wall", (0.03, 0.0), 1.0)},
    "lid": {"-x": ("wall", None, 1.0), "+x": ("wall", None, 1.0), "-y": ("wall", None, 1.0), "+y": ("wall", (0.04, 0.0), 1.0)},
    "neem_x": {"-y": ("wall", None, 1.0), "+y": ("wall", None, 1.0), "-x": ("velocity_neem", (0.04, 0.0), 1.0),
               "+x": ("pressure_neem", None, 1.0)},
    "neem_y": {"-y": ("pressure_neem", None, 1.0), "+y": ("velocity_neem", (0.0, -0.02), 1.0)},
    "zh_abb": {"-y": ("wall", None, 1.0), "+y": ("wall", None, 1.0), "-x": ("velocity_zh", (0.03, 0.0), 1.0),
               "+x": ("pressure_abb", None, 1.0)},
    "abb_y": {"-y": ("pressure_abb", None, 1.0), "+y": ("pressure_abb", None, 0.999)},
    "wet_eq": {"-y": ("wall_eq", None, 1.0), "+y": ("wall_eq", (0.02, 0.0), 1.0)},
    "wet_neem": {"-y": ("wall_neem", None, 1.0), "+y": ("wall_neem", (0.02, 0.0), 1.0), "-x": ("pressure_abb", None, 1.0),
                 "+x": ("pressure_abb", None, 0.999)},
    "wet_nebb": {"-y": ("wall_nebb0", None, 1.0), "+y": ("wall_nebb", (0.02, 0.0), 1.0)},
}


def start(shape, seed):
    rng = np.random.default_rng(seed)
    n = shape[0] * shape[1]
    return 1 + 1e-3 * rng.standard_normal(n), 0.02 + 2e-3 * rng.standard_normal((n, 2))


def solids(shape, seed):
    """Blobs away from the open faces, one against a wall, one spanning rows."""
    nx, ny = shape
    s = np.zeros((ny, nx), np.uint8)
    if nx >= 16 and ny >= 12:
        s[ny // 3:ny // 3 + 3, nx // 3:nx // 3 + 4] = 1
        s[:2, nx // 2:nx // 2 + 3] = 1
        rng = np.random.default_rng(seed)
        for _ in range(nx * ny // 200):
            s[rng.integers(3, ny - 3), rng.integers(5, nx - 5)] = 1
    return s.reshape(-1)


def both(shape, storage, faces, steps, solid=None, omega=1.2, force=(0.0, 0.0, 0.0)):
    from lbm_amd import capi

    rho, u = start(shape, 3)
    out = []
    for many in (True, False):
        lat = capi.Lattice(shape, storage=storage, omega=omega, force=force, faces=faces, solid=solid)
        lat.init(rho, u)
        for n in steps:
            if many:
                lat.step(n)
            else:
                for _ in range(n):
                    lat.step(1)
        out.append(lat.populations())
        lat.close()
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("faces", list(FACES))
@pytest.mark.parametrize("shape", [(5, 5), (17, 9), (64, 16), (65, 33), (131, 70), (300, 7), (7, 300)])
def test_multi_equals_single_steps(faces, shape):
    for force in ((0.0, 0.0, 0.0), (1e-5, 0.0, 0.0), (1e-5, -2e-5, 0.0)) if faces in ("walls", "periodic") else ((0.0, 0.0, 0.0),):
        a, b = both(shape, "f32", FACES[faces], (2, 9, 16, 5), force=force)
        assert np.isfinite(a).all() and np.array_equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("storage", ["f64", "f16"])
@pytest.mark.parametrize("force", [(1e-5, 0.0, 0.0), (0.0, 2e-5, 0.0)])
def test_multi_with_a_force(storage, force):
    a, b = both((150, 77), storage, FACES["walls"], (3, 8, 13), force=force)
    assert np.isfinite(a).all() and np.array_equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("storage", ["f32", "f64", "f16", "bf16"])
@pytest.mark.parametrize("faces", ["periodic", "lid", "neem_x", "zh_abb"])
def test_multi_with_solids_every_storage(storage, faces):
    for shape in ((150, 77), (500, 300), (640, 410)):
        a, b = both(shape, storage, FACES[faces], (3, 8, 13), solid=solids(shape, 5))
        assert np.isfinite(a).all() and np.array_equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("storage,shape", [("f32", (2101, 1803)), ("f64", (1501, 1302)), ("f16", (20, 380000))])
def test_multi_beyond_the_caches(storage, shape):
    a, b = both(shape, storage, FACES["neem_x"], (5, 4))
    assert np.isfinite(a).all() and np.array_equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("storage", ["f32", "f64", "f16"])
def test_multi_batch_equals_domains_alone(storage):
    """A batch's multi-step tiles (domains cut evenly, uneven sizes, some
    without solids) against every domain stepped one step per launch."""
    from lbm_amd import capi

    shapes = [(5, 6), (33, 20), (64, 32), (200, 61), (517, 130)]
    kinds = ["lid", "zh_abb", "periodic", "neem_x", "zh_abb"]
    doms, fields = [], []
    for k, (shape, f) in enumerate(zip(shapes, kinds)):
        solid = solids(shape, k) if k in (1, 3, 4) else None
        doms.append({"shape": shape, "omega": 1.0 + 0.1 * k, "faces": FACES[f], "solid": solid})
        fields.append(start(shape, k))
    b = capi.Batch(doms, storage=storage)
    b.init(np.concatenate([f[0] for f in fields]), np.concatenate([f[1] for f in fields]))
    for interval, cycles in ((2, 1), (4, 2), (26, 3)):
        b.run(interval, 0.0, interval * cycles)
    for k, d in enumerate(doms):
        lat = capi.Lattice(d["shape"], storage=storage, omega=d["omega"], faces=d["faces"], solid=d["solid"])
        lat.init(*fields[k])
        for _ in range(2 + 8 + 78):
            lat.step(1)
        assert np.array_equal(b.populations(k), lat.populations()), k
        lat.close()
    b.close()
