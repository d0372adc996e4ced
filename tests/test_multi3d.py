"""Two D3Q19 steps per launch (k_multi3d) against as many single steps: the
same arithmetic, so the populations are equal bit for bit.  Sizes around the
tile edges (regions of 512 or 256 columns), axes smaller than a tile and its
halo, few planes per slab, every face kind the kernel has rules for, solids
on and off faces, all storage forms, odd step counts; the domains are just
above the least number of cells the kernel is used for (multi3d_class)."""
import numpy as np
import pytest

WALL = ("wall", None, 1.0)
FACES = {
    "periodic": {},
    "channel": {"-y": WALL, "+y": WALL, "-z": WALL, "+z": WALL},
    "z_walls": {"-z": WALL, "+z": ("wall", (0.0, 0.02, 0.0), 1.0)},
    "lid": {"-x": WALL, "+x": ("wall", (0.0, 0.0, 0.02), 1.0), "-y": WALL, "+y": ("wall", (0.04, 0.0, 0.01), 1.0, 3),
            "-z": WALL, "+z": ("wall", (0.01, 0.02, 0.0), 1.0, 1)},
    "neem": {"-y": WALL, "+y": ("wall", (0.02, 0.0, 0.0), 1.0), "-z": WALL, "+z": WALL,
             "-x": ("velocity_neem", (0.04, 0.0, 0.0), 1.0), "+x": ("pressure_neem", None, 1.0)},
    "neem_periodic": {"-x": ("pressure_neem", None, 1.001), "+x": ("velocity_neem", (0.03, 0.0, 0.0), 1.0)},
}


def solids(shape, faces):
    nx, ny, nz = shape
    rng = np.random.default_rng(7)
    s = rng.random((nz, ny, nx)) < 0.03
    if "neem" in faces:  # some solids next to the open faces, none across a whole section
        s[:, :, 0] = False
        s[:, :, -1] = False
    return s.reshape(-1).astype(np.uint8)


def both(shape, storage, faces, steps, solid=None, force=(0.0, 0.0, 0.0)):
    from lbm_amd import capi

    rng = np.random.default_rng(3)
    n = shape[0] * shape[1] * shape[2]
    rho, u = 1 + 1e-3 * rng.standard_normal(n), 0.02 + 2e-3 * rng.standard_normal((n, 3))
    out = []
    for many in (True, False):
        lat = capi.Lattice(shape, storage=storage, omega=1.3, force=force, faces=faces, solid=solid)
        lat.init(rho, u)
        for k in steps:
            for _ in range(1 if many else k):
                lat.step(k if many else 1)
        out.append(lat.populations())
        lat.close()
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("faces", list(FACES))
@pytest.mark.parametrize("shape", [(5, 5, 31500), (33, 31, 770), (8800, 30, 3), (100, 98, 81), (4, 1020, 200), (393, 3, 680)])
def test_two_steps_equal_single_steps(faces, shape):
    storage = "f64" if "neem" in faces else "f32"
    force = (1e-5, 2e-6, 0.0) if faces in ("periodic", "channel") else (0.0, 0.0, 0.0)
    for f in {(0.0, 0.0, 0.0), (force[0], 0.0, 0.0), force}:
        a, b = both(shape, storage, FACES[faces], (2, 5), force=f)
        assert np.isfinite(a).all() and np.array_equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("storage", ["f32", "f64"])
@pytest.mark.parametrize("faces", ["periodic", "lid", "neem"])
def test_two_steps_with_solids(storage, faces):
    shape = (107, 90, 83)
    for solid in (None, solids(shape, faces)):
        a, b = both(shape, storage, FACES[faces], (4, 3), solid=solid)
        assert np.isfinite(a).all() and np.array_equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("storage", ["f16", "bf16"])
def test_two_steps_16_bit_box(storage):
    a, b = both((150, 143, 149), storage, {}, (2, 3), force=(1e-5, 2e-6, 0.0))
    assert np.isfinite(a).all() and np.array_equal(a, b)
