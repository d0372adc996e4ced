"""Read-backs around the sizes where their path changes (16 MB in pinned
chunks of 2 MB; small domains of a batch through pinned memory): the initial
state, whose density and velocity the first collision keeps, comes back to
within the FP64 rounding of a sum of 9 or 19 populations of order one."""
import numpy as np
import pytest

from lbm_amd import capi, poisson


def start(n, dim, seed):
    rng = np.random.default_rng(seed)
    return 1 + 1e-2 * rng.standard_normal(n), 0.05 * rng.standard_normal((n, dim))


# (1 + dim) doubles per cell: one cell short of 16 MB, 16 MB, one row and some
# chunks more, an array that ends inside a chunk in 3D
@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(40, 30), (863, 809), (1024, 683), (1031, 1021), (64, 64, 128), (101, 103, 97)])
def test_macros_of_the_initial_state(shape):
    n, dim = int(np.prod(shape)), len(shape)
    rho, u = start(n, dim, n)
    lat = capi.Lattice(shape, storage="f64", omega=1.0, faces={})
    lat.init(rho, u)
    for _ in range(2):
        r, v = lat.macros()
        assert np.abs(r - rho).max() < 1e-14 and np.abs(v - u).max() < 1e-14
    f = lat.populations()
    assert np.abs(f.sum(0) - rho).max() < 1e-13 or np.abs(f.sum(0) + 1 - rho).max() < 1e-13
    lat.close()


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny", [(64, 64), (1447, 1449), (2000, 1500)])
def test_phi_of_the_initial_state(nx, ny):
    phi0 = np.random.default_rng(nx).random(nx * ny)
    p = poisson.Poisson(5, nx, ny, 1.0, 0.0)
    p.set_faces({f: ("neumann", None, k) for k, f in enumerate(("-x", "+x", "-y", "+y"))})
    p.init(phi0)
    assert np.abs(p.phi() - phi0).max() < 1e-14
    p.close()


@pytest.mark.gpu
@pytest.mark.parametrize("ndom", [3, 9])
def test_macros_of_batch_domains(ndom):
    shapes = [(20 + 7 * k, 10 + 3 * k) for k in range(ndom - 1)] + [(300, 301)]  # the last beyond 2 MB
    fields = [start(a * b, 2, a) for a, b in shapes]
    b = capi.Batch([{"shape": s, "omega": 1.0, "faces": {}} for s in shapes], storage="f64")
    b.init(np.concatenate([f[0] for f in fields]), np.concatenate([f[1] for f in fields]))
    for k in list(range(ndom)) + [0, ndom - 1, 1]:
        r, v = b.macros(k)
        assert np.abs(r - fields[k][0]).max() < 1e-14 and np.abs(v - fields[k][1]).max() < 1e-14, k
    b.close()
