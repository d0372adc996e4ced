"""Several Poisson steps per launch (k_poisson_multi) against as many calls
of one step: the same cell update on a tile in LDS, so phi and the check
values are equal bit for bit.  Windows smaller than a tile, one cell more than
whole tiles, every tile size of the plan, Dirichlet and Neumann faces in
several orders of application, calls that end in a check."""
import numpy as np
import pytest

FACES = {
    "dirichlet": (("-x", "d", 0), ("+x", "d", 1), ("-y", "d", 2), ("+y", "d", 3)),
    "neumann_x": (("-x", "n", 0), ("+x", "n", 1), ("-y", "d", 2), ("+y", "d", 3)),
    "neumann_y": (("-x", "d", 3), ("+x", "n", 1), ("-y", "n", 2), ("+y", "n", 0)),
    "neumann": (("-x", "n", 2), ("+x", "n", 3), ("-y", "n", 0), ("+y", "n", 1)),
}


def run(Q, nx, ny, faces, many, calls):
    from lbm_amd import poisson

    rng = np.random.default_rng(nx + ny)
    p = poisson.Poisson(Q, nx, ny, 1.3, -0.003)
    spec = {}
    for name, kind, prio in FACES[faces][:2 if Q == 3 else 4]:
        n = ny if name in ("-x", "+x") else nx
        spec[name] = ("dirichlet", rng.random(n), prio) if kind == "d" else ("neumann", None, prio)
    p.set_faces(spec)
    p.init(rng.random(nx * ny))
    out = []
    for n in calls:
        for _ in range(1 if many else n):
            p.step(n if many else 1)
        out += [p.phi(), np.array([p.step_check()[0]]), np.array([p.step_check()[0]])]
    out.append(p.phi())
    p.close()
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("faces", list(FACES))
@pytest.mark.parametrize("Q,nx,ny", [(3, 5, 1), (3, 65, 1), (3, 16500, 1), (3, 140000, 1), (5, 5, 5), (9, 5, 7), (9, 5, 300),
                                     (5, 300, 6), (9, 64, 64), (5, 129, 127), (9, 200, 130), (5, 301, 200), (9, 290, 222),
                                     (9, 513, 300)])
def test_multi_equals_single_steps(Q, nx, ny, faces):
    for a, b in zip(*(run(Q, nx, ny, faces, many, (2, 40, 13, 3)) for many in (True, False))):
        assert np.isfinite(a).all() and np.array_equal(a, b)
