"""Read-backs of one handle from several host threads: a batch's domains
(through pinned memory that its kernel writes, and through device staging),
and populations large enough for the pinned chunks."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from lbm_amd import capi


def start(shape, seed):
    rng = np.random.default_rng(seed)
    n = int(np.prod(shape))
    return 1 + 1e-2 * rng.standard_normal(n), 0.05 * rng.standard_normal((n, len(shape)))


@pytest.mark.gpu
@pytest.mark.parametrize("shapes", [[(90 + 5 * k, 60) for k in range(12)], [(120 * (k + 1), 200) for k in range(6)],
                                    [(1100, 900 + 10 * k) for k in range(4)]])
def test_batch_domains_from_several_threads(shapes):
    fields = [start(s, k) for k, s in enumerate(shapes)]
    b = capi.Batch([{"shape": s, "omega": 1.0, "faces": {}} for s in shapes], storage="f64")
    b.init(np.concatenate([f[0] for f in fields]), np.concatenate([f[1] for f in fields]))

    def read(i):
        k = i % len(shapes)
        if i % 5 == 4:
            return np.abs(b.populations(k).sum(0) - fields[k][0]).max()
        r, v = b.macros(k)
        return max(np.abs(r - fields[k][0]).max(), np.abs(v - fields[k][1]).max())

    with ThreadPoolExecutor(6) as pool:  # collision keeps density and velocity, to the rounding of nine additions
        assert max(pool.map(read, range(60))) < 1e-14 * 10
    b.close()


@pytest.mark.gpu
def test_populations_from_several_threads():
    lat = capi.Lattice((700, 600), storage="f64", omega=1.2)
    lat.init(*start((700, 600), 1))
    lat.step(3)
    alone = lat.populations()
    with ThreadPoolExecutor(4) as pool:
        for f in pool.map(lambda _: lat.populations(), range(8)):
            assert np.array_equal(f, alone)
    lat.close()
