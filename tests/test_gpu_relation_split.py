"""Neighbour lists bit-exact with the oracle on both sides of the size from which
one wave instead of four builds a chunk of 64 particles (262,144 particles; inner
relations in 3D 153,600),
with a last chunk of a few particles, a window-shuffled order (sources of many
cells in a chunk), and a cluster whose search boxes hold more candidates than
the build keeps in registers (512)."""
import numpy as np
import pytest

from sphinxsys_amd import _capi as capi
from tests.test_gpu_parity import Pair, jittered_lattice, shuffled

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,m,cluster", [(2, 511, 0), (2, 513, 700), (3, 63, 600), (3, 64, 0), (3, 65, 600), (3, 4, 0),
                                           (3, 53, 600), (3, 54, 600)])
def test_lists_built_by_one_and_four_waves(hip, oracle, dim, m, cluster):
    dp = 0.02
    fluid = shuffled(jittered_lattice(dim, m, dp, 8), 200, 9)
    rng = np.random.default_rng(10)
    fluid = np.concatenate([fluid, 2.5 * dp + rng.uniform(0.0, 1.5 * dp, size=(cluster, dim))])
    wall = jittered_lattice(dim, m, dp, 11, jitter=0.0)
    wall = wall[wall[:, -1] < 2 * dp].copy()
    wall[:, -1] -= 2 * dp
    pr = Pair(hip, oracle, fluid, dp, wall, np.tile(np.eye(dim)[-1], (len(wall), 1)), capi.MIXED)
    for name in ("inner", "walls"):
        for g, o in zip(*[[s[name]] if name == "inner" else s[name] for s in pr.sides]):
            for a, b in zip(g.read(), o.read()):
                assert np.array_equal(a, b), name
    pr.close()
