"""The FP64 neighbour sums against the oracle at the sizes where their form
changes (eight, four and one lanes per particle, the last from LDS-staged
records), bodies of less than a wave, last blocks of a few particles, and orders
in which the blocks of 256 particles have few enough distinct neighbours to be
staged (particles sorted), too many (a lattice's rows, a full shuffle) or some of
each (a sorted body shuffled in windows), the others read from global memory.

Gate: 1e-10 relative L2, the FP64 gate of the same comparison on smaller bodies.
Several lanes add every 4th or 8th term and then each other's sums, so the terms
(20 in 2D, 80 in 3D) come in another order than the oracle's.  A sum of m terms in
any order is off by at most m eps times the sum of their magnitudes, 80 x 1.1e-16
= 9e-15 of it, and terms of random sign leave a result of a tenth to a hundredth
of that sum: 1e-12, and as much again for the roundings of the terms."""
import numpy as np
import pytest

from sphinxsys_amd import _capi as capi
from sphinxsys_amd import cases, ck
from tests.test_gpu_parity import FP64_GATE, Pair, jittered_lattice, rel_l2, shuffled

pytestmark = pytest.mark.gpu


# distinct neighbours of a block that the summation, the first and the second pass stage
CAPS = {2: (768, 768, 768), 3: (1536, 1344, 1440)}


def distinct_neighbours(relation):
    """Per block of 256 particles, from its lists."""
    size, offset, index = relation.read()
    return np.array([len(np.unique(index[offset[i]:offset[min(i + 256, len(size))]])) for i in range(0, len(size), 256)])


@pytest.mark.parametrize("dim,m,order", [(2, 7, "rows"), (2, 362, "sorted"), (2, 363, "sorted"), (2, 363, "windows"),
                                         (2, 363, "rows"), (2, 363, "shuffled"),
                                         (3, 5, "rows"), (3, 25, "sorted"), (3, 26, "rows"), (3, 54, "sorted"),
                                         (3, 55, "sorted"), (3, 55, "windows"), (3, 55, "rows"), (3, 55, "shuffled")])
def test_fp64_sums_staged_and_not(hip, oracle, dim, m, order):
    dp = 0.02
    fluid = jittered_lattice(dim, m, dp, 3)
    wall = jittered_lattice(dim, m, dp, 5, jitter=0.0)
    wall = wall[wall[:, -1] < 3 * dp].copy()
    wall[:, -1] -= 3 * dp
    if order == "shuffled":
        fluid = shuffled(fluid, 0, 4)
    pr = Pair(hip, oracle, fluid, dp, wall, np.tile(np.eye(dim)[-1], (len(wall), 1)), capi.FP64, rho0=1000.0, c0=20.0)
    if order in ("sorted", "windows"):
        pr.both(lambda s: ck.ParticleSortCK(s["f"], s["fc"]).exec())
        if order == "windows":
            pr.write("Position", shuffled(pr.read("Position")[0], 300, 4))
        pr.both(lambda s: ck.UpdateCellLinkedList(s["fc"]).exec())
        pr.both(lambda s: ck.UpdateRelation(s["inner"], *s["walls"]).exec())
    if m in (363, 55):
        staged = [np.mean(distinct_neighbours(pr.gpu["inner"]) <= cap) for cap in CAPS[dim]]
        print(f"{dim}D {order}: staged blocks {staged}", flush=True)
        for part in staged:
            assert {"sorted": part > 0.5, "windows": 0.05 < part < 0.95}.get(order, part < 0.05), staged
    rng = np.random.default_rng(6)
    n = len(fluid)
    pr.write("Compression", 1.0 + rng.uniform(-0.01, 0.01, n))
    pr.write("CompressionRate", rng.uniform(-0.5, 0.5, n))
    pr.write("Velocity", rng.normal(scale=0.3, size=(n, dim)))
    pr.both(lambda s: ck.CompressionSummation(s["inner"], *s["walls"]).exec())
    pr.both(lambda s: ck.LinearCorrectionMatrixComplex(s["inner"], *s["walls"], alpha=0.5).exec())
    pr.both(lambda s: ck.FreeSurfaceIndicationComplexSpatialTemporalCK(s["inner"], *s["walls"]).exec())
    g, c = pr.read("Indicator")
    assert np.array_equal(g, c)
    names = ["CompressionSummation", "LinearCorrectionMatrix", "PositionDivergence"]
    for correction in (capi.CORRECTION_NONE, capi.CORRECTION_LINEAR):
        pr.both(lambda s: ck.AcousticStep1stHalf(s["inner"], *s["walls"], correction=correction).exec(2e-5))
        pr.both(lambda s: ck.AcousticStep2ndHalf(s["inner"], *s["walls"], correction=correction).exec(2e-5))
        for name in names + ["Pressure", "Force", "CompressionRate", "Compression", "Velocity", "Displacement"]:
            g, c = pr.read(name)
            assert rel_l2(g, c) < FP64_GATE, (correction, name)
        pr.both(lambda s: ck.ViscousForceCK(s["inner"], *s["walls"], mu=0.1, correction=correction).exec())
        pr.both(lambda s: ck.KernelGradientIntegral(s["inner"], *s["walls"], correction=correction).exec())
        for name in ("ViscousForce", "KernelGradientIntegral"):
            g, c = pr.read(name)
            assert rel_l2(g, c) < FP64_GATE, (correction, name)
    pr.close()


@pytest.mark.parametrize("precision", [capi.FP64, capi.MIXED])
def test_lists_rebuilt_between_batch_steps(hip, precision):
    """A caller that rebuilds a scene's lists between two batch steps may leave
    their staging sets (FP64) to the next reader: the batched scene still equals itself alone."""
    geom = cases.dambreak_2d(dp=0.0038)  # 138,000 particles: staged in both precisions
    alone, batched = (cases.DamBreak(hip, geom, precision) for _ in range(2))
    for sc in (alone, batched):
        sc.initialize()
        sc.ctx.synchronize()
    batch = ck.BatchAdvection(hip, [batched.advection], options=dict(use_graph=1, autotune=0))
    for _ in range(4):
        alone.advection_step()
        batch.exec()
        batched.complex_relation.exec()
        batched.ctx.synchronize()
    for name in ("Position", "Velocity", "Compression", "Force"):
        assert np.array_equal(alone.fluid.read(name), batched.fluid.read(name)), name
    batch.close()
    alone.close()
    batched.close()
