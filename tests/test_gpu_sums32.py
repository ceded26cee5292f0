"""The FP32-mixed neighbour sums of 2D bodies at the size where their form changes
(98,304 particles: four ordered lanes per particle below, one lane with LDS-staged
records from there on), against the FP64 oracle and against each other.

Tolerances against the oracle: those of the same comparisons on 40 particles a
side (test_gpu_parity.py, test_gpu_correction.py), times m / 40 for m a side:
positions are rounded to float relative to the domain, 6e-8 m dp, so the error of
a distance in units of h, and with it that of every sum, grows with m."""
import numpy as np
import pytest

from sphinxsys_amd import _capi as capi
from sphinxsys_amd import ck
from tests.test_gpu_parity import Pair, jittered_lattice, rel_l2, shuffled
from tests.test_gpu_sums64 import distinct_neighbours

pytestmark = pytest.mark.gpu

DP = 0.02


def slab(m):
    wall = jittered_lattice(2, m, DP, 5, jitter=0.0)
    wall = wall[wall[:, -1] < 3 * DP].copy()
    wall[:, -1] -= 3 * DP
    return wall, np.tile([0.0, 1.0], (len(wall), 1))


@pytest.mark.parametrize("m,ordered", [(313, 1.0), (313, 0.0), (314, 1.0), (314, 0.5), (314, 0.0)])
def test_mixed_sums_against_the_oracle(hip, oracle, m, ordered):
    """A part of the particles in a lattice's rows, whose blocks of 256 have few
    enough distinct neighbours to be staged, the rest shuffled, whose blocks have
    too many."""
    fluid = jittered_lattice(2, m, DP, 3)
    cut = int(ordered * len(fluid))
    fluid[cut:] = np.random.default_rng(4).permutation(fluid[cut:])
    pr = Pair(hip, oracle, fluid, DP, *slab(m), capi.MIXED, rho0=1000.0, c0=20.0)
    for cap in (1400, 1536):  # of the passes, of the other sums
        part = np.mean(distinct_neighbours(pr.gpu["inner"]) <= cap)
        print(f"{m} a side, {ordered} in rows: blocks staged {part}", flush=True)
        assert abs(part - ordered) < 0.05, part
    rng = np.random.default_rng(6)
    n = len(fluid)
    pr.write("Compression", 1.0 + rng.uniform(-0.01, 0.01, n))
    pr.write("CompressionRate", rng.uniform(-0.5, 0.5, n))
    pr.write("Velocity", rng.normal(scale=0.3, size=(n, 2)))

    def check(**tolerances):
        for name, tol in tolerances.items():
            g, c = pr.read(name)
            assert rel_l2(g, c) < tol * m / 40, (name, rel_l2(g, c))

    pr.both(lambda s: ck.CompressionSummation(s["inner"], *s["walls"]).exec())
    check(CompressionSummation=1e-6)
    pr.both(lambda s: ck.LinearCorrectionMatrixComplex(s["inner"], *s["walls"], alpha=0.5).exec())
    check(LinearCorrectionMatrix=1e-4)
    pr.both(lambda s: ck.FreeSurfaceIndicationComplexSpatialTemporalCK(s["inner"], *s["walls"]).exec())
    check(PositionDivergence=1e-5)
    g, c = pr.read("Indicator")
    assert np.count_nonzero(g != c) <= 0.005 * n
    for correction, force in ((capi.CORRECTION_NONE, 2e-4), (capi.CORRECTION_LINEAR, 5e-4)):
        pr.both(lambda s: ck.AcousticStep1stHalf(s["inner"], *s["walls"], correction=correction).exec(2e-5))
        check(Pressure=1e-5, Force=force, CompressionRate=5e-4, Velocity=1e-5)
        pr.both(lambda s: ck.AcousticStep2ndHalf(s["inner"], *s["walls"], correction=correction).exec(2e-5))
        check(Force=force, CompressionRate=5e-4, Compression=1e-6)
    pr.close()


@pytest.mark.parametrize("window", [None, 1024])
def test_four_ordered_lanes_equal_one_lane(hip, window):
    """A body below the line and the same particles with a distant block that lifts
    it over the line: every sum of the common particles is equal bit for bit."""
    m = 313
    fluid = jittered_lattice(2, m, DP, 3)
    if window is not None:
        fluid = shuffled(fluid, window, 4)
    n = len(fluid)
    block = jittered_lattice(2, 20, DP, 7) + [(m + 20) * DP, 0.0]
    wall, normals = slab(m)
    lo, up = np.array([-0.1, -0.2]), np.array([(m + 45) * DP, (m + 5) * DP])
    rng = np.random.default_rng(6)
    k = n + len(block)
    compression, rate = 1.0 + rng.uniform(-0.01, 0.01, k), rng.uniform(-0.5, 0.5, k)
    velocity = rng.normal(scale=0.3, size=(k, 2))
    read = []
    for x in (fluid, np.concatenate([fluid, block])):
        ctx = ck.Context(hip)
        f = ck.Body(ctx, 2, len(x), DP, capi.BODY_FLUID, capi.MIXED, rho0=1000.0, c0=20.0)
        w = ck.Body(ctx, 2, len(wall), DP, capi.BODY_SOLID, capi.MIXED, rho0=1000.0, c0=20.0)
        for b, p in ((f, x), (w, wall)):
            b.write("Position", p)
            b.write("VolumetricMeasure", np.full(len(p), DP ** 2))
        w.write("NormalDirection", normals)
        for name, v in (("Compression", compression), ("CompressionRate", rate), ("Velocity", velocity)):
            f.write(name, v[: len(x)])
        fc, wc = ck.CellLinkedList(f, lo, up), ck.CellLinkedList(w, lo, up)
        inner, contact = ck.Inner(f, fc), ck.Contact(f, w, wc)
        for c in (fc, wc):
            ck.UpdateCellLinkedList(c).exec()
        ck.UpdateRelation(inner, contact).exec()
        ck.CompressionSummation(inner, contact).exec()
        out = {"CompressionSummation": f.read("CompressionSummation")}
        ck.LinearCorrectionMatrixComplex(inner, contact, alpha=0.5).exec()
        for correction in (capi.CORRECTION_NONE, capi.CORRECTION_LINEAR):
            for half in (ck.AcousticStep1stHalf, ck.AcousticStep2ndHalf):
                half(inner, contact, correction=correction).exec(2e-5)
                for name in ("Pressure", "Force", "CompressionRate", "Compression", "Velocity", "Displacement"):
                    out[half.__name__, correction, name] = f.read(name)
        read.append(out)
        for o in (contact, inner, fc, wc, f, w, ctx):
            o.close()
    below, above = read
    for key in below:
        assert np.array_equal(below[key], above[key][:n]), key
