"""ParticleSortCK bit-exact with the oracle around the sizes up to which one
workgroup sorts the keys (8,192; powers of two and their neighbours), with many
equal keys: sequence, identifiers and every evolving variable."""
import numpy as np
import pytest

from sphinxsys_amd import _capi as capi
from sphinxsys_amd import ck

pytestmark = pytest.mark.gpu

FIELDS = ["SortSequence", "OriginalID", "SortedID", "Position", "VolumetricMeasure", "Velocity", "Mass", "ForcePrior",
          "Compression", "CompressionRate", "PreviousSurfaceIndicator", "PreviousViscousForce"]


@pytest.mark.parametrize("kind", [capi.BODY_FLUID, capi.BODY_SOLID])
@pytest.mark.parametrize("n,dim", [(1, 2), (2, 3), (3, 2), (1023, 3), (4096, 2), (4097, 3), (8192, 3), (8193, 2)])
def test_sort_of_one_workgroup(hip, oracle, n, dim, kind):
    rng = np.random.default_rng(n)
    fields = [f for f in FIELDS if kind == capi.BODY_FLUID or not f.startswith("Previous")]
    x = rng.random((n, dim))
    values = {"Velocity": rng.normal(size=(n, dim)), "ForcePrior": rng.normal(size=(n, dim)),
              "Compression": rng.normal(size=n), "CompressionRate": rng.normal(size=n),
              "PreviousSurfaceIndicator": rng.integers(0, 2, n), "PreviousViscousForce": rng.normal(size=(n, dim))}
    volume = 1.0 + rng.random(n)
    read = []
    for lib in (hip, oracle):
        ctx = ck.Context(lib)
        body = ck.Body(ctx, dim, n, 0.05, kind, rho0=2.0, c0=1.0)
        body.write("Position", x)
        body.write("VolumetricMeasure", volume)
        for f, v in values.items():
            if f in fields:
                body.write(f, v)
        cll = ck.CellLinkedList(body, np.zeros(dim), np.ones(dim))  # cells of 0.13: many particles in each
        ck.UpdateCellLinkedList(cll).exec()
        ck.ParticleSortCK(body, cll).exec()
        read.append([body.read(f) for f in fields])
        # the records of the neighbour search follow the order
        ck.UpdateCellLinkedList(cll).exec()
        inner = ck.Inner(body, cll)
        ck.UpdateRelation(inner).exec()
        read[-1] += list(inner.read())
        for o in (inner, cll, body, ctx):
            o.close()
    for f, g, c in zip(fields + ["size", "offset", "index"], *read):
        assert np.array_equal(g, c), f
