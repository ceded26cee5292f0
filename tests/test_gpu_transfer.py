"""Body.write followed by Body.read returns the written values in the body's
precision, exactly, for each device layout (three arrays, 4-wide records, one
array, matrix components, 32-bit integers), with sizes on both sides of the
context's own pinned buffer (262,144 bytes), of one half of a staging buffer
(8 MiB) and over more than two halves, and of the sizes up to which a field of one
array is copied as it lies: reads of 131,072 doubles, 524,288 floats and 262,144
identifiers, writes of 524,288 doubles and 1,048,576 32-bit values, 8,192
velocities in double and 131,072 in float; after a synchronization and behind
queued work."""
import numpy as np
import pytest

from sphinxsys_amd import _capi as capi
from sphinxsys_amd import ck

pytestmark = pytest.mark.gpu

# name, values per particle in D dimensions, kept in double in both precisions
FIELDS = [("Position", lambda d: d, True), ("Velocity", lambda d: d, False), ("Pressure", lambda d: 1, False),
          ("Compression", lambda d: 1, False), ("Force", lambda d: d, False),
          ("LinearCorrectionMatrix", lambda d: d * d, False)]


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("precision", [capi.FP64, capi.MIXED])
@pytest.mark.parametrize("n", [1, 257, 3641, 8192, 8193, 10923, 32769, 131072, 131073, 262144, 262145, 349526, 524288,
                               524289, 800001, 1048576, 1048577])
def test_write_read_round_trip(hip, dim, precision, n):
    rng = np.random.default_rng(n)
    ctx = ck.Context(hip)
    body = ck.Body(ctx, dim, n, 0.01, capi.BODY_FLUID, precision)
    kept = {}
    for name, width, double in FIELDS:
        v = rng.normal(size=(n, width(dim)) if width(dim) > 1 else n)
        v.flat[0] = -0.0
        if name == "Compression":
            v = 1.0 + 0.01 * v
        if name == "LinearCorrectionMatrix":
            v = v.reshape(n, dim, dim)
        body.write(name, v)
        if precision == capi.MIXED and not double:
            v = (v - 1.0).astype(np.float32).astype(float) + 1.0 if name == "Compression" else v.astype(np.float32)
        kept[name] = v.astype(float)
    ids = rng.permutation(n).astype(np.uint32)
    body.write("OriginalID", ids)
    setup = ck.AdvectionStepSetup(body)  # sets the volumes and displacements, which are not read here
    for queued in (False, True):
        for name, v in kept.items():
            if queued:
                setup.exec()  # returns before its kernel ends
            got = body.read(name)
            assert np.array_equal(got, v) and np.array_equal(np.signbit(got), np.signbit(v)), (name, queued)
    assert np.array_equal(body.read("OriginalID"), ids)
    body.close()
    ctx.close()
