"""Observer interpolation with neighbour counts around the 64 lanes of a wave
(none, one, one less and one more than a wave, several waves' worth), against
the oracle.

Tolerances: the weights are positive, so the quotient of two sums of m <= 200
terms is off by at most a few m eps: 200 x 2.2e-16 x 8 < 1e-12 in FP64.  In
FP32-mixed the float positions (|x| < 1, h = 0.13) move q by up to
2 x 6e-8 / 0.13 = 1e-6, the kernel by less than 3 times that of its mean, and
the sums add 200 x 6e-8 = 1.2e-5 at most: 3e-5."""
import numpy as np
import pytest

from sphinxsys_amd import _capi as capi
from sphinxsys_amd import ck

pytestmark = pytest.mark.gpu


def observed(lib, dim, precision, points, pressure, velocity, observers):
    ctx = ck.Context(lib)
    fluid = ck.Body(ctx, dim, len(points), 0.1, capi.BODY_FLUID, precision)
    obs = ck.Body(ctx, dim, len(observers), 0.1, capi.BODY_OBSERVER, precision)
    for body, x in ((fluid, points), (obs, observers)):
        body.write("Position", x)
        body.write("VolumetricMeasure", np.full(len(x), 0.1 ** dim))
    fluid.write("Pressure", pressure)
    fluid.write("Velocity", velocity)
    cll = ck.CellLinkedList(fluid, np.zeros(dim), np.ones(dim))
    contact = ck.Contact(obs, fluid, cll)
    ck.UpdateCellLinkedList(cll).exec()
    ck.UpdateRelation(contact).exec()
    sizes = contact.read()[0]
    out = ck.InterpolationContact(contact, "Pressure").exec(), ck.InterpolationContact(contact, "Velocity").exec()
    for o in (contact, cll, obs, fluid, ctx):
        o.close()
    return sizes, out


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("precision", [capi.FP64, capi.MIXED])
@pytest.mark.parametrize("m", [1, 63, 64, 65, 200])
def test_interpolation_around_a_wave_of_neighbours(hip, oracle, dim, precision, m):
    rng = np.random.default_rng(m + 10 * dim)
    centre = np.full(dim, 0.5)
    d = rng.normal(size=(m, dim))
    d *= (0.2 * rng.random(m) ** (1.0 / dim) / np.linalg.norm(d, axis=1))[:, None]
    points = centre + d
    observers = np.stack([np.full(dim, 0.95), centre])  # the first has no neighbour
    pressure, velocity = 1.0 + rng.random(m), 1.0 + rng.random((m, dim))
    sizes, got = observed(hip, dim, precision, points, pressure, velocity, observers)
    sizes_ref, want = observed(oracle, dim, capi.FP64, points, pressure, velocity, observers)
    assert np.array_equal(sizes, sizes_ref) and list(sizes) == [0, m]
    tol = 1e-12 if precision == capi.FP64 else 3e-5
    for g, w in zip(got, want):
        assert np.all(g[0] == 0.0) and np.all(w[0] == 0.0)
        assert np.all(np.abs(g[1] - w[1]) <= tol * np.abs(w[1])), (g, w)


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("precision", [capi.FP64, capi.MIXED])
@pytest.mark.parametrize("n_obs", [32768, 32769])
def test_interpolation_of_many_observers(hip, oracle, dim, precision, n_obs):
    """Both sides of the observer count from which one thread instead of a wave
    takes an observer, the last workgroup with one observer; the same tolerances."""
    rng = np.random.default_rng(n_obs + dim)
    m = 40 if dim == 2 else 12  # spacing 0.025 and 0.083, h = 0.13: at most 350 neighbours
    axis = (np.arange(m) + 0.5) / m
    points = np.stack([g.ravel() for g in np.meshgrid(*[axis] * dim, indexing="ij")], axis=1)
    pressure, velocity = 1.0 + rng.random(len(points)), 1.0 + rng.random((len(points), dim))
    observers = rng.random((n_obs, dim))
    sizes, got = observed(hip, dim, precision, points, pressure, velocity, observers)
    sizes_ref, want = observed(oracle, dim, capi.FP64, points, pressure, velocity, observers)
    assert np.array_equal(sizes, sizes_ref) and sizes.min() > 0 and sizes.max() <= 350
    tol = (1e-12 if precision == capi.FP64 else 3e-5) * 350 / 200
    for g, w in zip(got, want):
        assert np.all(np.abs(g - w) <= tol * np.abs(w)), np.max(np.abs(g - w) / np.abs(w))
