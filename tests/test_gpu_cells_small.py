"""Cell lists bit-exact with the oracle on both sides of the sizes up to which one
workgroup makes them (4,096 particles, 16,384 cells), with one particle, with
particles out of cell order and with many particles in a cell."""
import numpy as np
import pytest

from sphinxsys_amd import _capi as capi
from sphinxsys_amd import ck

pytestmark = pytest.mark.gpu


def cell_list(lib, x, spacing, noalloc):
    ctx = ck.Context(lib)
    body = ck.Body(ctx, x.shape[1], len(x), 0.01, capi.BODY_FLUID)
    body.write("Position", x)
    cll = ck.CellLinkedList(body, np.zeros(x.shape[1]), np.ones(x.shape[1]), grid_spacing=spacing, buffer_width=0)
    lib.call("sphx_update_cell_linked_list_noalloc" if noalloc else "sphx_update_cell_linked_list", cll.h)
    out = cll.n_cells, cll.read()
    for o in (cll, body, ctx):
        o.close()
    return out


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("n,dim,per_axis", [(1, 2, 5), (63, 3, 1), (1024, 2, 128), (1025, 2, 129), (4096, 3, 25),
                                            (4097, 3, 25), (3000, 3, 26), (500, 2, 1)])
def test_cell_list_of_one_workgroup(hip, oracle, n, dim, per_axis, noalloc):
    rng = np.random.default_rng(n)
    x = rng.random((n, dim))
    x[: n // 4] = 0.5 + 0.2 / per_axis * (x[: n // 4] - 0.5)  # a quarter of them around one point
    got, want = (cell_list(lib, x, 1.0 / per_axis, noalloc) for lib in (hip, oracle))
    assert got[0] == want[0] == per_axis ** dim
    assert np.array_equal(got[1][0], want[1][0]) and np.array_equal(got[1][1], want[1][1])
