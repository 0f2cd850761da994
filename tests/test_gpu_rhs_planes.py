"""The vorticity right-hand side where its tiles and z chunks end: rows of 255
to 261 words, row groups with remainders, chunks of 2, 4, 8 and 16 planes and a
plane more or less, a NaN and an infinity among the values, both difference
orders, against the oracle: bit-identical."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

CASES = [
    # ncell, nghost, bound_cond
    ((85, 4, 3), 2, (0, 0, 0)),        # 255 words, 2 planes per chunk
    ((86, 5, 9), 2, (0, 0, 0)),
    ((87, 7, 2), 3, (0, 1, 0)),
    ((60, 130, 61), 2, (0, 0, 0)),     # 4 planes
    ((90, 134, 65), 2, (1, 0, 0)),     # 8
    ((171, 130, 65), 2, (0, 0, 1)),    # 16
]


@pytest.mark.parametrize("fd_order", [2, 4])
@pytest.mark.parametrize("case", CASES, ids=[str(i) for i in range(len(CASES))])
def test_vorticity_rhs_tiles_bit_identical(case, fd_order):
    import pmlib3d_amd as pm
    ncell, ng, bc = case
    print("case", case, fd_order, flush=True)
    g = O.make_geom(ncell, ng, [-0.5, -1.0, -0.25], (0.05, 0.06, 0.07), bc, 3)
    patch = pm.Patch(xmin=tuple(g.xmin), xmax=tuple(g.xmax), ncell=tuple(g.ncell), dx=tuple(g.dx),
                     bound_cond=tuple(g.bound_cond), nghost=g.nghost)
    rng = np.random.default_rng(sum(ncell))
    shape = (3,) + O.mesh_extent(g)
    w, u, d0 = [np.asfortranarray(rng.normal(size=shape)) for _ in range(3)]
    want = O.vort_rhs(g, w, u, 0.011, fd_order, dvort=d0)
    assert np.array_equal(pm.vorticity_rhs(patch, w, u, 0.011, fd_order=fd_order, dvort=d0, interp_order=3), want)
    w[(0,) + tuple(np.array(shape[1:]) // 2)] = np.nan
    u[(2,) + tuple(np.array(shape[1:]) // 3)] = np.inf
    with np.errstate(all="ignore"):
        want = O.vort_rhs(g, w, u, 0.011, fd_order, dvort=d0)
    got = pm.vorticity_rhs(patch, w, u, 0.011, fd_order=fd_order, dvort=d0, interp_order=3)
    assert np.array_equal(got, want, equal_nan=True)
