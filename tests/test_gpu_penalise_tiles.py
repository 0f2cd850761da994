"""The penalisation kernel where its tiles and z chunks end (63 to 66 cells
along x, 7 to 17 along y, chunks of 4, 8 and 32 planes and a plane more), with
a chi and velocities that vary cell by cell, NaN and an infinity included,
against the oracle: the vorticity bit-identical, the sums within 1e-12 of the
largest."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

CASES = [
    # ncell, nghost, bound_cond, fd_order
    ((63, 7, 4), 2, (0, 0, 0), 4),
    ((64, 8, 5), 2, (0, 0, 0), 4),
    ((65, 9, 33), 3, (0, 0, 0), 2),
    ((66, 17, 9), 2, (0, 1, 0), 4),
    ((129, 16, 8), 1, (0, 0, 0), 2),
    ((6, 250, 70), 2, (1, 0, 0), 4),
    ((520, 520, 33), 2, (0, 0, 0), 4),     # chunks of 32 planes
]


@pytest.mark.parametrize("case", CASES, ids=[str(i) for i in range(len(CASES))])
def test_penalise_tiles_match_oracle(case):
    import pmlib3d_amd as pm
    ncell, ng, bc, fd = case
    print("case", case, flush=True)
    g = O.make_geom(ncell, ng, [-0.5, -1.0, -0.25], 1.0 / 16, bc)
    patch = pm.Patch(xmin=tuple(g.xmin), xmax=tuple(g.xmax), ncell=tuple(g.ncell), dx=tuple(g.dx),
                     bound_cond=tuple(g.bound_cond), nghost=g.nghost)
    rng = np.random.default_rng(sum(ncell) + fd)
    shape = (3,) + O.mesh_extent(g)
    vel, vort, field = [np.asfortranarray(rng.normal(size=shape)) for _ in range(3)]
    chi = np.asfortranarray(rng.uniform(size=shape[1:]))
    want, sums = O.penalise(g, vel, chi, vort, solid_vel=field, relax=0.8, fd_order=fd)
    got, got_sums = pm.penalise(patch, vel, chi, vort, solid_vel=field, us_const=None, relax=0.8, fd_order=fd)
    assert np.array_equal(got, want)
    assert np.abs(got_sums - sums).max() <= 1e-12 * np.abs(sums).max()
    # one bad cell spoils what its stencils reach and no more
    at = tuple((np.array(shape[1:]) // 2))
    for a, v in ((vel, np.nan), (field, np.inf)):
        a[(1,) + at] = v
        with np.errstate(all="ignore"):
            want = O.penalise(g, vel, chi, vort, solid_vel=field, relax=0.8, fd_order=fd)[0]
        got = pm.penalise(patch, vel, chi, vort, solid_vel=field, us_const=None, relax=0.8, fd_order=fd)[0]
        assert np.array_equal(got, want, equal_nan=True)
