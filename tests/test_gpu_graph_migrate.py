"""The recorded step's migration over many tiles of particles, with movers on
every axis and drops on the free ones, with its tile offsets added by the tiles
themselves and (large capacity) by their own launch, against the eager step:
the same particles, bit-identical, after every step."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("capacity", [40000, 2200000])
@pytest.mark.parametrize("bc,rk", [((0, 0, 0), 2), ((1, 1, 0), 3), ((1, 1, 1), 2)])
def test_recorded_migration_matches_eager_step(bc, rk, capacity):
    import pmlib3d_amd as pm
    n, h = 32, 2.0 / 32
    print("case", bc, rk, capacity, flush=True)
    patch = pm.Patch(xmin=(-1.0,) * 3, xmax=(1.0,) * 3, ncell=(n,) * 3, dx=(h,) * 3, bound_cond=bc)
    rng = np.random.default_rng(rk + sum(bc))
    pos = np.asfortranarray(rng.uniform(-1.0, 1.0, size=(3, 30000)))
    vort = np.asfortranarray(rng.normal(size=pos.shape) * 20.0)
    kw = dict(order=6, eps_radius=2.0, rk_order=rk, interp_order=3, capacity=capacity, precision=pm.FP64)
    eager, gs = pm.VortexStep(patch, **kw), pm.GraphVortexStep(patch, **kw)
    eager.load(pos, vort)
    gs.load(pos, vort)
    for k in range(3):
        before = eager.np
        eager.step(0.05 * h, 1e-2)
        gs.step(0.05 * h, 1e-2)
        a, b = eager.fetch(), gs.fetch()
        print("step", k, "particles", before, a[0].shape[1], b[0].shape[1], flush=True)
        assert a[0].shape == b[0].shape
        for x, y in zip(a, b):
            assert np.array_equal(x, y)
