"""The map by classes (one classification for all axes, the list moved as
indices and class bytes, coordinates wrapped in the gather) on patches with
periodic axes, at tile edges and beyond the tiles that add their own offsets,
with few and many leaving, with particles that need several wraps (the general
path), in place and into a spare set, against the oracle: bit-identical."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bc", [(1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1)])
@pytest.mark.parametrize("n,speed,order", [(1, 2.0, 1), (2047, 0.3, 2), (2048, 0.02, 2), (2049, 0.3, 3),
                                           (5000, 8.0, 2), (50001, 0.05, 1), (2100001, 0.2, 2)])
def test_map_matches_oracle(n, speed, order, bc):
    import torch
    import pmlib3d_amd as pm
    print("case", n, speed, order, bc, flush=True)
    g = O.make_geom((12, 10, 8), 1, [-0.5, -0.4, -0.3], 1.0 / 10, bc, 3)
    patch = pm.Patch(xmin=tuple(g.xmin), xmax=tuple(g.xmax), ncell=tuple(g.ncell), dx=tuple(g.dx),
                     bound_cond=tuple(g.bound_cond), nghost=g.nghost)
    rng = np.random.default_rng(n + order + sum(bc))
    lo, hi = np.array(g.xmin), np.array(g.xmax)
    arrs = [np.asfortranarray(rng.uniform(lo + 1e-3, hi - 1e-3, size=(n, 3)).T)]
    arrs += [np.asfortranarray(rng.normal(size=(3, n)) * s) for s in (speed, 1.0, 0.5, 0.3 * speed, 0.2)]
    ref = O.advance(g, order, order, 0.4, *[a.copy(order="F") for a in arrs])
    left = ref[0].shape[1]
    carried = (0, 2, 4, 5) if order > 1 else (0, 2)
    dev = lambda: [torch.from_numpy(a.ravel(order="F")).cuda() for a in arrs]
    ptrs = lambda ts: [t.data_ptr() for t in ts]
    ops = pm.ParticleOps(patch, interp_order=3)
    here, there, spare = dev(), dev(), [torch.full_like(t, -7.0) for t in dev()]
    assert ops.advance(order, order, 0.4, ptrs(here), n) == left
    got, swapped = ops.advance(order, order, 0.4, ptrs(there), n, spare=ptrs(spare))
    assert got == left
    for k in carried:
        for ts in (here, spare if swapped else there):
            assert np.array_equal(ts[k][:3 * left].cpu().numpy().reshape((3, left), order="F"), ref[k])
