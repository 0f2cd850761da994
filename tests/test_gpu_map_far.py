"""Which map a call takes is read off the update: particles that one wrap brings
back into the patch, and single ones among many that it does not, on each axis
and at the edges of both (one wrap that ends just inside, or on the upper bound
by rounding; dropped ones far outside a free axis), in place and into a spare
set, against the oracle: bit-identical.  The bounds are exact in binary: where a
period taken off the upper bound rounds to below the lower one, the reference's
loop (particles/pmlib_particles_advance.f:145-166) does not end."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bc", [(1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 1, 1)])
@pytest.mark.parametrize("n", [1, 3000, 70001])
@pytest.mark.parametrize("what", ["one wrap", "far below", "far above", "edge", "far on free axes"])
def test_single_far_particles(bc, n, what):
    import torch
    import pmlib3d_amd as pm
    print("case", bc, n, what, flush=True)
    g = O.make_geom((12, 10, 8), 1, [0.0, -0.625, 0.0], 1.0 / 8, bc, 3)
    patch = pm.Patch(xmin=tuple(g.xmin), xmax=tuple(g.xmax), ncell=tuple(g.ncell), dx=tuple(g.dx),
                     bound_cond=tuple(g.bound_cond), nghost=g.nghost)
    rng = np.random.default_rng(n + sum(bc) + len(what))
    lo, hi = np.array(g.xmin), np.array(g.xmax)
    pos = rng.uniform(lo + 1e-3, hi - 1e-3, size=(n, 3)).T
    vel = rng.uniform(-0.3, 0.3, size=(3, n))     # leaves by less than a period
    k = n // 2
    for d in range(3):
        length = hi[d] - lo[d]
        if bc[d] and what == "far below":
            vel[d, k] = lo[d] - 1.5 * length - pos[d, k]
        elif bc[d] and what == "far above":
            vel[d, k] = hi[d] + 3.25 * length - pos[d, k]
        elif bc[d] and what == "edge":
            # on the bounds, just beyond them, and one period further
            at = [hi[d], np.nextafter(lo[d], -9), np.nextafter(hi[d], 9), hi[d] + length, lo[d] - length, lo[d]]
            at += [-1e-20] if lo[d] == 0.0 else []    # one wrap ends on the upper bound
            for i, x in enumerate(at[:n]):
                pos[d, (k + i) % n], vel[d, (k + i) % n] = x, 0.0
        elif not bc[d] and what == "far on free axes":
            vel[d, k] = 20.0
    arrs = [np.asfortranarray(a) for a in (pos, vel, rng.normal(size=(3, n)), rng.normal(size=(3, n)),
                                           np.zeros((3, n)), np.zeros((3, n)))]
    ref = O.advance(g, 2, 1, 1.0, *[a.copy(order="F") for a in arrs])
    left = ref[0].shape[1]
    dev = lambda: [torch.from_numpy(a.ravel(order="F")).cuda() for a in arrs]  # noqa: E731
    ptrs = lambda ts: [t.data_ptr() for t in ts]  # noqa: E731
    ops = pm.ParticleOps(patch, interp_order=3)
    here, there, spare = dev(), dev(), [torch.full_like(t, -7.0) for t in dev()]
    assert ops.advance(2, 1, 1.0, ptrs(here), n) == left
    got, swapped = ops.advance(2, 1, 1.0, ptrs(there), n, spare=ptrs(spare))
    assert got == left
    for a in (0, 2, 4, 5):
        for ts in (here, spare if swapped else there):
            assert np.array_equal(ts[a][:3 * left].cpu().numpy().reshape((3, left), order="F"), ref[a])
