"""Bin keys of large sets, whose threads take several particles: particles in
random order, runs of neighbouring lanes in one bin (across
wavefront edges too), and particles without a bin, against the oracle's
deposition.  Bar: FP64 1e-12 relative L-inf (sums of the same terms in another
order)."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import rel_linf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,bc", [(6291456, (0, 0, 0)), (8388608 + 77, (1, 1, 0))])
def test_large_set_deposition_matches_oracle(n, bc):
    import torch
    import pmlib3d_amd as pm
    print("case", n, bc, flush=True)
    g = O.make_geom((128, 128, 128), 0, [-1.0, -0.5, -2.0], 1.0 / 64, bc, 3)
    patch = pm.Patch(xmin=tuple(g.xmin), xmax=tuple(g.xmax), ncell=tuple(g.ncell), dx=tuple(g.dx),
                     bound_cond=tuple(g.bound_cond), nghost=g.nghost)
    rng = np.random.default_rng(n)
    lo, hi, h = np.array(g.xmin), np.array(g.xmax), np.array(g.dx)
    pos = rng.uniform(lo - 3 * h, hi + 3 * h, size=(n, 3))
    runs = np.repeat(np.arange(n), rng.integers(1, 5, n))[:n]      # runs of 1 to 4 in one place ...
    half = np.arange(n) < n // 2
    pos[half] = pos[runs[half]]
    pos[:70] = (lo + hi) / 2                                       # ... and one beyond a wavefront
    pos = np.asfortranarray(pos.T)
    val = np.asfortranarray(rng.normal(size=pos.shape))
    ref = O.p2m(g, pos, val)
    d = [torch.from_numpy(a.ravel(order="F")).cuda() for a in (pos, val)]
    mesh = torch.zeros(ref.size, dtype=torch.float64, device="cuda")
    ops = pm.ParticleOps(patch, interp_order=3, precision=pm.FP64)
    ops.p2m(d[0].data_ptr(), d[1].data_ptr(), n, mesh.data_ptr())
    err = rel_linf(mesh.cpu().numpy().reshape(ref.shape, order="F"), ref)
    print("error", err, flush=True)
    assert err <= 1e-12
