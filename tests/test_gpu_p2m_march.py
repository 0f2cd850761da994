"""The deposition of large meshes (marching wavefronts) against the oracle,
where its tiles end: x segments of 63 to 65 and more nodes, y chunks and z
groups with remainders, bin rows of more particles than are staged at a time
and of none, both kernels, boundary kinds, mesh types, accumulation, and meshes
on both sides of the rule that chooses it.

Bars: FP64 1e-12 relative L-inf (sums of the same terms in another order);
FP32 1e-6 relative L2 (below the rule compensated FP32 sums, above it FP64 sums
rounded once, periodic images added in FP32)."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import rel_l2, rel_linf

pytestmark = pytest.mark.gpu

CASES = [
    # ncell, nghost, bound_cond, interp_order
    ((4, 96, 95), 0, (0, 0, 0), 3),      # a few x nodes
    ((63, 98, 85), 0, (0, 0, 0), 3),     # segments of 63 nodes ...
    ((64, 127, 64), 0, (0, 0, 0), 3),    # (just below the FP64 rule)
    ((64, 131, 64), 0, (0, 0, 0), 3),    # ... 64 ...
    ((65, 64, 64), 0, (0, 0, 0), 3),     # ... and 65, at the FP64 rule's edge
    ((126, 70, 67), 0, (1, 1, 1), 3),    # just above the FP32 rule
    ((72, 70, 70), 1, (1, 0, 1), 3),     # above the FP64 rule, below the FP32 one
    ((130, 91, 61), 2, (0, 1, 0), 3),
    ((66, 64, 77), 0, (0, 0, 0), 4),
    ((60, 95, 97), 0, (1, 1, 1), 4),
    ((129, 62, 70), 3, (0, 1, 1), 4),
]


def _particles(g, seed):
    """Uniform ones well over the mesh's sides, a crowd in one cell and one
    along an x line, and a lone one where nothing else is."""
    rng = np.random.default_rng(seed)
    lo, hi, h = np.array(g.xmin), np.array(g.xmax), np.array(g.dx)
    mid = (lo + hi) / 2
    uni = rng.uniform(lo - 2 * h, [hi[0] + 2 * h[0], hi[1] + 2 * h[1], mid[2]], size=(12000, 3))
    cell = mid + rng.uniform(-0.4, 0.4, size=(150, 3)) * h
    line = mid + np.array([0, 5, -7]) * h + np.stack([rng.uniform(lo[0] - mid[0], hi[0] - mid[0], 500),
                                                      rng.uniform(-0.4, 0.4, 500) * h[1],
                                                      rng.uniform(-0.4, 0.4, 500) * h[2]], axis=1)
    lone = (hi - 2.25 * h)[None]
    pos = np.asfortranarray(np.concatenate([uni, cell, line, lone]).T)
    return pos, np.asfortranarray(rng.normal(size=pos.shape))


@pytest.mark.parametrize("precision", [0, 1], ids=["f64", "f32"])
@pytest.mark.parametrize("case", CASES, ids=[str(i) for i in range(len(CASES))])
def test_large_mesh_deposition_matches_oracle(case, precision):
    import torch
    import pmlib3d_amd as pm
    prec, dt = [(pm.FP64, torch.float64), (pm.FP32, torch.float32)][precision]
    ncell, ng, bc, io = case
    print("case", case, precision, flush=True)
    g = O.make_geom(ncell, ng, [-1.0, -0.5, -2.0], 1.0 / 16, bc, io)
    patch = pm.Patch(xmin=tuple(g.xmin), xmax=tuple(g.xmax), ncell=tuple(g.ncell), dx=tuple(g.dx),
                     bound_cond=tuple(g.bound_cond), nghost=g.nghost)
    pos, val = _particles(g, sum(ncell) + io)
    dev = torch.device("cuda:0")
    ops = pm.ParticleOps(patch, interp_order=io, precision=prec)
    ext = (3,) + O.mesh_extent(g)
    d_pos = torch.from_numpy(pos.ravel(order="F")).to(dev)
    d_val = torch.from_numpy(val.ravel(order="F")).to(dev)
    base = np.asfortranarray(np.random.default_rng(1).normal(size=ext).astype(np.float32).astype(np.float64))
    for clear in (True, False):
        d_mesh = torch.from_numpy(base.ravel(order="F")).to(dev).to(dt)
        ops.p2m(d_pos.data_ptr(), d_val.data_ptr(), pos.shape[1], d_mesh.data_ptr(), clear=clear)
        got = d_mesh.double().cpu().numpy().reshape(ext, order="F")
        ref = O.p2m(g, pos, val) if clear else O.p2m(g, pos, val, base.copy(order="F"), clear=False)
        if precision == 0:
            assert rel_linf(got, ref) <= 1e-12
        else:
            assert rel_l2(got, ref) <= 1e-6
