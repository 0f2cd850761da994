"""The mesh-to-particle gather's stencil rows read as runs of nodes: meshes
narrower than the stencil and little wider, stencils that leave the mesh on
either side of x, by one node or altogether, among ones that do not, and meshes
that hold infinities and NaN, against the oracle.

Bars: FP64 bit-identical, non-finite results included; FP32 1e-6 relative L2."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("io,bc", [(3, (0, 0, 0)), (3, (0, 1, 0)), (3, (1, 0, 0)), (4, (0, 0, 0)), (4, (1, 1, 0))])
@pytest.mark.parametrize("nx", [1, 2, 3, 4, 5, 6, 7, 9, 70])
def test_m2p_rows_match_oracle(nx, io, bc):
    import torch
    import pmlib3d_amd as pm
    if bc[0]:
        nx = max(nx, 6)   # (a periodic axis has at least two ghost layers' cells)
    print("case", nx, io, bc, flush=True)
    h = 1.0 / 16
    g = O.make_geom((nx, 8, 7), 0, [-0.5, -1.0, -0.25], h, bc, io)
    patch = pm.Patch(xmin=tuple(g.xmin), xmax=tuple(g.xmax), ncell=tuple(g.ncell), dx=tuple(g.dx),
                     bound_cond=tuple(g.bound_cond), nghost=g.nghost)
    rng = np.random.default_rng(nx + 10 * io)
    lo, hi = np.array(g.xmin), np.array(g.xmax)
    pos = rng.uniform(lo - [6 * h, h, 0.4 * h], hi + [6 * h, h, h], size=(2000, 3))
    pos[:600, 0] = np.sort(rng.uniform(lo[0], hi[0], 600))   # wavefronts with none and with a few outside
    pos = np.asfortranarray(pos.T)
    mesh = np.asfortranarray(rng.normal(size=(3,) + O.mesh_extent(g)))
    assert np.array_equal(pm.interp_mesh_field(patch, mesh, pos, interp_order=io), O.m2p(g, mesh, pos))
    d_pos = torch.from_numpy(pos.ravel(order="F")).cuda()
    d_m = torch.from_numpy(mesh.ravel(order="F")).cuda().float()
    d_out = torch.empty_like(d_pos)
    pm.ParticleOps(patch, io, pm.FP32).m2p(d_m.data_ptr(), d_pos.data_ptr(), pos.shape[1], d_out.data_ptr())
    assert rel_l2(d_out.cpu().numpy().reshape(pos.shape, order="F"), O.m2p(g, mesh, pos)) <= 1e-6
    bad = mesh.copy(order="F")
    at = rng.integers(0, mesh[0].size, 4)
    for v, i in zip((np.inf, -np.inf, np.nan, np.inf), at):
        bad[(rng.integers(0, 3),) + np.unravel_index(i, mesh.shape[1:], order="F")] = v
    with np.errstate(all="ignore"):
        want = O.m2p(g, bad, pos)
    assert np.array_equal(pm.interp_mesh_field(patch, bad, pos, interp_order=io), want, equal_nan=True)
