"""The separable mesh-to-mesh kernels against the oracle where their tiles end:
meshes of one tile and of several with remainders, ratios 1 to 8 and broken
ones, cells of other proportions in the two meshes (a deposit from a mesh
coarser along an axis, interpolations from meshes finer along an axis, up to
one whose tile does not fit in LDS), both kernels and mesh types, clearing and
accumulating.

Bars: FP64 1e-13 of the largest value (sums of up to 48 terms per axis in
another order); FP32 5e-7 of it (FP64 sums rounded once per axis)."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

# (ncell, nghost, dx) from, the same to, bound_cond, interp_order
H = 1.0 / 16
CASES = [
    (((20, 18, 16), 2, H), ((10, 9, 8), 2, 2 * H), (0, 0, 0), 3),        # deposit, one tile
    (((262, 30, 20), 2, H), ((131, 15, 10), 2, 2 * H), (0, 0, 0), 3),    # several along x
    (((24, 140, 12), 3, H), ((12, 70, 6), 3, 2 * H), (0, 1, 0), 4),      # ... along y
    (((72, 48, 160), 3, H), ((18, 12, 40), 3, 4 * H), (1, 0, 1), 4),     # ... along z
    (((96, 80, 64), 3, H), ((12, 10, 8), 3, 8 * H), (0, 0, 0), 4),
    (((40, 44, 36), 1, H), ((16, 18, 14), 2, 2.5 * H), (0, 0, 0), 3),    # not a whole ratio
    (((30, 16, 45), 2, (H, 2 * H, H)), ((15, 32, 15), 2, (2 * H, H, 3 * H)), (0, 0, 0), 3),
    (((10, 9, 8), 2, 2 * H), ((20, 18, 16), 2, H), (0, 0, 0), 3),        # interpolation, one tile
    (((131, 15, 10), 3, 2 * H), ((262, 30, 20), 1, H), (0, 0, 0), 4),
    (((12, 70, 40), 3, 2 * H), ((24, 140, 80), 3, H), (0, 1, 1), 4),
    (((20, 22, 24), 2, H), ((20, 22, 24), 2, H), (1, 1, 1), 3),          # ratio 1
    (((12, 10, 8), 3, 8 * H), ((96, 80, 64), 2, H), (0, 0, 0), 4),
    (((16, 90, 30), 2, (1.5 * H, H / 6, H)), ((24, 15, 20), 2, (H, H, 1.5 * H)), (0, 0, 0), 3),
    (((8, 2100, 6), 2, (2 * H, H / 60, H)), ((16, 35, 6), 2, (H, H, H)), (0, 0, 0), 4),   # not in LDS
]


def _geoms(side, bc, io):
    import pmlib3d_amd as pm
    ncell, ng, dx = side
    xmin = (-0.5, -1.0, -0.25)
    g = O.make_geom(ncell, ng, xmin, dx, bc, io)
    return g, pm.Patch(xmin=tuple(g.xmin), xmax=tuple(g.xmax), ncell=tuple(g.ncell), dx=tuple(g.dx),
                       bound_cond=tuple(g.bound_cond), nghost=g.nghost)


@pytest.mark.parametrize("precision", [0, 1], ids=["f64", "f32"])
@pytest.mark.parametrize("case", CASES, ids=[str(i) for i in range(len(CASES))])
def test_m2m_tiles_match_oracle(case, precision, monkeypatch):
    import torch
    import pmlib3d_amd as pm
    monkeypatch.setenv("PMGPU_M2M_EXACT", "0")
    prec, dt = [(pm.FP64, torch.float64), (pm.FP32, torch.float32)][precision]
    src, dst, bc, io = case
    print("case", case, precision, flush=True)
    gf, pf = _geoms(src, bc, io)
    gt, pt = _geoms(dst, bc, io)
    rng = np.random.default_rng(io + sum(src[0]))
    draw = lambda g: np.asfortranarray(rng.normal(size=(3,) + O.mesh_extent(g)).astype(np.float32).astype(np.float64))
    fr, base = draw(gf), draw(gt)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a.ravel(order="F"))).cuda().to(dt)
    d_from = dev(fr)
    for clear in (True, False):
        d_to = dev(base)
        pm.interp_mesh_mesh_device(pf, pt, prec, d_from.data_ptr(), d_to.data_ptr(), clear=clear, interp_order=io)
        got = d_to.double().cpu().numpy().reshape(base.shape, order="F")
        want = O.interp_mesh_mesh(gf, gt, fr, base, clear=clear)
        assert np.abs(got - want).max() <= (1e-13, 5e-7)[precision] * np.abs(want).max()
