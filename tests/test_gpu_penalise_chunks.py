"""The penalisation kernel at the chunk lengths that its grid chooses (64 planes
and a remainder, 16, 8, 4), in both precisions and orders, with and without the
sums, against the oracle.  FP64: the vorticity bit-identical, the sums within
1e-12 of the largest.  FP32, from inputs exact in it: 2e-6 relative L-inf of the
vorticity (about a dozen roundings of terms no larger than the result's largest)
and 1e-5 of the largest sum (sums of FP32 vorticities, whose errors partly
cancel)."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import rel_linf

pytestmark = pytest.mark.gpu

CASES = [
    # ncell, nghost, bound_cond, fd_order
    ((65, 953, 127), 2, (0, 0, 0), 4),     # FP64 64 planes and 63
    ((130, 190, 135), 2, (0, 0, 0), 4),
    ((63, 5, 4), 1, (0, 0, 0), 2),
    ((64, 8, 9), 2, (0, 1, 0), 2),
    ((66, 15, 33), 2, (1, 0, 0), 2),
    ((129, 150, 70), 1, (0, 0, 0), 2),
]


@pytest.mark.parametrize("precision", [0, 1], ids=["f64", "f32"])
@pytest.mark.parametrize("case", CASES, ids=[str(i) for i in range(len(CASES))])
def test_penalise_chunks_match_oracle(case, precision):
    import torch
    import pmlib3d_amd as pm
    ncell, ng, bc, fd = case
    print("case", case, precision, flush=True)
    prec, dt = [(pm.FP64, torch.float64), (pm.FP32, torch.float32)][precision]
    g = O.make_geom(ncell, ng, [-0.5, -1.0, -0.25], 1.0 / 16, bc)
    patch = pm.Patch(xmin=tuple(g.xmin), xmax=tuple(g.xmax), ncell=tuple(g.ncell), dx=tuple(g.dx),
                     bound_cond=tuple(g.bound_cond), nghost=g.nghost)
    rng = np.random.default_rng(sum(ncell) + fd)
    shape = (3,) + O.mesh_extent(g)
    vel, vort = [np.asfortranarray(rng.normal(size=shape).astype(np.float32).astype(np.float64)) for _ in range(2)]
    chi = np.asfortranarray(rng.uniform(size=shape[1:]).astype(np.float32).astype(np.float64))
    want, sums = O.penalise(g, vel, chi, vort, relax=0.75, fd_order=fd)
    dev = lambda a: torch.from_numpy(a.ravel(order="F")).cuda().to(dt)  # noqa: E731
    d_vel, d_chi = dev(vel), dev(chi)
    diag = torch.zeros(8, dtype=torch.float64, device="cuda:0")
    for d_diag in (None, diag.data_ptr()):
        d_vort = dev(vort)
        pm.penalise_device_noalloc(patch, prec, d_vel.data_ptr(), d_chi.data_ptr(), d_vort.data_ptr(), d_diag=d_diag,
                                   relax=0.75, fd_order=fd)
        got = d_vort.double().cpu().numpy().reshape(shape, order="F")
        if precision == 0:
            assert np.array_equal(got, want)
        else:
            assert rel_linf(got, want) <= 2e-6
    got = diag[:5].cpu().numpy()
    assert np.abs(got - sums[:5]).max() <= (1e-12 if precision == 0 else 1e-5) * np.abs(sums).max()
