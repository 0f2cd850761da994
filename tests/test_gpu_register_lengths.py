"""The register-resident transforms of 3 2^k and 5 2^k points (8, m, 8 and
8, q, 2^j with L / 8 threads per line) on each axis they serve, whole and
half-empty lines, every output of the z pass (one launch per field, the
filtered velocity of periodic boxes among them), and the scalar solve, against
the oracle at the solver's bars (FP64 1e-12 relative L-inf, FP32 1e-5
relative L2)."""
import numpy as np
import pytest

import pmlib3d_amd as pm
from oracle import oracle as O
from tests.helpers import blob_field, rel_l2, rel_linf

pytestmark = pytest.mark.gpu

LENGTHS = [48, 80, 96, 160, 192, 320, 384, 640, 768]


def _agree(got, ref, prec):
    e = rel_linf(got, ref) if prec == pm.FP64 else rel_l2(got, ref)
    assert e <= (1e-12 if prec == pm.FP64 else 1e-5), e


# (a periodic box's long waves carry the FP32 rounding of its mean, divided by
# k^2: no measure of the transforms)
@pytest.mark.parametrize("prec,periodic", [(pm.FP64, False), (pm.FP64, True), (pm.FP32, False)],
                         ids=["f64-free", "f64-periodic", "f32-free"])
@pytest.mark.parametrize("L", LENGTHS)
def test_lines_of_every_length(L, prec, periodic):
    bc = (1, 1, 1) if periodic else (0, 0, 0)
    m = L if periodic else L // 2
    h = 1.0 / 16
    k = 32 if periodic else 16   # (the scalar solve takes specialised lengths only)
    for n in ((k, k, m), (k, m, k)):
        print("case", L, n, bc, prec, flush=True)
        xmin = [-0.5 * h * v for v in n]
        g, q = O.make_geom(n, 0, xmin, h, bc), O.make_params(4, 1, 2.0)
        w = blob_field(g, seed=L + periodic, nblob=4, width=0.02)
        Gh = O.poisson_setup(g, q)
        patch = pm.Patch(xmin=tuple(xmin), xmax=tuple(-v for v in xmin), ncell=n, dx=(h,) * 3, bound_cond=bc, nghost=0)
        s = pm.PoissonSolver(patch, prec, order=4, kernel=1, eps_radius=2.0, interp_order=3)
        s.setup()
        for reproj, psi in ((False, False), (True, True), (True, False)):
            for got, ref in zip(s.solve(w, reproj=reproj, calc_vecpot=psi),
                                O.poisson_solve(g, q, Gh, w, False, reproj, psi)):
                assert (got is None) == (ref is None)
                if ref is not None:
                    _agree(got, ref, prec)
        _agree(s.solve_scalar(np.asfortranarray(w[0])), O.poisson_solve(g, q, Gh, w, False, False, True)[2][0], prec)
