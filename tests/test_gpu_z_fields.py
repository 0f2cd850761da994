"""Solves with more outputs than the velocity, whose z pass forms them in one
launch or in a launch each by length, precision, boundary kind and number of
blocks: both sides of that choice, every combination of outputs, against the
oracle at the solver's bars (FP64 1e-12 relative L-inf, FP32 1e-5 relative L2;
periodic boxes in FP64 only: their long waves carry the FP32 rounding of the
mean, divided by k^2)."""
import numpy as np
import pytest

import pmlib3d_amd as pm
from oracle import oracle as O
from tests.helpers import blob_field, rel_l2, rel_linf

pytestmark = pytest.mark.gpu

FREE, MIXED, PERIODIC = (0, 0, 0), (1, 1, 0), (1, 1, 1)
CASES = [((16, 16, m), FREE) for m in (32, 64, 128, 256, 512, 80, 320)]                # few blocks
CASES += [((48, 64, m), FREE) for m in (32, 256, 80, 96)]                              # many
CASES += [((16, 20, 256), MIXED), ((96, 128, 96), MIXED), ((30, 16, 512), MIXED)]
CASES += [((16, 16, m), PERIODIC) for m in (64, 256, 512, 160, 384, 768, 1024)]
CASES += [((96, 96, 96), PERIODIC), ((128, 96, 64), PERIODIC)]


@pytest.mark.parametrize("n,bc,prec", [(n, bc, p) for n, bc in CASES for p in (pm.FP64, pm.FP32)
                                       if p == pm.FP64 or bc != PERIODIC])
def test_outputs_of_the_z_pass(n, bc, prec):
    h = 1.0 / 16
    print("case", n, bc, prec, flush=True)
    xmin = [-0.5 * h * v for v in n]
    g, q = O.make_geom(n, 0, xmin, h, bc), O.make_params(6, 1, 2.0)
    w = blob_field(g, seed=sum(n), nblob=4, width=0.02)
    Gh = O.poisson_setup(g, q)
    patch = pm.Patch(xmin=tuple(xmin), xmax=tuple(-v for v in xmin), ncell=n, dx=(h,) * 3, bound_cond=bc, nghost=0)
    s = pm.PoissonSolver(patch, prec, order=6, kernel=1, eps_radius=2.0, interp_order=3)
    s.setup()
    for reproj, psi in ((False, True), (True, False), (True, True)):
        for got, ref in zip(s.solve(w, reproj=reproj, calc_vecpot=psi), O.poisson_solve(g, q, Gh, w, False, reproj, psi)):
            assert (got is None) == (ref is None)
            if ref is not None:
                e = rel_linf(got, ref) if prec == pm.FP64 else rel_l2(got, ref)
                assert e <= (1e-12 if prec == pm.FP64 else 1e-5), e
