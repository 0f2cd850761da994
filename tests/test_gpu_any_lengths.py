"""Solves at transform lengths without a compile-time specialisation: every
radix of the run-time engine (2 .. 13) as first, middle and last stage, one
stage alone, rows that end inside a step, all outputs, both kernels and every
boundary condition, against the oracle at the solver's own bars (FP64 1e-12
relative L-inf, FP32 1e-5 relative L2)."""
import numpy as np
import pytest

import pmlib3d_amd as pm
from oracle import oracle as O
from tests.helpers import blob_field, rel_l2, rel_linf

pytestmark = pytest.mark.gpu

# cells per axis (free axes transform twice as many): the long axis walks
# through the passes
LONG = [9, 11, 13, 14, 15, 21, 22, 25, 26, 27, 33, 35, 39, 45, 49, 50, 54, 63, 65, 66, 77, 81, 91, 98, 99, 117, 121,
        125, 126, 130, 143, 169, 180, 195, 198, 231, 242, 250, 273]
FREE = [((m, 6, 5), (5, m, 6), (6, 7, m))[i % 3] for i, m in enumerate(LONG)]
FREE += [((m, 6, 5), (5, m, 6), (6, 7, m))[(i + 1) % 3] for i, m in enumerate(LONG[::2])]


def _solve(n, bc, ng, prec, order, kernel, reproj, psi):
    # a power of two: the kernel grid's origin is then exactly r = 0 (kernel 2
    # divides by r^3, and a rounded origin is noise in the oracle as well)
    h = 1.0 / 16
    xmin = [-0.5 * h * v for v in n]
    g = O.make_geom(n, ng, xmin, h, bc)
    w = blob_field(g, seed=sum(n))
    ref = O.poisson_solve(g, O.make_params(order, kernel, 2.0), O.poisson_setup(g, O.make_params(order, kernel, 2.0)), w,
                          False, reproj, psi)
    p = pm.Patch(xmin=tuple(xmin), xmax=tuple(-v for v in xmin), ncell=n, dx=(h,) * 3, bound_cond=bc, nghost=ng)
    s = pm.PoissonSolver(p, prec, order=order, kernel=kernel, eps_radius=2.0, interp_order=3)
    s.setup()
    return s.solve(w, reproj=reproj, calc_vecpot=psi), ref


def _check(got, ref, prec):
    for a, b in zip(got, ref):
        assert (a is None) == (b is None)
        if a is not None:
            e = rel_linf(a, b) if prec == pm.FP64 else rel_l2(a, b)
            assert e <= (1e-12 if prec == pm.FP64 else 1e-5), e


@pytest.mark.parametrize("n", FREE)
def test_free_velocity(n):
    got, ref = _solve(n, (0, 0, 0), 0, pm.FP64, 4, 1, False, False)
    _check(got, ref, pm.FP64)


@pytest.mark.parametrize("n,bc,ng", [((22, 21, 31), (0, 0, 0), 2), ((13, 22, 45), (0, 0, 0), 0),
                                     ((42, 50, 27), (1, 1, 0), 0), ((26, 44, 70), (1, 1, 1), 0),
                                     ((90, 14, 36), (1, 1, 1), 0)])
@pytest.mark.parametrize("prec", [pm.FP64, pm.FP32])
@pytest.mark.parametrize("kernel", [1, 2])
def test_all_outputs(n, bc, ng, prec, kernel):
    got, ref = _solve(n, bc, ng, prec, 6, kernel, True, kernel == 1)
    _check(got, ref, prec)


@pytest.mark.parametrize("n", [(5, 6, 6), (11, 9, 13), (125, 7, 63), (6, 143, 50), (7, 9, 165)])
def test_single_precision(n):
    got, ref = _solve(n, (0, 0, 0), 0, pm.FP32, 4, 1, False, True)
    _check(got, ref, pm.FP32)
