"""Solves at transform lengths from 1400 to 4200 without a compile-time
specialisation: five-stage plans, blocks of one unit of three lines up to the
160 KB of a CU, lines whose three-line unit does not fit (2401, 2450, 2520 ..),
which the former kernels still transform, and lengths past the run-time
engine's 4096.  Thin boxes with the long axis in each place, at the solver's
own bars: FP64 1e-12 relative L-inf, FP32 1e-5 relative L2 of the velocity.
Rounding noise is white and a long thin box amplifies it where |k| is small,
by about sqrt(L / 190) in a box of 4 x 5 cells: five at 4096, 2e-6 in FP32.

The reference is the oracle's kernel (green_real) with numpy's transforms: the
oracle's own transform advances its twiddles by repeated multiplication, as the
Fortran does, and is off by about L roundings, 1e-12 at 3328."""
import numpy as np
import pytest

import pmlib3d_amd as pm
from oracle import oracle as O
from tests.helpers import blob_field, rel_linf
from tests.test_gpu_any_lengths import _check

FREE = (0, 0, 0)
PER = (1, 1, 1)
MIXED = (1, 1, 0)


def _reference(g, prm, w, outputs):
    """velocity, reprojected vorticity and stream function of the mesh w (no
    free-side ghosts), poisson/pmlib_poisson_solve.f:119-233"""
    M = g.ncell[:]
    per = [b == 1 for b in g.bound_cond]
    L = [m if p else 2 * m for m, p in zip(M, per)]
    lo = [O.ng_side(g, d) for d in range(3)]
    cut = tuple([slice(None)] + [slice(lo[d], lo[d] + M[d]) for d in range(3)])
    W = np.fft.fftn(w[cut], s=L, axes=(1, 2, 3))
    k = np.stack(np.meshgrid(*[np.fft.fftfreq(L[d], g.dx[d]) for d in range(3)], indexing="ij"))
    k2 = (k * k).sum(0)
    s2 = (2 * np.pi * prm.regularisation_radius * max(g.dx)) ** 2 * k2
    zeta = (1 + 0.5 * s2) * np.exp(-0.5 * s2)   # order 4
    if all(per):
        # regularised only where the vorticity is formed too
        G = np.where(k2 > 0, (zeta if outputs else 1) / (4 * np.pi ** 2 * np.where(k2 > 0, k2, 1)), 0)
    else:
        G = O.green_real(g, prm).reshape(L, order="F")
        G = np.fft.fftn(np.fft.fftshift(G)) * g.dx[0] * g.dx[1] * g.dx[2]
    ik = 2j * np.pi * k
    vel = G * np.cross(ik, W, axis=0)
    psi = G * W
    vort = zeta * W + ik * (G * (ik * W).sum(0))
    out = []
    for f, want in ((vel, True), (vort, outputs), (psi, outputs)):
        if want:
            m = O.new_mesh(g)
            m[cut] = np.fft.ifftn(f, axes=(1, 2, 3)).real[:, :M[0], :M[1], :M[2]]
            for d in range(3):
                if per[d]:
                    a = np.moveaxis(m, d + 1, 0)
                    n, h = M[d], lo[d]
                    a[:h], a[h + n:] = a[n:n + h].copy(), a[h:2 * h].copy()
        out.append(m if want else None)
    return out


def _problem(n, bc):
    h = 1.0 / 16
    g = O.make_geom(n, 0, [-0.5 * h * v for v in n], h, bc)
    return g, O.make_params(4, 1, 2.0), blob_field(g, seed=sum(n))


@pytest.mark.parametrize("n,bc", [((5, 6, 7), FREE), ((20, 6, 5), FREE), ((8, 6, 5), MIXED), ((8, 6, 10), PER)])
@pytest.mark.parametrize("outputs", [False, True])
def test_reference(n, bc, outputs):
    g, prm, w = _problem(n, bc)
    ref = O.poisson_solve(g, prm, O.poisson_setup(g, prm), w, False, outputs, outputs)
    for a, b in zip(_reference(g, prm, w, outputs), ref):
        assert (a is None) == (b is None)
        assert a is None or rel_linf(a, b) < 1e-13


def _compare(n, bc, prec, outputs=False):
    g, prm, w = _problem(n, bc)
    p = pm.Patch(xmin=tuple(g.xmin), xmax=tuple(-v for v in g.xmin), ncell=n, dx=tuple(g.dx), bound_cond=bc, nghost=0)
    s = pm.PoissonSolver(p, prec, order=4, kernel=1, eps_radius=2.0, interp_order=3)
    s.setup()
    _check(s.solve(w, reproj=outputs, calc_vecpot=outputs), _reference(g, prm, w, outputs), prec)


def _box(axis, m):
    n = [5, 4, 6]
    n[axis] = m
    return tuple(n)


# transform lengths of the y and z passes (a free axis transforms 2 n)
EVEN = [1408, 1664, 2106, 2400, 2450, 2520, 2816, 3072, 3328, 3380, 3750, 3872, 3888, 4116, 4200]


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [pm.FP64, pm.FP32])
@pytest.mark.parametrize("L", EVEN)
@pytest.mark.parametrize("axis", [1, 2])
def test_free(axis, L, prec):
    _compare(_box(axis, L // 2), FREE, prec)


# a free x axis transforms n complex words; above 2720 only lengths whose three
# lines fit the run-time engine (the former kernel takes 3 L / 8 threads)
@pytest.mark.gpu
@pytest.mark.parametrize("prec", [pm.FP64, pm.FP32])
@pytest.mark.parametrize("L", [1408, 1875, 2106, 2400, 2401, 2450, 2520, 2625, 2816, 3125, 3328])
def test_free_x(L, prec):
    _compare(_box(0, L), FREE, prec)


# a periodic x axis transforms n / 2 complex words
@pytest.mark.gpu
@pytest.mark.parametrize("n,bc", [((6, 2106, 4), MIXED), ((6, 3750, 5), MIXED), ((3750, 6, 5), MIXED),
                                  ((4900, 6, 5), MIXED), ((6, 4, 1664), PER), ((6, 4, 3328), PER), ((6, 4, 3750), PER),
                                  ((6, 4, 4116), PER), ((4800, 4, 6), PER)])
def test_periodic(n, bc):
    _compare(n, bc, pm.FP64)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [(5, 4, 832), (4, 5, 1225), (5, 4, 1664), (4, 5, 2058)])
def test_all_outputs(n):
    _compare(n, FREE, pm.FP64, True)
