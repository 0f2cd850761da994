"""The deposition of large meshes when the particles fill a part of the mesh:
its y chunks and the order of its tiles follow how much of the mesh holds
particles, and its empty tiles are stored without a march.  Against the oracle
(FP64 1e-12 relative L-inf, FP32 1e-6 relative L2), independent of the chunks bit
for bit (particles of no strength elsewhere change the chunks and nothing near
the set), and in time: a small cube must not cost what the full mesh does."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import rel_l2, rel_linf

pytestmark = pytest.mark.gpu


def _cells(g, lo, hi, rng):
    """One particle in each cell of the index box [lo, hi), off its centre."""
    i = np.meshgrid(*[np.arange(a, b) for a, b in zip(lo, hi)], indexing="ij")
    c = np.stack([v.ravel(order="F") for v in i]).astype(float)
    return np.array(g.xmin)[:, None] + (c + 0.5 + rng.uniform(-0.4, 0.4, size=c.shape)) * np.array(g.dx)[:, None]


def _boxes(n):
    third = [v // 3 for v in n]
    return {
        "one": ([v // 2 for v in n], [v // 2 + 1 for v in n]),
        "cube": (third, [2 * v // 3 for v in n]),
        "corner": ([v - v // 4 for v in n], n),                          # the mesh's last tiles
        "slab": ([0, 0, n[2] // 2], [n[0], n[1], n[2] // 2 + 3]),
        "column": ([n[0] // 2, 0, n[2] // 2], [n[0] // 2 + 2, n[1], n[2] // 2 + 2]),
        "third": ([0, 0, 0], [n[0], n[1], n[2] // 3]),
        "more than half": ([0, 0, 0], [n[0], n[1], int(0.58 * n[2])]),
    }


def _deposit(pm, torch, patch, prec, io, pos, val, base, clear):
    dt = torch.float64 if prec == pm.FP64 else torch.float32
    mesh = torch.from_numpy(base.ravel(order="F")).cuda().to(dt)
    d_pos, d_val = [torch.from_numpy(np.ascontiguousarray(a.T).ravel()).cuda() for a in (pos, val)]
    pm.ParticleOps(patch, interp_order=io, precision=prec).p2m(d_pos.data_ptr(), d_val.data_ptr(), pos.shape[1],
                                                               mesh.data_ptr(), clear=clear)
    return mesh.double().cpu().numpy().reshape(base.shape, order="F")


@pytest.mark.parametrize("precision", [0, 1], ids=["f64", "f32"])
@pytest.mark.parametrize("n,ng,bc,io", [((96, 100, 94), 0, (0, 0, 0), 3), ((130, 66, 90), 1, (1, 0, 1), 3),
                                        ((70, 71, 92), 0, (0, 0, 0), 4)])
@pytest.mark.parametrize("box", ["one", "cube", "corner", "slab", "column", "third", "more than half"])
def test_partly_filled_mesh(n, ng, bc, io, precision, box):
    import torch
    import pmlib3d_amd as pm
    print("case", n, io, precision, box, flush=True)
    prec = (pm.FP64, pm.FP32)[precision]
    g = O.make_geom(n, ng, [-1.0, -0.5, -2.0], 1.0 / 16, bc, io)
    patch = pm.Patch(xmin=tuple(g.xmin), xmax=tuple(g.xmax), ncell=n, dx=tuple(g.dx), bound_cond=bc, nghost=ng)
    rng = np.random.default_rng(sum(n) + io + len(box))
    lo, hi = _boxes(n)[box]
    pos = _cells(g, lo, hi, rng)
    val = rng.normal(size=pos.shape)
    base = np.asfortranarray(rng.normal(size=(3,) + O.mesh_extent(g)).astype(np.float32).astype(np.float64))
    fpos, fval = np.asfortranarray(pos), np.asfortranarray(val)
    got = _deposit(pm, torch, patch, prec, io, pos, val, base, True)
    added = _deposit(pm, torch, patch, prec, io, pos, val, base, False)
    for a, ref in ((got, O.p2m(g, fpos, fval)), (added, O.p2m(g, fpos, fval, base.copy(order="F"), clear=False))):
        assert (rel_linf(a, ref) if precision == 0 else rel_l2(a, ref)) <= (1e-12 if precision == 0 else 1e-6)
    # particles of no strength in every cell: other chunks, the same sums
    more = _cells(g, [0, 0, 0], n, rng)
    full = _deposit(pm, torch, patch, prec, io, np.concatenate([pos, more], axis=1),
                    np.concatenate([val, np.zeros_like(more)], axis=1), base, True)
    assert np.array_equal(got, full)


def test_a_small_cube_costs_less_than_the_full_mesh():
    """2 % of the cells of 256^3: with chunks made for the full mesh half of its
    time (655 us of 1,310), a fifth with its own."""
    import torch
    import pmlib3d_amd as pm
    n, h = 256, 2.0 / 256
    patch = pm.Patch(xmin=(-1.0,) * 3, xmax=(1.0,) * 3, ncell=(n,) * 3, dx=(h,) * 3)
    ops = pm.ParticleOps(patch, interp_order=3, precision=pm.FP32)
    mesh = torch.zeros(3 * n ** 3, dtype=torch.float32, device="cuda:0")

    def time(a, b):
        c = -1.0 + (torch.arange(a, b, dtype=torch.float64, device="cuda:0") + 0.5) * h
        pos = torch.stack(torch.meshgrid(c, c, c, indexing="ij")[::-1], dim=-1).contiguous()
        val = torch.ones_like(pos)
        best = 1e9
        for _ in range(6):
            s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            s.record()
            ops.p2m(pos.data_ptr(), val.data_ptr(), (b - a) ** 3, mesh.data_ptr(), clear=True)
            e.record()
            torch.cuda.synchronize()
            best = min(best, s.elapsed_time(e))
        return best

    cube, full = time(93, 163), time(0, n)
    print("cube %.3f ms, full mesh %.3f ms" % (cube, full))
    assert cube <= 0.35 * full
