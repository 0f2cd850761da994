"""What a user of the framework has it do, case by case: inputs, one pass
through the public entry points, the work it cannot do without, and the
result in 64 bits by plain torch.

A case names its kind of call (`op`), the interior cells of its patch, its
boundary conditions, the precision of its meshes and the options in use:

  solve    one Poisson solve: velocity, and on request the stream function
           and the reprojected vorticity
  batch    the scalar solves of several small patches as one captured graph
  transfer particles to mesh and back (deposition, then gather)
  step     one remeshed vortex step, all arrays on the GPU
  graph    several recorded vortex steps on a small patch
  penal    penalisation_solve around a sphere
  refine   a refinement patch to its parent, and the parent to the patch

Meshes are flat tensors in the reference's layout (component fastest, then
x, y, z).  Outputs that an FP32 mesh produced are returned in 32 bits, also
where the particle arrays hold them in 64: after a remesh every strength and
velocity is a mesh value, so nothing is lost by that.
"""
import math

import numpy as np
import torch

import pmlib3d_amd as pm

DEV = "cuda:0"
FREE, MIXED, PERIODIC = "free", "mixed", "periodic"
BC = {FREE: (0, 0, 0), MIXED: (1, 1, 0), PERIODIC: (1, 1, 1)}


# ------------------------------------------------------------------- cases
def listed():
    return [
        # one small vortex ring, stream function and velocity: the interactive
        # and the validation size, where launches and latency count
        dict(name="ring-64-f64", op="solve", nx=64, ny=64, nz=64, bc=FREE, f32=False, ng=0, order=4, psi=True,
             reproj=False),
        # the headline solve: velocity of 256^3 cells, unbounded, FP32
        dict(name="solve-256-f32", op="solve", nx=256, ny=256, nz=256, bc=FREE, f32=True, ng=0, order=4, psi=False,
             reproj=False),
        # a ragged box with ghost layers and every output: reprojected
        # vorticity and stream function beside the velocity
        dict(name="solve-ragged-f64", op="solve", nx=156, ny=96, nz=121, bc=FREE, f32=False, ng=2, order=6, psi=True,
             reproj=True),
        # the wall-normal unbounded, otherwise periodic box of the turbulence runs
        dict(name="solve-mixed-384-f64", op="solve", nx=384, ny=384, nz=384, bc=MIXED, f32=False, ng=0, order=4,
             psi=False, reproj=False),
        # two dozen local patches of uneven sizes, one component each
        dict(name="batch-24-f32", op="batch", patches=24, shapes=4, f32=True, order=4),
        # M6* deposition and gather on a periodic box, an odd particle count
        dict(name="transfer-m6-f64", op="transfer", nx=112, ny=96, nz=80, bc=PERIODIC, f32=False, ng=0, m6=True,
             drop=133, jitter=0.1),
        # one step of the two-ring flow from its scattered initial set
        dict(name="step-128-f64", op="step", nx=128, ny=128, nz=128, bc=FREE, f32=False, ng=0, order=6, visc=0.0,
             rk=2, start="scattered"),
        # a viscous step in the running state (particles on the cell centres),
        # periodic sides with migration, stretching and diffusion
        dict(name="step-visc-160-f32", op="step", nx=160, ny=160, nz=156, bc=MIXED, f32=True, ng=2, order=4,
             visc=1e-3, rk=2, start="remeshed"),
        # a small flow as recorded steps without host synchronisation
        dict(name="graph-64-f32", op="graph", nx=64, ny=64, nz=64, bc=FREE, f32=True, ng=0, order=6, steps=4),
        # the flow past a sphere: penalisation iterations and solves
        dict(name="penal-252-f64", op="penal", nx=252, ny=252, nz=252, bc=FREE, f32=False, ng=2, order=4, iters=1000),
        # a refinement patch of 256^3 cells and its parent, both directions
        dict(name="refine-256-f32", op="refine", nx=256, ny=256, nz=256, bc=FREE, f32=True, ng=2, m6=False, ratio=2),
        # the large run: 56.6M particles, periodic x and y
        dict(name="step-384-f32", op="step", nx=384, ny=384, nz=384, bc=MIXED, f32=True, ng=0, order=4, visc=0.0,
             rk=2, start="remeshed"),
    ]


def _size(rng, lo, hi):
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return n + -n % rng.choice([1, 2, 4, 8, 16])


def _fitted(c):
    """The case with every axis cut to the next transform length the solver
    takes (factors up to 13, even)."""
    for d, k in enumerate(("nx", "ny", "nz")):
        free = BC[c["bc"]][d] == 0
        while True:
            n = 2 * (c[k] + 2 * c["ng"]) if free else c[k]
            for f in (2, 3, 5, 7, 11, 13):
                while n % f == 0:
                    n //= f
            if n == 1 and (free or c[k] % 2 == 0):
                break
            c[k] -= 1
    return c


def draw(rng):
    """One more case: sizes over the same ranges, the options of the kind."""
    op = rng.choice(["solve"] * 4 + ["batch"] + ["transfer"] * 2 + ["step"] * 3 + ["graph", "penal", "refine"])
    if op == "batch":
        return dict(op=op, patches=rng.randint(4, 24), shapes=rng.randint(5, 1000), f32=rng.random() < 0.5,
                    order=rng.choice([4, 6]))
    bc = rng.choice([FREE, FREE, MIXED, PERIODIC])
    hi = {"solve": 256, "transfer": 160, "step": 200, "graph": 96, "penal": 160, "refine": 192}[op]
    lo = 48 if op == "penal" else 32
    base = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    n = [_size(rng, 0.8 * base, 1.2 * base) for _ in range(3)]
    c = dict(op=op, nx=n[0], ny=n[1], nz=n[2], bc=bc, f32=rng.random() < 0.5, ng=rng.choice([0, 2]))
    if op == "solve":
        c.update(order=rng.choice([2, 4, 6, 8]), psi=rng.random() < 0.5, reproj=rng.random() < 0.4)
    elif op == "transfer":
        c.update(m6=rng.random() < 0.5, drop=rng.randint(1, 9999), jitter=rng.choice([0.0, 0.1, 0.4]))
        c["ng"] = rng.choice([0, 1, 3])
    elif op == "step":
        c.update(order=rng.choice([4, 6]), visc=rng.choice([0.0, 1e-3]), rk=rng.choice([1, 2, 3]),
                 start=rng.choice(["scattered", "remeshed"]))
        c["ng"] = 2 if c["visc"] else c["ng"]
    elif op == "graph":
        c.update(order=rng.choice([4, 6]), steps=rng.randint(1, 6))
    elif op == "penal":
        c.update(order=rng.choice([4, 6]), iters=rng.randint(2, 8), bc=FREE, ng=2)
    else:
        r = rng.choice([2, 4])
        c.update(m6=rng.random() < 0.5, ratio=r, ng=2, **{k: c[k] + -c[k] % (2 * r) for k in ("nx", "ny", "nz")})
    return c if op in ("transfer", "refine") else _fitted(c)


# ---------------------------------------------------------------- geometry
def _patch(c, **kw):
    n = (c["nx"], c["ny"], c["nz"])
    h = 2.0 / n[0]
    return pm.Patch(xmin=tuple(-0.5 * h * v for v in n), xmax=tuple(0.5 * h * v for v in n), ncell=n, dx=(h,) * 3,
                    bound_cond=BC[c["bc"]], nghost=c["ng"], **kw)


def _interp(c):
    return 4 if c.get("m6") else 3


def _dtype(c):
    return torch.float32 if c["f32"] else torch.float64


def _prec(c):
    return pm.FP32 if c["f32"] else pm.FP64


def _ghosts(p, io):
    return [p.nghost if b == 0 else (3 if io == 4 else 2) for b in p.bound_cond]


def _centres(p, ng):
    """Cell-centre coordinates per axis with ng[d] ghost cells a side."""
    return [p.xmin[d] + (torch.arange(-ng[d], p.ncell[d] + ng[d], dtype=torch.float64, device=DEV) + 0.5) * p.dx[d]
            for d in range(3)]


def _gen(seed):
    return np.random.default_rng(seed)


# ------------------------------------------------------------------ inputs
def _blobs(ax, h, rng, count=32):
    """(z, y, x, 3) field: Gaussian blobs of a few cells' width in the inner
    part of the box, normal strengths."""
    w = torch.zeros((len(ax[2]), len(ax[1]), len(ax[0]), 3), dtype=torch.float64, device=DEV)
    half = [float(a.abs().max()) for a in ax]
    for _ in range(count):
        c, s, amp = rng.uniform(-0.6, 0.6, 3) * half, rng.uniform(2, 6) * h, rng.normal(size=3)
        gx, gy, gz = [torch.exp(-(a - float(c[d])) ** 2 / (2 * s * s)) for d, a in enumerate(ax)]
        g = gz[:, None, None] * gy[None, :, None] * gx[None, None, :]
        for q in range(3):
            w[..., q].add_(g, alpha=float(amp[q]))
    return w


def _waves(p, ax, rng, count=12):
    """Solenoidal random Fourier modes, decaying towards free sides."""
    w = torch.zeros((len(ax[2]), len(ax[1]), len(ax[0]), 3), dtype=torch.float64, device=DEV)
    length = [p.xmax[d] - p.xmin[d] for d in range(3)]
    for _ in range(count):
        k = rng.integers(-8, 9, 3)
        k[0] = k[0] or 1
        kv = np.array([2 * math.pi * k[d] / length[d] for d in range(3)])
        a = np.cross(rng.normal(size=3), kv / np.linalg.norm(kv))
        ph = rng.uniform(0, 2 * math.pi)
        e = [torch.polar(torch.ones_like(x), float(kv[d]) * x) for d, x in enumerate(ax)]
        exy = e[1][:, None] * e[0][None, :] * complex(math.cos(ph), math.sin(ph))
        m = (e[2].real[:, None, None] * exy.real - e[2].imag[:, None, None] * exy.imag) * (8.0 / math.sqrt(count))
        for q in range(3):
            w[..., q].add_(m, alpha=float(a[q]))
    for d in range(3):
        if p.bound_cond[d] == 0:
            env = torch.exp(-(ax[d] / (0.15 * length[d])) ** 2)
            w *= env.view([-1 if 2 - d == i else 1 for i in range(3)] + [1])
    return w


def _rings(x, y, z, rng, scale):
    """Two coaxial Gaussian-core vortex rings at the points, (..., 3)."""
    out = torch.zeros(x.shape + (3,), dtype=torch.float64, device=DEV)
    rho, th = torch.sqrt(x * x + y * y), torch.atan2(y, x)
    for R, zc in ((0.4, 0.0), (0.5, 0.2)):
        R, zc, s = scale * (R + rng.uniform(-0.02, 0.02)), scale * zc, scale * 0.08
        wt = scale * scale / (math.pi * s * s) * torch.exp(-((rho - R) ** 2 + (z - zc) ** 2) / (s * s))
        out[..., 0] -= torch.sin(th) * wt
        out[..., 1] += torch.cos(th) * wt
    return out


def _field(p, c, seed, io):
    """Vorticity mesh (z, y, x, 3) with ghost cells, FP64."""
    ax = _centres(p, _ghosts(p, io))
    rng = _gen(seed)
    if c["bc"] == FREE and c["op"] in ("step", "graph"):
        Z, Y, X = torch.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
        return _rings(X, Y, Z, rng, min(-p.xmin[d] for d in range(3)))
    return _blobs(ax, p.dx[0], rng) if c["bc"] == FREE else _waves(p, ax, rng)


def _scattered(p, seed, jitter):
    """One particle per cell in (k, j, i) order: the centre, moved along by a
    smooth flow of up to half a cell and by a seeded jitter (in cells)."""
    ax, h = _centres(p, [0, 0, 0]), p.dx[0]
    Z, Y, X = torch.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    pos = torch.stack([X, Y, Z], dim=-1)
    pos += 0.5 * h * torch.stack([torch.sin(2 * Y) * torch.cos(3 * Z), torch.sin(3 * Z + 1) * torch.cos(2 * X),
                                  torch.sin(2 * X + 2) * torch.cos(3 * Y)], dim=-1)
    g = torch.Generator(device=DEV).manual_seed(seed)
    pos += jitter * h * (2 * torch.rand(pos.shape, dtype=torch.float64, device=DEV, generator=g) - 1)
    pos = pos.view(-1, 3)
    for d in range(3):
        length = p.xmax[d] - p.xmin[d]
        if p.bound_cond[d]:
            pos[:, d] = torch.remainder(pos[:, d] - p.xmin[d], length) + p.xmin[d]
        pos[:, d].clamp_(p.xmin[d], p.xmax[d] - 1e-9 * length)
    return pos


def _transfer_inputs(c, seed):
    p = _patch(c)
    pos = _scattered(p, seed, c["jitter"])
    pos = pos[:max(1, pos.shape[0] - c["drop"])].contiguous()
    g = torch.Generator(device=DEV).manual_seed(seed + 7)
    val = torch.randn(pos.shape, dtype=torch.float64, device=DEV, generator=g)
    mesh = torch.randn(3 * int(np.prod(pm.mesh_extent(p, _interp(c)))), dtype=torch.float64, device=DEV, generator=g)
    return p, pos, val, mesh.to(_dtype(c))


def _step_inputs(c, seed):
    """(patch, positions, strengths) of a step's particle set; positions None
    where it is seeded from the mesh, strengths then the mesh."""
    p = _patch(c)
    if c.get("start") == "remeshed":
        return p, None, _field(p, c, seed, 3).to(_dtype(c))
    pos = _scattered(p, seed, 0.1)
    if c["bc"] == FREE:
        w = _rings(pos[:, 0], pos[:, 1], pos[:, 2], _gen(seed), min(-v for v in p.xmin))
    else:
        w = _waves(p, _centres(p, [0, 0, 0]), _gen(seed)).reshape(-1, 3)
    return p, pos, w.contiguous()


def _threshold(w):
    return 1e-6 * float(w.abs().max())


def _shapes(c):
    rng = _gen(c["shapes"])
    return [tuple(int(v) for v in rng.choice([32, 48, 64, 96, 128, 160], 3)) for _ in range(c["patches"])]


def _batch_inputs(c, seed):
    h, rng, out = 1.0 / 128, _gen(seed), []
    for n in _shapes(c):
        p = pm.Patch(xmin=tuple(-v * h / 2 for v in n), xmax=tuple(v * h / 2 for v in n), ncell=n, dx=(h,) * 3)
        out.append((p, _blobs(_centres(p, [0, 0, 0]), h, rng, count=6)[..., 0].contiguous().to(_dtype(c))))
    return out


def _penal_inputs(c, seed):
    p = _patch(c)
    ax = _centres(p, _ghosts(p, 3))
    w = _blobs(ax, p.dx[0], _gen(seed))
    u = 0.05 * _blobs(ax, 3 * p.dx[0], _gen(seed + 1), count=8)
    u[..., 0] += 1.0
    Z, Y, X = torch.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    r = torch.sqrt(X * X + Y * Y + Z * Z)
    a = 1e4 * 0.5 * p.dx[0] * 0.5 * (1.0 - torch.tanh((r - 0.25) / (2.0 * p.dx[0])))
    dt = _dtype(c)
    return p, (a / (1.0 + a)).to(dt), u.to(dt), w.to(dt)


PENAL = dict(relaxation=1.0, tolerance=0.01, fd_order=4, vel_inf=(1.0, 0.0, 0.0), reproject=True)


def _refine_inputs(c, seed):
    p = _patch(c, level=1 + int(math.log2(c["ratio"])), parent=(1, 0))
    io, g = _interp(c), torch.Generator(device=DEV).manual_seed(seed)
    parent = pm.pmlib_topology_parent(p, interp_order=io)
    fine, coarse = [torch.randn(3 * int(np.prod(pm.mesh_extent(q, io))), dtype=torch.float64, device=DEV, generator=g)
                    .to(_dtype(c)) for q in (p, parent)]
    return p, parent, fine, coarse


# ----------------------------------------------------------------- prepare
class _Owned:
    """A view of `count` FP64 numbers of device memory that a handle owns,
    good for as long as the handle lives."""

    def __init__(self, address, count):
        self.__cuda_array_interface__ = dict(shape=(count,), typestr="<f8", data=(address, False), version=3)


def _solver(p, c, io=3):
    s = pm.PoissonSolver(p, _prec(c), order=c["order"], kernel=1, eps_radius=2.0, interp_order=io)
    s.setup()
    return s


def prepare(case, seed):
    c, op = case, case["op"]
    s = dict(case=c)
    if op == "solve":
        p = _patch(c)
        s.update(solver=_solver(p, c), w=_field(p, c, seed, 3).to(_dtype(c)).view(-1))
        for k, want in (("vel", True), ("psi", c["psi"]), ("vort", c["reproj"])):
            s[k] = torch.zeros_like(s["w"]) if want else None
    elif op == "batch":
        inputs = _batch_inputs(c, seed)
        s.update(solvers=[_solver(p, c) for p, _ in inputs], w=[w for _, w in inputs])
        s["psi"] = [torch.zeros_like(w) for w in s["w"]]
        s["batch"] = pm.PoissonBatch(s["solvers"])
    elif op == "transfer":
        p, s["pos"], s["val"], s["field"] = _transfer_inputs(c, seed)
        s.update(ops=pm.ParticleOps(p, _interp(c), _prec(c)), mesh=torch.zeros_like(s["field"]),
                 out=torch.zeros_like(s["pos"]))
    elif op in ("step", "graph"):
        p, pos, w = _step_inputs(c, seed)
        kw = dict(order=c["order"], eps_radius=2.0, interp_order=3, precision=_prec(c))
        s.update(pos=pos if pos is None else pos.view(-1), w=w.view(-1), count=0 if pos is None else pos.shape[0],
                 dt=0.5 * p.dx[0], cut=_threshold(w))
        if op == "step":
            s["step"] = pm.VortexStep(p, rk_order=c["rk"], visc=c["visc"] or None, **kw)
        else:
            s["step"] = pm.GraphVortexStep(p, rk_order=2, **kw)
    elif op == "penal":
        p, s["chi"], u, w = _penal_inputs(c, seed)
        s.update(solver=_solver(p, c), u=u.view(-1), w=w.view(-1), dt=0.5 * p.dx[0])
        s.update(vel=torch.zeros_like(s["u"]), vort=torch.zeros_like(s["w"]))
    else:
        s["patch"], s["parent"], s["fine"], s["coarse"] = _refine_inputs(c, seed)
        s.update(to_parent=torch.zeros_like(s["coarse"]), to_patch=torch.zeros_like(s["fine"]))
    return s


# --------------------------------------------------------------------- run
def _ptr(t):
    return None if t is None else t.data_ptr()


def _particles(n, pos, vort, vel, c):
    """A copy of the n remeshed particles for the caller's program, in arrays
    of one row a cell (a handle's own arrays end with the handle)."""
    rows = 3 * c["nx"] * c["ny"] * c["nz"]
    out = {"pos": pos, "vort": vort, "vel": vel}
    for k, a in out.items():
        out[k] = torch.zeros(rows, dtype=torch.float64 if k == "pos" else _dtype(c), device=DEV)
        out[k][:3 * n] = a[:3 * n]
    return out


def run(s):
    c, op = s["case"], s["case"]["op"]
    if op == "solve":
        s["solver"].solve_device(_ptr(s["w"]), _ptr(s["vel"]), _ptr(s["vort"]), _ptr(s["psi"]), reproj=c["reproj"],
                                 calc_vecpot=c["psi"])
        return {k: s[k] for k in ("vel", "psi", "vort") if s[k] is not None}
    if op == "batch":
        s["batch"].solve_scalar([_ptr(w) for w in s["w"]], [_ptr(f) for f in s["psi"]])
        return s["psi"]
    if op == "transfer":
        n = s["pos"].shape[0]
        s["ops"].p2m(_ptr(s["pos"]), _ptr(s["val"]), n, _ptr(s["mesh"]), clear=True)
        s["ops"].m2p(_ptr(s["field"]), _ptr(s["pos"]), n, _ptr(s["out"]))
        return {"mesh": s["mesh"], "part": s["out"].to(s["mesh"].dtype)}
    if op == "step":
        st = s["step"]
        if s["pos"] is None:
            st.seed_from_mesh(_ptr(s["w"]), s["cut"])
        else:
            st.load_device(s["pos"], s["w"], s["count"])
        st.step(s["dt"], s["cut"])
        return dict(_particles(st.np, *[st.arrays[k] for k in ("pos", "vort", "vel")], c), n=st.np)
    if op == "graph":
        st = s["step"]
        st.load_device(s["pos"], s["w"], s["count"])
        for _ in range(c["steps"]):
            st.step(s["dt"], s["cut"])
        n, status = st.sync()
        pos, vel, vort = [torch.as_tensor(_Owned(st.ptrs[i], 3 * n), device=DEV) for i in range(3)]
        return dict(_particles(n, pos, vort, vel, c), n=n, status=status)
    if op == "penal":
        s["vel"].copy_(s["u"])
        s["vort"].copy_(s["w"])
        force, count, residual = pm.penalisation_solve_device(
            s["solver"], _ptr(s["chi"]), _ptr(s["vel"]), _ptr(s["vort"]), max_iter=c["iters"], dtime=s["dt"], **PENAL)
        real = np.float32 if c["f32"] else np.float64
        return {"vel": s["vel"], "vort": s["vort"], "iterations": count, "force": force.astype(real)}
    io, prec = _interp(c), _prec(c)
    pm.interp_mesh_mesh_device(s["patch"], s["parent"], prec, _ptr(s["fine"]), _ptr(s["to_parent"]), clear=True,
                               interp_order=io)
    pm.interp_mesh_mesh_device(s["parent"], s["patch"], prec, _ptr(s["coarse"]), _ptr(s["to_patch"]), clear=True,
                               interp_order=io)
    return {"parent": s["to_parent"], "patch": s["to_patch"]}


# -------------------------------------------------------------------- work
def _solve_flops(M, L, cin, cout):
    """Real operations of the pruned transforms (5/2 n log2 n a real line)."""
    f = lambda n: 2.5 * n * math.log2(n)  # noqa: E731
    lines = [M[1] * M[2], 2 * (L[0] // 2 + 1) * M[2], 2 * (L[0] // 2 + 1) * L[1]]
    return (cin + cout) * sum(lines[d] * f(L[d]) for d in range(3))


def _dims(p):
    M = [p.ncell[d] + (0 if p.bound_cond[d] else 2 * p.nghost) for d in range(3)]
    return M, [m if b else 2 * m for m, b in zip(M, p.bound_cond)]


def work(case):
    c, op = case, case["op"]
    size = 4 if c["f32"] else 8
    if op == "batch":
        every = [([v for v in n], [2 * v for v in n]) for n in _shapes(c)]
        return dict(bytes=sum(2 * size * float(np.prod(M)) for M, _ in every),
                    flops=sum(_solve_flops(M, L, 1, 1) for M, L in every))
    io = _interp(c)
    p = _patch(c)
    M, L = _dims(p)
    cells, inner = float(np.prod(pm.mesh_extent(p, io))), float(np.prod(p.ncell))
    taps = 216 if io == 4 else 64
    solve = _solve_flops(M, L, 3, 3)
    if op == "solve":
        outs = 1 + c["psi"] + c["reproj"]
        return dict(bytes=3 * (1 + outs) * size * cells, flops=_solve_flops(M, L, 3, 3 * outs))
    if op == "transfer":
        n = max(1.0, inner - c["drop"])
        return dict(bytes=n * 96 + 6 * size * cells, flops=n * taps * 14)
    if op in ("step", "graph"):
        # per stage: deposition, solve, gather, update; then deposition and remesh
        stages, steps = (c["rk"], 1) if op == "step" else (2, c["steps"])
        stage = inner * (48 + 24 + 24 + 24 * 5) + 9 * size * cells
        rhs = c.get("visc", 0.0) != 0.0
        stage += (9 * size * cells + 24 * 4 * inner) if rhs else 0
        flops = inner * taps * (14 + (7 if rhs else 0)) + solve
        end = inner * (48 + 24 * 4) + 6 * size * cells
        return dict(bytes=steps * (stages * stage + end), flops=steps * (stages * flops + inner * taps * 7))
    if op == "penal":
        # about ten iterations to the tolerance, each a curl and a solve, and the final solve
        k = min(c["iters"], 10)
        return dict(bytes=(k * (13 + 6) + 15) * size * cells, flops=(k + 1) * solve)
    coarse = cells / c["ratio"] ** 3
    return dict(bytes=6 * size * (cells + coarse), flops=6 * cells * (5 if io == 4 else 3) * 4)


# ------------------------------------------------- the result in 64 bits
def _axes(t, d, vals):
    return vals.view([-1 if 2 - d == i else 1 for i in range(3)])


def _green(p, order, eps):
    """The regularised kernel on the transform grid, origin first, summed
    over the nearest periodic images, as (z, y, x)."""
    M, L = _dims(p)
    ax = []
    for d in range(3):
        i = torch.arange(L[d], dtype=torch.float64, device=DEV)
        ax.append(torch.where(i < L[d] / 2, i, i - L[d]) * p.dx[d])
    G = torch.zeros(L[2], L[1], L[0], dtype=torch.float64, device=DEV)
    b = p.bound_cond
    poly = {2: [0.0], 4: [1.0], 6: [1.75, -0.25], 8: [2.375, -2.0 / 3.0, 1.0 / 24.0]}[order]
    at0 = {2: 1.0, 4: 1.5, 6: 1.875, 8: 2.1875}[order] * math.sqrt(2.0) / (4.0 * math.pi ** 1.5 * eps)
    for kk in range(-b[2], b[2] + 1):
        for jj in range(-b[1], b[1] + 1):
            for ii in range(-b[0], b[0] + 1):
                x, y, z = [_axes(G, d, ax[d] + s * L[d] * p.dx[d]) for d, s in enumerate((ii, jj, kk))]
                r = torch.sqrt(x * x + y * y + z * z)
                rho = r / eps
                q = sum(a * rho ** (2 * n + 1) for n, a in enumerate(poly))
                v = q * torch.exp(-0.5 * rho * rho) / math.sqrt(2.0 * math.pi) + torch.erf(rho / math.sqrt(2.0))
                G += torch.where(r == 0, torch.full_like(r, at0), v / (4.0 * math.pi * r))
    return G


def _fill_ghosts(m, p, ng):
    for d in range(3):
        if p.bound_cond[d]:
            t, n, g = m.transpose(0, 2 - d), p.ncell[d], ng[d]
            t[:g] = t[n:n + g].clone()
            t[g + n:] = t[g:2 * g].clone()
    return m


def _exact_solve(p, order, w, io=3, psi=False, reproj=False, scalar=False, cache=None):
    """(velocity, stream function, reprojected vorticity) of the mesh w
    (z, y, x, component), FP64."""
    M, L = _dims(p)
    ng = _ghosts(p, io)
    lo = [ng[d] if p.bound_cond[d] else 0 for d in range(3)]
    inner = tuple(slice(lo[2 - i], lo[2 - i] + M[2 - i]) for i in range(3))
    eps = 2.0 * max(p.dx)
    k = []
    for d in range(3):
        i = torch.arange(L[d], dtype=torch.float64, device=DEV)
        k.append(_axes(None, d, torch.where(i < L[d] // 2, i, i - L[d]) / (L[d] * p.dx[d])))
    k2 = k[0] ** 2 + k[1] ** 2 + k[2] ** 2
    zeta = None
    if reproj:
        s2 = (2.0 * math.pi * eps) ** 2 * k2
        zeta = sum(a * s2 ** n for n, a in enumerate([1.0, 0.5, 0.125, 1.0 / 48.0][:order // 2])) * torch.exp(-0.5 * s2)
    if cache is not None and "G" in cache:
        G = cache["G"]
    else:
        if all(p.bound_cond):
            G = (1.0 if zeta is None else zeta) / (4.0 * math.pi ** 2 * torch.where(k2 > 0, k2, torch.ones_like(k2)))
            G[0, 0, 0] = 0.0
        else:
            G = torch.fft.fftn(_green(p, order, eps)) * (p.dx[0] * p.dx[1] * p.dx[2])
        if cache is not None:
            cache["G"] = G
    f = [torch.fft.fftn(w[..., q][inner], s=(L[2], L[1], L[0])) for q in range(w.shape[-1])]

    def back(a):
        return torch.fft.ifftn(a).real[:M[2], :M[1], :M[0]]

    def mesh(parts):
        out = torch.zeros_like(w)
        for q, a in enumerate(parts):
            out[..., q][inner] = back(a)
        return _fill_ghosts(out, p, ng)

    if scalar:
        return mesh([G * f[0]])
    t = 2.0j * math.pi * G
    vel = mesh(t * (k[(q + 1) % 3] * f[(q + 2) % 3] - k[(q + 2) % 3] * f[(q + 1) % 3]) for q in range(3))
    pot = mesh(G * f[q] for q in range(3)) if psi else None
    vort = None
    if reproj:
        div = t * (k[0] * f[0] + k[1] * f[1] + k[2] * f[2])
        vort = mesh(zeta * f[q] + 2.0j * math.pi * k[q] * div for q in range(3))
    return vel, pot, vort


def _weight(io, x):
    x = x.abs()
    if io == 3:
        near = 1.0 - 2.5 * x ** 2 + 1.5 * x ** 3
        return torch.where(x < 1, near, torch.where(x < 2, 0.5 * (2 - x) ** 2 * (1 - x), torch.zeros_like(x)))
    a = -1.0 / 12.0 * (x - 1) * (25 * x ** 4 - 38 * x ** 3 - 3 * x ** 2 + 12 * x + 12)
    b = 1.0 / 24.0 * (x - 1) * (x - 2) * (25 * x ** 3 - 114 * x ** 2 + 153 * x - 48)
    c = -1.0 / 24.0 * (x - 2) * (x - 3) ** 3 * (5 * x - 8)
    zero = torch.zeros_like(x)
    return torch.where(x < 1, a, torch.where(x < 2, b, torch.where(x < 3, c, zero)))


def _taps(p, io, pos):
    """Per axis and stencil slot: mesh index (ghosts included) and weight,
    zero and clamped outside the mesh."""
    ns, ng, out = (6 if io == 4 else 4), _ghosts(p, io), []
    for d in range(3):
        t = (pos[:, d] - p.xmin[d]) / p.dx[d] - 0.5
        base, E, axis = torch.floor(t), p.ncell[d] + 2 * ng[d], []
        for s in range(ns):
            i = base + (s - ns // 2 + 1)
            ok = (i >= -ng[d]) & (i < p.ncell[d] + ng[d])
            axis.append(((i + ng[d]).clamp(0, E - 1).long(), torch.where(ok, _weight(io, t - i), torch.zeros_like(t))))
        out.append(axis)
    return out


def _exact_p2m(p, io, pos, val):
    E = pm.mesh_extent(p, io)
    mesh = torch.zeros(E[2] * E[1] * E[0], 3, dtype=torch.float64, device=DEV)
    X, Y, Z = _taps(p, io, pos)
    for iz, wz in Z:
        for iy, wy in Y:
            for ix, wx in X:
                mesh.index_add_(0, (iz * E[1] + iy) * E[0] + ix, (wx * wy * wz)[:, None] * val)
    mesh = mesh.view(E[2], E[1], E[0], 3)
    ng = _ghosts(p, io)
    for d in range(3):
        if p.bound_cond[d]:
            t, n, g = mesh.transpose(0, 2 - d), p.ncell[d], ng[d]
            both = t[:2 * g] + t[n:n + 2 * g]
            t[:2 * g] = both
            t[n:n + 2 * g] = both
    return mesh


def _exact_m2p(p, io, mesh, pos):
    E, out = pm.mesh_extent(p, io), torch.zeros_like(pos)
    flat = mesh.reshape(-1, 3)
    X, Y, Z = _taps(p, io, pos)
    for iz, wz in Z:
        for iy, wy in Y:
            for ix, wx in X:
                out += (wx * wy * wz)[:, None] * flat[(iz * E[1] + iy) * E[0] + ix]
    return out


def _diff(a, axis, h, second=False):
    """4th-order central differences along axis (edges meaningless)."""
    m2, m1, p1, p2 = [torch.roll(a, s, axis) for s in (2, 1, -1, -2)]
    if second:
        return (-(m2 + p2) / 12.0 + 4.0 / 3.0 * (m1 + p1) - 2.5 * a) / (h * h)
    return ((m2 - p2) / 6.0 + 4.0 / 3.0 * (p1 - m1)) / (2.0 * h)


def _exact_rhs(p, w, u, visc):
    ng = _ghosts(p, 3)
    out = torch.zeros_like(w)
    full = sum(visc * _diff(w, 2 - d, p.dx[d], True) + w[..., d:d + 1] * _diff(u, 2 - d, p.dx[d]) for d in range(3))
    i = tuple(slice(ng[2 - a], ng[2 - a] + p.ncell[2 - a]) for a in range(3))
    out[i] = full[i]
    return _fill_ghosts(out, p, ng)


def _exact_step(p, c, pos, w, dt, cut, rk, visc, cache):
    """One remeshed step from the particle set (pos, w): the new set."""
    A = {1: [0.0], 2: [0.0, -0.5], 3: [0.0, -5.0 / 9.0, -153.0 / 128.0]}[rk]
    C = {1: [1.0], 2: [0.5, 1.0], 3: [1.0 / 3.0, 15.0 / 16.0, 8.0 / 15.0]}[rk]
    pos, w, vr, dr = pos.clone(), w.clone(), torch.zeros_like(pos), torch.zeros_like(pos)
    u = None
    for a, b in zip(A, C):
        m = _exact_p2m(p, 3, pos, w)
        u = _exact_solve(p, c["order"], m, cache=cache)[0]
        vr = a * vr + dt * _exact_m2p(p, 3, u, pos)
        if visc:
            dr = a * dr + dt * _exact_m2p(p, 3, _exact_rhs(p, m, u, visc), pos)
            w += b * dr
        pos += b * vr
        keep = torch.ones(pos.shape[0], dtype=torch.bool, device=DEV)
        for d in range(3):
            length = p.xmax[d] - p.xmin[d]
            if p.bound_cond[d]:
                pos[:, d] -= length * torch.floor((pos[:, d] - p.xmin[d]) / length)
            else:
                keep &= (pos[:, d] >= p.xmin[d]) & (pos[:, d] < p.xmax[d])
        pos, w, vr, dr = pos[keep], w[keep], vr[keep], dr[keep]
    return _exact_remesh(p, _exact_p2m(p, 3, pos, w), u, cut)


def _exact_remesh(p, m, u, cut):
    ng = _ghosts(p, 3)
    i = tuple(slice(ng[2 - a], ng[2 - a] + p.ncell[2 - a]) for a in range(3))
    m, u = m[i].reshape(-1, 3), (u[i].reshape(-1, 3) if u is not None else None)
    keep = (m * m).sum(-1).sqrt() > cut
    ax = _centres(p, [0, 0, 0])
    Z, Y, X = torch.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    return torch.stack([X, Y, Z], -1).view(-1, 3)[keep], m[keep], (u[keep] if u is not None else None)


def _exact_penal(c, seed):
    p, chi, u, w = _penal_inputs(c, seed)
    chi, u, w = chi.double(), u.double(), w.double()
    cache, h, ng = {}, p.dx[0], 2
    ins = (slice(ng, -ng),) * 3
    vp, vort, up = -u, torch.zeros_like(w), torch.zeros_like(u)
    ax = _centres(p, [0, 0, 0])
    Z, Y, X = torch.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    x = torch.stack([X, Y, Z], -1)
    force, residual, count = torch.zeros(3, dtype=torch.float64, device=DEV), 0.0, 0
    while count == 0 or (residual > PENAL["tolerance"] and count < c["iters"]):
        count += 1
        f = chi[..., None] * (vp - up)
        dd = lambda q, d: _diff(f[..., q], 2 - d, h)[ins]  # noqa: E731
        curl = torch.stack([dd(2, 1) - dd(1, 2), dd(0, 2) - dd(2, 0), dd(1, 0) - dd(0, 1)], -1)
        vort[ins] += curl
        up = _exact_solve(p, c["order"], vort, cache=cache)[0]
        df = -torch.linalg.cross(x, curl).sum((0, 1, 2)) * h ** 3 / (0.5 * h)
        force = force + df
        residual = float(df.norm() / force.norm())
    vel, _, new = _exact_solve(p, c["order"], w + vort, reproj=True, cache=cache)
    vel[..., 0] += 1.0
    return {"vel": vel.view(-1), "vort": new.view(-1), "iterations": None, "force": force}


def exact(case, seed):
    c, op = case, case["op"]
    if op == "solve":
        p = _patch(c)
        w = _field(p, c, seed, 3).to(_dtype(c)).double()
        vel, pot, vort = _exact_solve(p, c["order"], w, psi=c["psi"], reproj=c["reproj"])
        return {k: v.view(-1) for k, v in (("vel", vel), ("psi", pot), ("vort", vort)) if v is not None}
    if op == "batch":
        return [_exact_solve(p, c["order"], w.double()[..., None], scalar=True)[..., 0] for p, w in _batch_inputs(c, seed)]
    io = _interp(c)
    if op == "transfer":
        p, pos, val, field = _transfer_inputs(c, seed)
        E = pm.mesh_extent(p, io)
        return {"mesh": _exact_p2m(p, io, pos, val).view(-1),
                "part": _exact_m2p(p, io, field.double().view(E[2], E[1], E[0], 3), pos)}
    if op in ("step", "graph"):
        if c["nx"] * c["ny"] * c["nz"] > 9_000_000:
            return None   # minutes of plain torch
        p, pos, w = _step_inputs(c, seed)
        cut, cache, dt, u = _threshold(w), {}, 0.5 * p.dx[0], None
        if pos is None:
            pos, w, _ = _exact_remesh(p, w.double(), None, cut)
        for _ in range(c.get("steps", 1)):
            pos, w, u = _exact_step(p, c, pos, w, dt, cut, c.get("rk", 2), c.get("visc", 0.0), cache)
        out = {k: torch.zeros(3 * c["nx"] * c["ny"] * c["nz"], dtype=torch.float64, device=DEV)
               for k in ("pos", "vort", "vel")}
        for k, a in (("pos", pos), ("vort", w), ("vel", u)):
            out[k][:a.numel()] = a.reshape(-1)
        return out
    if op == "penal":
        return _exact_penal(c, seed)
    p, parent, fine, coarse = _refine_inputs(c, seed)
    centres = _centres(p, _ghosts(p, io))
    Z, Y, X = torch.meshgrid(centres[2], centres[1], centres[0], indexing="ij")
    x = torch.stack([X, Y, Z], -1).view(-1, 3)
    inside = torch.ones(x.shape[0], dtype=torch.bool, device=DEV)
    for d in range(3):
        if p.bound_cond[d]:
            inside &= (x[:, d] >= p.xmin[d]) & (x[:, d] <= p.xmax[d])
    val = fine.double().view(-1, 3) * inside[:, None] / c["ratio"] ** 3
    E = pm.mesh_extent(parent, io)
    to_patch = _exact_m2p(parent, io, coarse.double().view(E[2], E[1], E[0], 3), x)
    Ef = pm.mesh_extent(p, io)
    to_patch = _fill_ghosts(to_patch.view(Ef[2], Ef[1], Ef[0], 3), p, _ghosts(p, io))
    return {"parent": _exact_p2m(parent, io, x, val).view(-1), "patch": to_patch.reshape(-1)}
