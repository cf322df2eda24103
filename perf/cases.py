"""The work that a user of this framework has it do, as measurable cases.

Three kinds, each through the public entry points of the library:

``solve``  one pressure-Poisson solve (``Multigrid.solve_device``) from a zero
           initial guess on device arrays in the caller's layout;
``step``   one time step of a flow (``saras_nse_set_fields``, ``_step``,
           ``_get_fields`` on device arrays), as a driver that owns its fields
           has ``timeAdvance`` do it;
``serve``  a batch of Poisson requests of mixed sizes through the request loop
           (``Server.submit`` / ``poll``), on host arrays by its nature.

Sizes, options and tolerances are those of the benchmark, the serving stream
and the validation decks of this repository.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "saras-cc_amd"))

import saras_amd as S  # noqa: E402
from saras_amd import serving  # noqa: E402


def listed():
    return [
        # the smallest request of the serving stream: a 2-D square of 64 cells
        # with Dirichlet walls, plain FP64; latency alone counts
        dict(name="solve_2d_64_fp64", kind="solve", dim=2, nx=64, ny=1, nz=64, walls="dirichlet", fp64=True,
             nu=2, tol=1e-8, coarse_tol=1e-10, inner=10, modes=8),
        # a large 2-D request of that stream, periodic, mixed precision
        dict(name="solve_2d_1024_mixed", kind="solve", dim=2, nx=1024, ny=1, nz=1024, walls="periodic", fp64=False,
             nu=2, tol=1e-8, coarse_tol=1e-10, inner=10, modes=8),
        # an ordinary 3-D request of that stream: 112 = 16 * 7 cells with walls
        # keep a coarsest level of 14 cells per axis
        dict(name="solve_3d_112_mixed", kind="solve", dim=3, nx=112, ny=112, nz=112, walls="neumann", fp64=False,
             nu=2, tol=1e-8, coarse_tol=1e-10, inner=10, modes=8),
        # a box of three different extents, Dirichlet walls, plain FP64
        dict(name="solve_3d_box_fp64", kind="solve", dim=3, nx=160, ny=64, nz=96, walls="dirichlet", fp64=True,
             nu=2, tol=1e-8, coarse_tol=1e-10, inner=10, modes=8),
        # the benchmark's headline: 256^3 periodic, 64 Fourier modes, to 1e-10
        dict(name="solve_3d_256_mixed", kind="solve", dim=3, nx=256, ny=256, nz=256, walls="periodic", fp64=False,
             nu=2, tol=1e-10, coarse_tol=1e-2, inner=4, modes=64),
        # the same problem by the plain FP64 path, the reference's arithmetic
        dict(name="solve_3d_256_fp64", kind="solve", dim=3, nx=256, ny=256, nz=256, walls="periodic", fp64=True,
             nu=2, tol=1e-10, coarse_tol=1e-2, inner=4, modes=64),
        # the largest solve of the benchmark
        dict(name="solve_3d_512_mixed", kind="solve", dim=3, nx=512, ny=512, nz=512, walls="periodic", fp64=False,
             nu=2, tol=1e-10, coarse_tol=1e-2, inner=4, modes=64),
        # the lid-driven cavity of the validation deck (2-D, 128 x 128, tanh
        # grids, Euler-CN, central differences, V(3,3) FP64 pressure cycles):
        # tens of thousands of such steps make a run
        dict(name="step_cavity_128", kind="step", flow="cavity", nx=128, ny=1, nz=128, fp64=True),
        # a small channel (constant pressure gradient, no-slip z walls, RK3,
        # upwind second-order scheme) of ragged extents, FP64 throughout
        dict(name="step_channel_ragged", kind="step", flow="channel", nx=72, ny=56, nz=100, fp64=True),
        # the benchmark's Rayleigh-Benard step: 256^3, tanh z, fourth-order
        # Morinishi, V(3,6) pressure cycles in mixed precision
        dict(name="step_convection_256", kind="step", flow="convection", nx=256, ny=256, nz=256, fp64=False),
        # the benchmark's large-eddy step: 384^3 Taylor-Green box with the
        # spiral sub-grid model, in its deck's precision recipe
        dict(name="step_les_384", kind="step", flow="les", nx=384, ny=384, nz=384, fp64=False),
        # the request loop: 32 requests of the serving stream at once
        dict(name="serve_32", kind="serve", count=32, mix=4, n3_hi=128, n2_hi=1024, fp64=False),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _friendly(rng, lo, hi):
    return serving.nearest_extent(_log(rng, lo, hi), lo, hi)


def _box(rng, axes, lo, hi):
    """Extents q 2^m of one m, q from 2 to 7: a box that coarsens to a few
    cells per axis, as the serving stream's extents do."""
    m = rng.choice([m for m in range(4, 9) if 2 << m >= lo // 2 and 4 << m <= hi])
    out = []
    while len(out) < axes:
        n = rng.randint(2, 7) << m
        if lo <= n <= hi:
            out.append(n)
    return out


def _tol(rng):
    return float("%.1e" % 10.0 ** -rng.uniform(5.0, 8.5))


def draw(rng):
    what = rng.choice(["solve2", "solve3", "solve3", "cavity", "channel", "convection", "les", "serve"])
    if what == "solve2":
        nx, nz = _box(rng, 2, 64, 2048)
        return dict(kind="solve", dim=2, nx=nx, ny=1, nz=nz,
                    walls=rng.choice(serving.KINDS), fp64=rng.random() < 0.5, nu=rng.choice([2, 2, 3]),
                    tol=_tol(rng), coarse_tol=1e-10, inner=10, modes=rng.choice([8, 8, 32]))
    if what == "solve3":
        nx, ny, nz = _box(rng, 3, 32, 320)
        return dict(kind="solve", dim=3, nx=nx, ny=ny, nz=nz, walls=rng.choice(serving.KINDS), fp64=rng.random() < 0.5,
                    nu=rng.choice([2, 2, 3]), tol=_tol(rng), coarse_tol=1e-10, inner=10,
                    modes=rng.choice([8, 8, 32]))
    if what == "cavity":
        return dict(kind="step", flow="cavity", nx=_friendly(rng, 64, 512), ny=1, nz=_friendly(rng, 64, 512), fp64=True)
    if what == "channel":
        return dict(kind="step", flow="channel", nx=4 * round(_log(rng, 10, 40)), ny=4 * round(_log(rng, 10, 40)),
                    nz=4 * round(_log(rng, 10, 40)), fp64=True)
    if what == "convection":
        return dict(kind="step", flow="convection", nx=_friendly(rng, 48, 320), ny=_friendly(rng, 48, 320),
                    nz=_friendly(rng, 48, 256), fp64=rng.random() < 0.5)
    if what == "les":
        n = _friendly(rng, 48, 320)
        return dict(kind="step", flow="les", nx=n, ny=n, nz=n, fp64=rng.random() < 0.3)
    return dict(kind="serve", count=rng.randint(8, 48), mix=rng.randint(0, 10 ** 6), n3_hi=rng.choice([64, 96, 128]),
                n2_hi=rng.choice([256, 512, 1024]), fp64=rng.random() < 0.3)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _lengths(c):
    """Cells of equal size: the longest axis has unit length."""
    m = max(c["nx"], c["ny"], c["nz"])
    return c["nx"] / m, c["ny"] / m, c["nz"] / m


def _solve_rhs(c, seed):
    """A sum of separable modes on the cell centres (sines for Dirichlet
    walls, cosines for Neumann ones, complex exponentials for a periodic box)
    with amplitudes ~ U(0.5, 1) |k|^-2, zero mean unless Dirichlet."""
    rng = np.random.default_rng(seed)
    n = [c["nx"], c["ny"], c["nz"]] if c["dim"] == 3 else [c["nx"], c["nz"]]
    kmax = 16 if c["modes"] > 8 else (4 if c["walls"] == "periodic" else 8)
    x = [(np.arange(m) + 0.5) / m for m in n]
    first, rest = [], []
    for _ in range(c["modes"]):
        while True:
            if c["walls"] == "periodic":
                k = rng.integers(-kmax, kmax + 1, len(n))
            else:
                k = rng.integers(1 if c["walls"] == "dirichlet" else 0, kmax + 1, len(n))
            if np.abs(k).max() >= 1:
                break
        amp = rng.uniform(0.5, 1.0) / float(k @ k)
        phase = np.exp(2j * np.pi * rng.uniform())
        if c["walls"] == "periodic":
            f = [np.exp(2j * np.pi * kk * xx) for kk, xx in zip(k, x)]
            f[0] = f[0] * phase
        else:
            g = np.sin if c["walls"] == "dirichlet" else np.cos
            f = [g(np.pi * kk * xx).astype(complex) for kk, xx in zip(k, x)]
        first += [amp * f[0].real, -amp * f[0].imag]
        tail = f[1] if len(n) == 2 else np.outer(f[1], f[2]).ravel()
        rest += [tail.real, tail.imag]
    a = torch.tensor(np.array(first), device="cuda").t().contiguous()
    core = (a @ torch.tensor(np.array(rest), device="cuda")).reshape(n)
    if c["walls"] != "dirichlet":
        core = core - core.mean()
    return core


def _padded(core, pad):
    out = torch.zeros([m + 2 * pad for m in core.shape], dtype=torch.float64, device="cuda")
    out[tuple(slice(pad, -pad) for _ in core.shape)] = core
    return out


class _View:
    """A tensor as the device array that the binding takes."""

    def __init__(self, t):
        self.t, self.ptr = t, ctypes.c_void_p(t.data_ptr())


def _prepare_solve(c, seed):
    per = (1, 1 if c["dim"] == 3 else 0, 1) if c["walls"] == "periodic" else (0, 0, 0)
    g = S.grid_desc((c["nx"], c["ny"], c["nz"]), dim=c["dim"], length=_lengths(c), periodic=per, pad=1)
    p = S.mg_params(vc_count=100, vc_tol=c["tol"], solve_flag=1, mg_tol=c["coarse_tol"], pre=c["nu"], post=c["nu"],
                    res_type=0, bc=S.BC_DIRICHLET if c["walls"] == "dirichlet" else S.BC_NEUMANN,
                    precision=S.PREC_FP64 if c["fp64"] else S.PREC_MIXED, inner_cycles=c["inner"], max_refine=100)
    b = _padded(_solve_rhs(c, seed), 1)
    torch.cuda.synchronize()
    return dict(kind="solve", mg=S.Multigrid(g, p), b=_View(b), x=_View(torch.zeros_like(b)),
                stream=torch.cuda.Stream())


def _axis(n, length, beta=None):
    """Cell centres of a uniform or double-sided tanh axis."""
    xi = (np.arange(n) + 0.5) / n
    if beta is None:
        return length * xi
    return length * (1.0 - np.tanh(beta * (1.0 - 2.0 * xi)) / np.tanh(beta)) / 2.0


def _noise(seed, shape):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return 2.0 * torch.rand(shape, dtype=torch.float64, device="cuda", generator=gen) - 1.0


def _flow(c, seed):
    """Grid, solver and step parameters, the core fields, and the pad of a flow."""
    n = (c["nx"], c["ny"], c["nz"])
    prec = S.PREC_FP64 if c["fp64"] else S.PREC_MIXED
    D, N = S.FBC_DIRICHLET, S.FBC_NEUMANN

    def grids(*axes):
        return torch.meshgrid(*[torch.tensor(a, device="cuda") for a in axes], indexing="ij")

    if c["flow"] == "cavity":
        g = S.grid_desc(n, dim=2, gtype=(S.GRID_TANH_DOUBLE, 0, S.GRID_TANH_DOUBLE), beta=(1.0, 1.0, 1.0), pad=1)
        mg = S.mg_params(vc_count=7, vc_tol=1e-6, solve_flag=0, mg_tol=1e-6, pre=3, post=3, res_type=1,
                         bc=S.BC_NEUMANN, precision=prec)
        vbc = [([D] * 6, [0.0, 0.0, 0.0, 0.0, 0.0, 1.0]), ([D] * 6, [0.0] * 6), ([D] * 6, [0.0] * 6)]
        prm = S.nse_params(dscheme=1, nlscheme=1, has_T=0, nu=1e-3, kappa=1e-3, dt=5e-4, cn_tol=1e-6, scheme=1,
                           vbc=vbc, pbc=([N] * 6, [0.0] * 6))
        # a vortex under the lid, vanishing at the walls
        x, y, z = grids(_axis(n[0], 1.0, 1.0), np.zeros(1), _axis(n[2], 1.0, 1.0))
        vx = -0.3 * torch.sin(math.pi * x) ** 2 * torch.sin(2 * math.pi * z) + 1e-3 * _noise(seed, x.shape)
        vz = 0.3 * torch.sin(2 * math.pi * x) * torch.sin(math.pi * z) ** 2 + 1e-3 * _noise(seed + 1, x.shape)
        return g, mg, prm, dict(vx=vx, vz=vz, p=0.05 * vx * vz), 1, 0.0
    if c["flow"] == "channel":
        m = max(n)
        length = (4.0 * n[0] / m, 4.0 * n[1] / m, 4.0 * n[2] / m)
        g = S.grid_desc(n, length=length, periodic=(1, 1, 0), pad=1)
        mg = S.mg_params(vc_count=10, vc_tol=1e-6, solve_flag=0, mg_tol=1e-6, pre=3, post=3, res_type=0,
                         bc=S.BC_NEUMANN, precision=prec)
        prm = S.nse_params(dscheme=1, nlscheme=2, has_T=0, nu=0.1, kappa=0.1, dt=1e-3, cn_tol=1e-6, scheme=0,
                           mean_pgrad=1.0, buoy=(0.0, 0.0, 0.0), vbc=[([D] * 6, [0.0] * 6)] * 3)
        x, y, z = grids(*[_axis(a, b) for a, b in zip(n, length)])
        base = 5.0 * z * (length[2] - z)
        wave = torch.sin(2 * math.pi * x / length[0]) * torch.cos(2 * math.pi * y / length[1])
        env = z * (length[2] - z)
        f = dict(vx=base + 0.1 * env * _noise(seed, x.shape), vy=0.2 * env * wave + 0.1 * env * _noise(seed + 1, x.shape),
                 vz=0.2 * env * wave + 0.1 * env * _noise(seed + 2, x.shape), p=0.1 * wave)
        return g, mg, prm, f, 1, 0.0
    if c["flow"] == "convection":
        m = max(n)
        length = (n[0] / m, n[1] / m, 1.0)
        g = S.grid_desc(n, length=length, periodic=(1, 1, 0), gtype=(0, 0, S.GRID_TANH_DOUBLE), beta=(1.0, 1.0, 1.5),
                        pad=2)
        mg = S.mg_params(vc_count=20, vc_tol=1e-6, solve_flag=0, mg_tol=1e-2, pre=3, post=6, bc=S.BC_NEUMANN,
                         precision=prec, inner_cycles=5, max_refine=10)
        ph = S.nse_physics(5, ra=1e7, pr=1.0, rbc_type=2, g=(0.0, 0.0, -1.0))
        prm = S.nse_params(dscheme=2, nlscheme=3, has_T=1, nu=ph["nu"], kappa=ph["kappa"], dt=1e-3, cn_tol=1e-6,
                           buoy=ph["buoy"])
        # rolls over the conduction profile
        x, y, z = grids(_axis(n[0], length[0]), _axis(n[1], length[1]), _axis(n[2], 1.0, 1.5))
        sx, cx = torch.sin(2 * math.pi * x / length[0]), torch.cos(2 * math.pi * x / length[0])
        f = dict(vx=-0.1 * sx * torch.sin(2 * math.pi * z), vz=0.2 * length[0] * 0.5 * cx * torch.sin(math.pi * z) ** 2,
                 vy=1e-2 * torch.sin(math.pi * z) * _noise(seed, x.shape),
                 t=1.0 - z + 0.1 * torch.sin(math.pi * z) * cx + 1e-3 * _noise(seed + 1, x.shape),
                 p=torch.ones_like(x))
        return g, mg, prm, f, 2, 0.0
    length = 2.0 * math.pi
    g = S.grid_desc(n, periodic=(1, 1, 1), length=(length,) * 3, pad=2)
    mg = S.mg_params(vc_count=20, vc_tol=1e-6, solve_flag=0, mg_tol=1e-2, pre=3, post=6, bc=S.BC_NEUMANN,
                     precision=prec, inner_cycles=2, max_refine=10)
    nu = S.nse_physics(2, re=1600.0)["nu"]
    prm = S.nse_params(dscheme=2, nlscheme=3, has_T=0, nu=nu, kappa=nu, dt=1e-3, cn_tol=1e-6, les=1,
                       les_sf32=0 if c["fp64"] else 1, vbc=[([D] * 6, [0.0] * 6)] * 3)
    x, y, z = grids(*[_axis(a, length) for a in n])
    f = dict(vx=torch.sin(x) * torch.cos(y) * torch.cos(z) + 0.01 * _noise(seed, x.shape),
             vy=-torch.cos(x) * torch.sin(y) * torch.cos(z) + 0.01 * _noise(seed + 1, x.shape),
             vz=0.01 * _noise(seed + 2, x.shape),
             p=(torch.cos(2 * x) + torch.cos(2 * y)) * (torch.cos(2 * z) + 2.0) / 16.0)
    # the sub-grid model enters once the run time exceeds five steps
    return g, mg, prm, f, 2, 1.0


def _prepare_step(c, seed):
    g, mg, prm, core, pad, time = _flow(c, seed)
    n = (c["nx"], c["ny"], c["nz"])
    ypad = 0 if g.dim == 2 else pad
    shape = (n[0] + 2 * pad, n[1] + 2 * ypad, n[2] + 2 * pad)
    fields, out = [], []
    for k in S.Nse.NAMES:
        f = torch.zeros(shape, dtype=torch.float64, device="cuda")
        if k in core:
            f[pad:-pad, ypad:shape[1] - ypad, pad:-pad] = core[k]
        fields.append(f)
        out.append(torch.zeros_like(f))
    torch.cuda.synchronize()
    s = S.Nse(g, mg, prm)
    del core
    return dict(kind="step", nse=s, time=time, fields=fields, out=out,
                into=[ctypes.c_void_p(f.data_ptr()) for f in fields],
                outof=[ctypes.c_void_p(f.data_ptr()) for f in out])


def _prepare_serve(c, seed):
    # the case fixes the sizes, the seed the right-hand sides
    reqs = serving.draw_requests(c["count"], seed=c["mix"], n3=(32, c["n3_hi"]), n2=(64, c["n2_hi"]))
    for r in reqs:
        r["rhs_seed"] = (r["rhs_seed"] + 1000003 * seed) % (1 << 31)
    prec = S.PREC_FP64 if c["fp64"] else S.PREC_MIXED
    b = [serving.request_rhs(r) for r in reqs]
    server = S.Server(mem_budget=32 << 30, slots=8, use_graphs=True, keep_resident=True, largest_first=True)
    return dict(kind="serve", server=server, b=b, x=[np.zeros_like(a) for a in b],
                grids=[serving.request_grid(r) for r in reqs],
                params=[serving.request_params(r, prec) for r in reqs])


def prepare(case, seed):
    make = {"solve": _prepare_solve, "step": _prepare_step, "serve": _prepare_serve}[case["kind"]]
    return make(case, seed)


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    if state["kind"] == "solve":
        x, stream = state["x"], state["stream"]
        with torch.cuda.stream(stream):
            x.t.zero_()
        state["mg"].solve_device(x, state["b"], stream.cuda_stream)
        return {"x": x.t}
    if state["kind"] == "step":
        s, lib = state["nse"], S.lib()
        S.check(lib.saras_nse_set_fields(s.h, *state["into"], S.PTR_DEVICE))
        s.set_time(state["time"])
        status, _ = s.step()
        S.check(status, (S.OK, S.NOT_CONVERGED))
        S.check(lib.saras_nse_get_fields(s.h, *state["outof"], S.PTR_DEVICE))
        return dict(zip(S.Nse.NAMES, state["out"]))
    server = state["server"]
    for tag, (b, x) in enumerate(zip(state["b"], state["x"])):
        x.fill(0.0)
        server.submit(state["grids"][tag], state["params"][tag], b, x, tag)
    left = len(state["b"])
    while left:
        for done in server.poll(256, wait_ms=1000):
            S.check(done["status"])
            left -= 1
    return list(state["x"])


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _solve_work(cells, tol, nu):
    """x and b read, x written once.  Operations: one V(nu, nu) cycle per
    decade of the tolerance, its sweeps and its residual at about 16
    operations per cell, the coarser levels adding an eighth each."""
    decades = max(1.0, -math.log10(tol))
    return 24.0 * cells, decades * (2 * nu + 1) * 16.0 * cells * 8.0 / 7.0


def work(case):
    if case["kind"] == "serve":
        nbytes = flops = 0.0
        # the stream's mean cube and square, by the logarithm of their extents
        for hi, lo, dim, share in ((case["n3_hi"], 32, 3, 0.75), (case["n2_hi"], 64, 2, 0.25)):
            span = math.log(hi / lo)
            cells = (hi ** dim - lo ** dim) / (dim * span) if span > 0 else float(lo ** dim)
            by, fl = _solve_work(cells, 1e-8, 2)
            nbytes += share * case["count"] * by
            flops += share * case["count"] * fl
        return {"bytes": nbytes, "flops": flops}
    cells = float(case["nx"] * case["ny"] * case["nz"])
    if case["kind"] == "solve":
        by, fl = _solve_work(cells, case["tol"], case["nu"])
        return {"bytes": by, "flops": fl}
    # every field that the flow has, in and out; per stage about 150 operations
    # per transported field, 1500 for the sub-grid model, and the pressure solve
    fields = {"cavity": 3, "channel": 4, "convection": 5, "les": 4}[case["flow"]]
    stages = 1 if case["flow"] == "cavity" else 3
    model = 1500.0 if case["flow"] == "les" else 0.0
    _, solve = _solve_work(cells, 1e-4, 3)
    return {"bytes": 16.0 * fields * cells, "flops": stages * ((fields - 1) * 150.0 + model) * cells + stages * solve}


# ---------------------------------------------------------------------------
# results in 64 bits, without the library
# ---------------------------------------------------------------------------
def exact(case, seed):
    """The discrete solution of a Dirichlet solve, by sine transforms.  With
    Neumann or periodic walls the solution is fixed only up to a constant, and
    a time step's or a batch's result is defined by iterations that stop at a
    tolerance: those have no such value."""
    if case["kind"] != "solve" or case["walls"] != "dirichlet":
        return None
    core = _solve_rhs(case, seed)
    three = case["dim"] == 3
    n = [case["nx"], case["ny"], case["nz"]] if three else [case["nx"], case["nz"]]
    length = _lengths(case) if three else (_lengths(case)[0], _lengths(case)[2])
    lam = torch.zeros([1] * len(n), dtype=torch.float64, device="cuda")
    v = core
    sines = []
    for a, m in enumerate(n):
        k = torch.arange(1, m + 1, dtype=torch.float64, device="cuda")
        i = torch.arange(m, dtype=torch.float64, device="cuda") + 0.5
        s = torch.sin(math.pi * k[:, None] * i[None, :] / m) * math.sqrt(2.0 / m)
        s[-1] *= math.sqrt(0.5)
        sines.append(s)
        h = length[a] / m
        shape = [1] * len(n)
        shape[a] = m
        lam = lam - (4.0 / h ** 2 * torch.sin(math.pi * k / (2 * m)) ** 2).reshape(shape)
        v = torch.movedim(torch.tensordot(s, v, dims=([1], [a])), 0, a)
    v = v / lam
    for a, s in enumerate(sines):
        v = torch.movedim(torch.tensordot(s.t(), v, dims=([1], [a])), 0, a)
    # the ghost layer holds the odd reflection of the edge cells, axis by axis
    out = _padded(v, 1)
    for a in range(len(n)):
        lo, hi = [slice(None)] * len(n), [slice(None)] * len(n)
        lo_in, hi_in = list(lo), list(hi)
        lo[a], lo_in[a], hi[a], hi_in[a] = 0, 1, -1, -2
        out[tuple(lo)] = -out[tuple(lo_in)]
        out[tuple(hi)] = -out[tuple(hi_in)]
    return {"x": out}
