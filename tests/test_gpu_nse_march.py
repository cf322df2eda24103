"""The marching right-hand side (k_rhs_march), Jacobi iteration (k_jacobi_march),
divergence and pressure correction (k_div_march, k_correct_march) against the
kernels per field and per cell, bit for bit: rows shorter and longer than a block, part-filled blocks in y and z,
one chunk of planes and several, z walls of both kinds with values and without
walls, with and without temperature, with and without the sub-grid stresses.
"""
import numpy as np
import pytest

import saras_amd as S

pytestmark = pytest.mark.gpu

D, N = S.FBC_DIRICHLET, S.FBC_NEUMANN
# n, z periodic, kind of the z walls (lo, hi) of the velocities and of T, has_T, les
CASES = [
    ((16, 16, 16), 0, (D, D), (D, D), 1, 0),
    ((8, 12, 12), 0, (D, N), (N, D), 1, 0),
    ((64, 8, 8), 0, (N, D), (D, N), 0, 0),
    ((4, 72, 72), 0, (D, D), (D, N), 1, 0),
    ((12, 6, 136), 1, None, None, 1, 0),
    ((36, 20, 8), 1, None, None, 0, 0),
    ((16, 16, 16), 1, None, None, 0, 1),
    ((8, 12, 72), 1, None, None, 1, 1),
]
IDS = ["x".join(map(str, c[0])) + ("-p" if c[1] else "-w") + ("-T" if c[4] else "") + ("-les" if c[5] else "") for c in CASES]


def make(case, march, monkeypatch):
    n, zp, vz, tz, has_t, les = case
    monkeypatch.setenv("SARAS_NO_NSE_MARCH", "0" if march else "1")
    g = S.grid_desc(n, periodic=(1, 1, zp), gtype=(0, 0, 0 if zp else 2), beta=(1.0, 1.0, 1.4), pad=2)
    vz, tz = vz or (D, D), tz or (D, D)
    vbc = [([D] * 4 + list(vz), [0.0] * 4 + [0.1 * (q + 1), -0.2 * q]) for q in range(3)]
    p = S.nse_params(dscheme=2, nlscheme=3, has_T=has_t, nu=3e-3, kappa=2e-3, dt=1e-3, cn_tol=1e-8, les=les,
                     vbc=vbc, tbc=([D] * 4 + list(tz), [0.0] * 4 + [0.7, -0.3]), buoy=(0.1, 0.0, -0.9))
    mg = S.mg_params(bc=S.BC_NEUMANN, precision=S.PREC_FP64, vc_count=2, vc_tol=1e-6, solve_flag=0, pre=2, post=2)
    return S.Nse(g, mg, p)


@pytest.mark.parametrize("case", CASES, ids=IDS)
def test_same_as_per_field_kernels(case, monkeypatch):
    n = case[0]
    a, b = make(case, True, monkeypatch), make(case, False, monkeypatch)
    shape = tuple(m + 4 for m in n)
    c = (slice(2, -2),) * 3
    rng = np.random.default_rng(17)
    f = {k: rng.standard_normal(shape) for k in ("vx", "vy", "vz", "p", "t")}
    f["pp"] = np.zeros(shape)
    for s in (a, b):
        s.set(**f)
        s.set_time(1.0)   # past the steps that run without the sub-grid model
    for stage in (0, 1, 2):
        ra, rb = a.rhs(stage), b.rhs(stage)
        assert ra.keys() == rb.keys()
        for k in ra:
            assert np.array_equal(ra[k][c], rb[k][c]), (stage, k)
    same_steps(a, b)


def same_steps(a, b):
    c = (slice(2, -2),) * 3
    for step in range(2):
        (ea, sa), (eb, sb) = a.step(), b.step()
        assert ea == eb == 0
        assert sa["jacobi_iters"] == sb["jacobi_iters"]
        fa, fb = a.get(), b.get()
        for k in fa:
            assert np.array_equal(fa[k][c], fb[k][c]), (step, k)
    a.close()
    b.close()


@pytest.mark.parametrize("scheme", [0, 1], ids=["rk3", "euler_cn"])
@pytest.mark.parametrize("n", [(4, 4, 4), (16, 6, 72), (40, 20, 12), (8, 12, 136)], ids=lambda n: "x".join(map(str, n)))
def test_walls_on_every_side(n, scheme, monkeypatch):
    def make(march):
        monkeypatch.setenv("SARAS_NO_NSE_MARCH", "0" if march else "1")
        g = S.grid_desc(n, periodic=(0, 0, 0), gtype=(2, 0, 1), beta=(1.1, 1.0, 0.8), pad=2)
        vbc = [([(D, N)[(w + q) % 2] for w in range(6)], [0.1 * w - 0.2 * q for w in range(6)]) for q in range(3)]
        p = S.nse_params(dscheme=2, nlscheme=1, has_T=1, nu=2e-2, kappa=3e-2, dt=2e-3, cn_tol=1e-9, scheme=scheme, vbc=vbc,
                         tbc=([N, D, D, N, D, D], [0.3, -0.1, 0.2, 0.0, 1.0, -1.0]), buoy=(0.1, 0.0, -0.9))
        mg = S.mg_params(bc=S.BC_NEUMANN, precision=S.PREC_FP64, vc_count=2, vc_tol=1e-6, solve_flag=0, pre=2, post=2)
        return S.Nse(g, mg, p)
    a, b = make(True), make(False)
    rng = np.random.default_rng(29)
    f = {k: 0.1 * rng.standard_normal(tuple(m + 4 for m in n)) for k in ("vx", "vy", "vz", "p", "t", "pp")}
    for s in (a, b):
        s.set(**f)
    same_steps(a, b)
