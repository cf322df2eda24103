"""The short roots and quotients of the time step's kernels (nse_round.hpp) against
IEEE arithmetic (NumPy's, on the host), bit for bit: every significand of the root
and of the constant's quotient, random pairs and the ends of the ranges that they
are stated for.  And the single-precision sub-grid stresses on cells too narrow
for them, which take the library's root and division.
"""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import oracle as O
import saras_amd as S
from test_gpu_nse import mg_kw

pytestmark = pytest.mark.gpu

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native")
LIB = os.path.join(HERE, "_build", "libround_check.so")
SIGNIFICANDS = np.arange(1 << 23, dtype=np.uint32)


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(LIB):
        subprocess.run(["make", "-C", HERE], check=True)
    return ctypes.CDLL(LIB)


def floats(exponent):
    """Every float of one binary exponent."""
    return (SIGNIFICANDS | np.uint32((exponent + 127) << 23)).view(np.float32)


def run(lib, kind, a, b=None):
    a = np.ascontiguousarray(a, np.float32)
    b = None if b is None else np.ascontiguousarray(np.broadcast_to(b, a.shape), np.float32)
    out = np.empty_like(a)
    assert lib.round_check_float(kind, ctypes.c_long(a.size), a.ctypes.data_as(ctypes.c_void_p),
                                 None if b is None else b.ctypes.data_as(ctypes.c_void_p),
                                 out.ctypes.data_as(ctypes.c_void_p)) == 0
    return out


def same(x, y):
    np.testing.assert_array_equal(x.view(np.uint32), y.view(np.uint32))


@pytest.mark.parametrize("exponent", [-100, -99, -95, -70, -1, 0, 1, 35, 72, 126, 127])
def test_root_every_significand(lib, exponent):
    a = floats(exponent)
    same(run(lib, 0, a), np.sqrt(a))


def test_root_outside_its_range(lib):
    a = np.float32([0.0, -0.0, 1e-45, 1e-38, 2.0 ** -101, np.nextafter(np.float32(2.0 ** -100), np.float32(0)),
                    -1e-45, -2.0 ** -30, -1.0, -3e38])
    np.testing.assert_array_equal(run(lib, 0, a), 0.0)


@pytest.mark.parametrize("exponent", [-60, -1, 0, 1, 36, 108, 119])
def test_quotient_of_the_constant(lib, exponent):
    b = floats(exponent)
    a = np.full_like(b, np.float32(0.573159))
    same(run(lib, 2, a, b), a / b)


@pytest.mark.parametrize("seed", range(4))
def test_quotients(lib, seed):
    rng = np.random.default_rng(seed)
    n = 1 << 22
    b = np.float32(rng.uniform(1, 2, n)) * np.float32(2.0) ** rng.integers(-35, 36, n).astype(np.float32)
    a = b * np.float32(rng.uniform(1, 2, n)) * np.float32(2.0) ** rng.integers(-24, 40, n).astype(np.float32)
    a[:4] = 0.0
    same(run(lib, 1, a, b), a / b)


def test_by6(lib):
    rng = np.random.default_rng(5)
    n = 1 << 22
    a = rng.uniform(1, 2, n) * 2.0 ** rng.integers(-1018, 1023, n).astype(float) * rng.choice([-1.0, 1.0], n)
    a[:8] = [0.0, -0.0, np.inf, -np.inf, np.nan, 6.0, -18.0, np.finfo(float).max]
    out = np.empty_like(a)
    assert lib.round_check_by6(ctypes.c_long(n), a.ctypes.data_as(ctypes.c_void_p), out.ctypes.data_as(ctypes.c_void_p)) == 0
    q = a / 6.0
    np.testing.assert_array_equal(out, q)
    np.testing.assert_array_equal(np.signbit(out[:4]), np.signbit(q[:4]))
    # subnormal quotients: within one unit
    a = rng.uniform(1, 2, 1 << 16) * 2.0 ** rng.integers(-1074, -1020, 1 << 16).astype(float)
    out = np.empty_like(a)
    assert lib.round_check_by6(ctypes.c_long(a.size), a.ctypes.data_as(ctypes.c_void_p),
                               out.ctypes.data_as(ctypes.c_void_p)) == 0
    assert np.abs(out.view(np.int64) - (a / 6.0).view(np.int64)).max() <= 1


@pytest.mark.parametrize("tanh", [False, True], ids=["uniform", "tanh"])
@pytest.mark.parametrize("width", [2e-16, 1e-13, 1e-3], ids=["2e-16", "1e-13", "1e-3"])
def test_stresses_of_narrow_cells(width, tanh):
    """The velocities shrink with the cells, so that the strain rates stay.  On
    stretched axes all 26 neighbour offsets are evaluated."""
    n = (8, 6, 72)
    length = tuple(width * m for m in n)
    kw = dict(has_T=0, nu=1.0 / 1600 * width ** 2, dt=1e-3, cn_tol=1e-10, les=1)
    mg = mg_kw(vc_count=2, vc_tol=1e-10, pre=2, post=2)
    geo = dict(periodic=(1, 1, 1), gtype=(2, 2, 2) if tanh else (0, 0, 0), beta=(0.8, 0.7, 0.9), length=length, pad=2)
    so = O.Nse(O.nse_desc(O.grid_desc(n, **geo), mg=O.mg_params(bc=O.BC_NEUMANN, **mg), **kw))
    ss = S.Nse(S.grid_desc(n, **geo), S.mg_params(bc=S.BC_NEUMANN, precision=S.PREC_FP64, **mg),
               S.nse_params(**kw, les_sf32=1))
    rng = np.random.default_rng(24)
    sh = so.shape
    z = np.zeros(sh)
    x, y, w = np.meshgrid(*[2 * np.pi * (np.arange(-2, m + 2) + 0.5) / m for m in n], indexing="ij")
    f = dict(vx=np.sin(x) * np.cos(y) * np.cos(w) + 0.1 * rng.uniform(-1, 1, sh),
             vy=-np.cos(x) * np.sin(y) * np.cos(w) + 0.1 * rng.uniform(-1, 1, sh), vz=0.1 * rng.uniform(-1, 1, sh),
             p=z, t=z, pp=z)
    f = {k: v * width for k, v in f.items()}
    so.set(**f)
    ss.set(**f)
    for _ in range(6):   # the steps before the model enters
        assert so.step() == 0
        assert ss.step()[0] == 0
    f = so.get()
    ss.set(**f)
    c = (slice(2, -2),) * 3
    ro, rs = so.rhs(0), ss.rhs(0)
    # the bars of the single-precision integral (test_gpu_sgs_march.py)
    for k in ("rx", "ry", "rz", "hx", "hy", "hz"):
        a, b = ro[k][c], rs[k][c]
        assert np.abs(a - b).max() <= 1e-6 * np.abs(a).max(), (k, np.abs(a - b).max(), np.abs(a).max())
    do = so.sgs_diag()
    dg, _ = ss.sgs()
    for q, k in enumerate(("sgke", "disp", "nusg")):
        assert abs(dg[k] - do[q]) <= 1e-6 * abs(do[q]), (k, dg[k], do[q])
