"""The single-workgroup bottom of the V-cycle at the sizes where its cell
tables, register cells and barriers can go wrong, bit for bit against the FP64
CPU oracle, and in FP32 against the multi-workgroup kernels: one cell of a
colour per lane of one wave and one more, one per thread and one more, the
register limit and levels beyond it, odd rows, odd periodic extents (a wrapped
neighbour of the cell's own colour) in each of those, every wall kind, and
coarsest levels that are smoothed as well as solved.
"""
import numpy as np
import pytest

import oracle as O
import saras_amd as S

pytestmark = pytest.mark.gpu

CASES = [
    # n, dim, periodic, bc: the coarsest level and the cells of a colour it has
    ((8, 8, 8), 3, (1, 1, 1), O.BC_NEUMANN),        # 2^3: 4
    ((10, 10, 10), 3, (1, 1, 1), O.BC_NEUMANN),     # 5^3, odd: 75 positions (> one wave)
    ((6, 6, 6), 3, (1, 1, 1), O.BC_NEUMANN),        # 3^3, odd: 18
    ((16, 16, 8), 3, (0, 0, 0), O.BC_DIRICHLET),    # 4 x 4 x 2: 16
    ((16, 16, 4), 3, (1, 1, 0), O.BC_NEUMANN),      # one level above 4 x 4 x 1
    ((32, 16, 32), 3, (0, 0, 0), O.BC_DIRICHLET),   # 16^2 x 8 level: 1024
    ((18, 18, 18), 3, (1, 1, 1), O.BC_NEUMANN),     # 9^3, odd: 405
    ((20, 20, 22), 3, (1, 1, 0), O.BC_NEUMANN),     # 10 x 10 x 11, odd rows: 600
    ((26, 26, 26), 3, (1, 1, 1), O.BC_NEUMANN),     # 13^3, odd: 1183
    ((28, 28, 28), 3, (0, 0, 0), O.BC_NEUMANN),     # 14^3: 1372
    ((28, 28, 28), 3, (0, 0, 0), O.BC_DIRICHLET),
    ((32, 32, 32), 3, (0, 0, 0), O.BC_NEUMANN),     # a 16^3 level: 2048
    ((34, 34, 34), 3, (1, 1, 1), O.BC_NEUMANN),     # 17^3, odd: 2601 (beyond the registers)
    ((36, 28, 50), 3, (1, 1, 0), O.BC_NEUMANN),     # 18 x 14 x 25, odd rows: 3276
    ((36, 28, 50), 3, (1, 0, 1), O.BC_DIRICHLET),   # the same, odd periodic z
    ((64, 1, 64), 2, (0, 0, 0), O.BC_DIRICHLET),    # all levels in the tail: 2048
    ((32, 1, 34), 2, (1, 0, 1), O.BC_NEUMANN),      # 16 x 17, odd z: 144
    ((130, 1, 30), 2, (0, 0, 1), O.BC_NEUMANN),     # 65 x 15, odd z: 520
]
IDS = [f"{d}d-{'x'.join(map(str, n))}-p{''.join(map(str, p))}-bc{b}" for n, d, p, b in CASES]


def rhs(mo, rng, compatible):
    shp = O.field_shape(mo.g, 1)
    b = np.zeros(shp)
    c = rng.standard_normal(tuple(s - 2 for s in shp))
    b[(slice(1, -1),) * len(shp)] = c - c.mean() if compatible else c
    return b


@pytest.mark.parametrize("solve_flag", [1, 0])
@pytest.mark.parametrize("case", CASES, ids=IDS)
def test_tail_bitexact(case, solve_flag):
    n, dim, per, bc = case
    kw = dict(vc_count=3, vc_tol=1e-12, mg_tol=1e-6, pre=2, post=3, sor=1.1 if solve_flag else 1.0,
              solve_flag=solve_flag)
    gt, beta = (0, 0, 0 if per[2] else 2), (1.0, 1.0, 0.6)
    mo = O.Multigrid(O.grid_desc(n, dim=dim, periodic=per, gtype=gt, beta=beta), O.mg_params(bc=bc, **kw))
    ms = S.Multigrid(S.grid_desc(n, dim=dim, periodic=per, gtype=gt, beta=beta),
                     S.mg_params(bc=S.BC_NEUMANN if bc == O.BC_NEUMANN else S.BC_DIRICHLET, **kw))
    rng = np.random.default_rng(21)
    b = rhs(mo, rng, bc == O.BC_NEUMANN)
    x0 = rhs(mo, rng, False) * 0.1
    xo, so = mo.solve(x0.copy(), b, 1)
    xs, ss, _ = ms.solve(x0.copy(), b)
    assert ss["cycles"] == so["cycles"] and ss["residual"] == so["residual"]
    if solve_flag:
        assert ss["coarse_iters_max"] == so["coarse_iters_max"]
    np.testing.assert_array_equal(xs, xo)


@pytest.mark.parametrize("solve_flag", [1, 0])
@pytest.mark.parametrize("case", CASES, ids=IDS)
def test_tail_fp32_matches_per_level(case, solve_flag, monkeypatch):
    n, dim, per, bc = case
    kw = dict(vc_count=4, vc_tol=1e-14, mg_tol=1e-10, pre=2, post=2, solve_flag=solve_flag, precision=S.PREC_MIXED,
              inner_cycles=2, max_refine=2, bc=S.BC_NEUMANN if bc == O.BC_NEUMANN else S.BC_DIRICHLET)
    g = S.grid_desc(n, dim=dim, periodic=per)
    out = []
    rng = np.random.default_rng(22)
    mo = O.Multigrid(O.grid_desc(n, dim=dim, periodic=per), O.mg_params(bc=bc))
    b = rhs(mo, rng, bc == O.BC_NEUMANN)
    for tail in (True, False):
        if not tail:
            monkeypatch.setenv("SARAS_NO_TAIL", "1")
        x, st, _ = S.Multigrid(g, S.mg_params(**kw)).solve(np.zeros_like(b), b)
        out.append((x, st["residual"], st["coarse_iters_max"]))
    np.testing.assert_array_equal(out[0][0], out[1][0])
    assert out[0][1:] == out[1][1:]
