"""The paired-row colour pass (k_rb_split) against its general form and the
FP64 CPU oracle, bit for bit: every pass of the finest and of a coarser level as
a launch of its own (no tiles), uniform and stretched axes, every wall kind, row
lengths that fill part of a wave, one wave and several, both SOR parameters.
"""
import numpy as np
import pytest

import oracle as O
import saras_amd as S

pytestmark = pytest.mark.gpu

CASES = [
    # n, dim, periodic, stretched, bc
    ((16, 16, 16), 3, (1, 1, 1), False, O.BC_NEUMANN),
    ((8, 24, 32), 3, (0, 0, 0), True, O.BC_DIRICHLET),
    ((16, 8, 48), 3, (1, 0, 1), False, O.BC_NEUMANN),
    ((12, 20, 16), 3, (0, 1, 0), True, O.BC_NEUMANN),
    ((8, 8, 272), 3, (0, 0, 0), False, O.BC_DIRICHLET),
    ((8, 8, 640), 3, (1, 1, 0), True, O.BC_NEUMANN),
    ((8, 8, 16), 3, (0, 0, 0), False, O.BC_DIRICHLET_TEST),
    ((48, 1, 64), 2, (0, 0, 1), False, O.BC_NEUMANN),
    ((24, 1, 160), 2, (1, 0, 0), True, O.BC_DIRICHLET),
    ((16, 1, 16), 2, (0, 0, 0), False, O.BC_DIRICHLET_TEST),
]
IDS = [f"{d}d-{'x'.join(map(str, n))}-p{''.join(map(str, p))}-{'tanh' if t else 'uni'}-bc{b}" for n, d, p, t, b in CASES]
BC = {O.BC_NEUMANN: S.BC_NEUMANN, O.BC_DIRICHLET: S.BC_DIRICHLET, O.BC_DIRICHLET_TEST: S.BC_DIRICHLET_TEST}


def grids(case):
    n, dim, per, tanh, bc = case
    gt = tuple(0 if per[a] or not tanh else 2 for a in range(3))
    kw = dict(dim=dim, periodic=per, gtype=gt, beta=(0.6, 0.5, 0.7))
    return O.grid_desc(n, **kw), S.grid_desc(n, **kw)


def rhs(g, rng, compatible):
    shp = O.field_shape(g, 1)
    b = np.zeros(shp)
    c = rng.standard_normal(tuple(s - 2 for s in shp))
    b[(slice(1, -1),) * len(shp)] = c - c.mean() if compatible else c
    return b


@pytest.mark.parametrize("general", [False, True])
@pytest.mark.parametrize("sor", [1.0, 1.2])
@pytest.mark.parametrize("case", CASES, ids=IDS)
def test_passes_bitexact(case, sor, general, monkeypatch):
    monkeypatch.setenv("SARAS_NO_TILE", "1")
    monkeypatch.setenv("SARAS_TAIL_LDS_KB", "1")   # (almost) every level by passes
    if general:
        monkeypatch.setenv("SARAS_RB_GENERAL", "1")
    go, gs = grids(case)
    kw = dict(vc_count=2, vc_tol=1e-14, mg_tol=1e-2, pre=2, post=2, sor=sor, solve_flag=0)
    mo, ms = O.Multigrid(go, O.mg_params(bc=case[4], **kw)), S.Multigrid(gs, S.mg_params(bc=BC[case[4]], **kw))
    rng = np.random.default_rng(41)
    b, x0 = rhs(go, rng, case[4] == O.BC_NEUMANN), rhs(go, rng, False) * 0.1
    xo, so = mo.solve(x0.copy(), b, 1)
    xs, ss, _ = ms.solve(x0.copy(), b)
    assert ss["residual"] == so["residual"]
    np.testing.assert_array_equal(xs, xo)


@pytest.mark.parametrize("sor", [1.0, 1.2])
@pytest.mark.parametrize("case", [c for c in CASES if c[4] != O.BC_DIRICHLET_TEST],
                         ids=[i for c, i in zip(CASES, IDS) if c[4] != O.BC_DIRICHLET_TEST])
def test_fp32_passes_match_general(case, sor, monkeypatch):
    monkeypatch.setenv("SARAS_NO_TILE", "1")
    monkeypatch.setenv("SARAS_TAIL_LDS_KB", "1")
    go, gs = grids(case)
    kw = dict(vc_count=6, vc_tol=1e-14, mg_tol=1e-6, pre=2, post=2, sor=sor, precision=S.PREC_MIXED, inner_cycles=3,
              max_refine=2, solve_flag=0, bc=BC[case[4]])
    b = rhs(go, np.random.default_rng(42), case[4] == O.BC_NEUMANN)
    out = []
    for general in (False, True):
        if general:
            monkeypatch.setenv("SARAS_RB_GENERAL", "1")
        x, st, _ = S.Multigrid(gs, S.mg_params(**kw)).solve(np.zeros_like(b), b)
        out.append((x, st["residual"]))
    np.testing.assert_array_equal(out[0][0], out[1][0])
    assert out[0][1] == out[1][1]
