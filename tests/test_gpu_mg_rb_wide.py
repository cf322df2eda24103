"""The forms of the split colour passes and the restriction for arrays of 4 GB
and more (64-bit offsets, vector numbers divided as they are), forced on small
levels: against the FP64 CPU oracle and, in FP32, against the usual forms, bit
for bit.
"""
import numpy as np
import pytest

import oracle as O
import saras_amd as S
from test_gpu_mg_rb import BC, CASES, IDS, grids, rhs

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def passes(monkeypatch):
    monkeypatch.setenv("SARAS_NO_TILE", "1")
    monkeypatch.setenv("SARAS_TAIL_LDS_KB", "1")   # (almost) every level by passes


@pytest.mark.parametrize("sor", [1.0, 1.2])
@pytest.mark.parametrize("case", CASES, ids=IDS)
def test_fp64_bitexact(case, sor, monkeypatch):
    monkeypatch.setenv("SARAS_RB_WIDE", "1")
    go, gs = grids(case)
    kw = dict(vc_count=2, vc_tol=1e-14, mg_tol=1e-2, pre=2, post=2, sor=sor, solve_flag=0)
    mo, ms = O.Multigrid(go, O.mg_params(bc=case[4], **kw)), S.Multigrid(gs, S.mg_params(bc=BC[case[4]], **kw))
    rng = np.random.default_rng(61)
    b, x0 = rhs(go, rng, case[4] == O.BC_NEUMANN), rhs(go, rng, False) * 0.1
    xo, so = mo.solve(x0.copy(), b, 1)
    xs, ss, _ = ms.solve(x0.copy(), b)
    assert ss["residual"] == so["residual"]
    np.testing.assert_array_equal(xs, xo)


@pytest.mark.parametrize("sor", [1.0, 1.2])
@pytest.mark.parametrize("case", [c for c in CASES if c[4] != O.BC_DIRICHLET_TEST],
                         ids=[i for c, i in zip(CASES, IDS) if c[4] != O.BC_DIRICHLET_TEST])
def test_fp32_matches(case, sor, monkeypatch):
    go, gs = grids(case)
    kw = dict(vc_count=6, vc_tol=1e-14, mg_tol=1e-6, pre=2, post=2, sor=sor, precision=S.PREC_MIXED, inner_cycles=3,
              max_refine=2, solve_flag=0, bc=BC[case[4]])
    b = rhs(go, np.random.default_rng(62), case[4] == O.BC_NEUMANN)
    out = []
    for wide in (False, True):
        if wide:
            monkeypatch.setenv("SARAS_RB_WIDE", "1")
        x, st, _ = S.Multigrid(gs, S.mg_params(**kw)).solve(np.zeros_like(b), b)
        out.append((x, st["residual"]))
    np.testing.assert_array_equal(out[0][0], out[1][0])
    assert out[0][1] == out[1][1]
