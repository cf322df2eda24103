"""Solved coarsest levels that fit the tail's LDS only without their right-hand
side (k_tail with it in global memory), against the CPU oracle (FP64, bit for bit)
and, in FP32, against the workgroup-wide solve in global memory (k_coarse).
"""
import numpy as np
import pytest

import oracle as O
import saras_amd as S
from test_gpu_mg_tile import rhs

pytestmark = pytest.mark.gpu

CASES = [
    # n (the coarsest level itself), dim, periodic, bc
    ((82, 1, 86), 2, (0, 0, 0), O.BC_DIRICHLET),
    ((85, 1, 86), 2, (1, 0, 1), O.BC_NEUMANN),     # an odd periodic extent
    ((83, 1, 90), 2, (0, 0, 1), O.BC_NEUMANN),
    ((18, 18, 22), 3, (0, 0, 0), O.BC_DIRICHLET),
    ((19, 18, 19), 3, (1, 1, 0), O.BC_NEUMANN),    # rows of odd length
    ((18, 15, 26), 3, (1, 1, 1), O.BC_NEUMANN),
]
IDS = [f"{d}d-{'x'.join(map(str, n))}-p{''.join(map(str, p))}-bc{b}" for n, d, p, b in CASES]


@pytest.mark.parametrize("levels", [1, 2])
@pytest.mark.parametrize("case", CASES, ids=IDS)
def test_fp64_bitexact(case, levels):
    n, dim, per, bc = case
    n = tuple(m if dim == 2 and a == 1 else m << (levels - 1) for a, m in enumerate(n))
    kw = dict(vc_count=2, vc_tol=1e-14, mg_tol=1e-1, pre=2, post=2, solve_flag=1)
    go, gs = O.grid_desc(n, dim=dim, periodic=per), S.grid_desc(n, dim=dim, periodic=per)
    mo = O.Multigrid(go, O.mg_params(bc=bc, **kw))
    ms = S.Multigrid(gs, S.mg_params(bc=S.BC_NEUMANN if bc == O.BC_NEUMANN else S.BC_DIRICHLET, **kw))
    rng = np.random.default_rng(71)
    b, x0 = rhs(go, rng, bc == O.BC_NEUMANN), rhs(go, rng, False) * 0.1
    xo, so = mo.solve(x0.copy(), b, 1)
    xs, ss, _ = ms.solve(x0.copy(), b)
    assert ss["residual"] == so["residual"]
    np.testing.assert_array_equal(xs, xo)


@pytest.mark.parametrize("n,dim,per", [((236, 1, 236), 2, (0, 0, 0)), ((230, 1, 246), 2, (1, 0, 1)), ((48, 46, 50), 3, (1, 1, 0))])
def test_fp32_matches_k_coarse(n, dim, per, monkeypatch):
    kw = dict(vc_count=6, vc_tol=1e-14, mg_tol=1e-4, pre=2, post=2, precision=S.PREC_MIXED, inner_cycles=3, max_refine=2,
              solve_flag=1, bc=S.BC_NEUMANN)
    b = rhs(O.grid_desc(n, dim=dim, periodic=per), np.random.default_rng(72), True)
    out = []
    for tail in (True, False):
        if not tail:
            monkeypatch.setenv("SARAS_NO_TAIL", "1")
        x, st, _ = S.Multigrid(S.grid_desc(n, dim=dim, periodic=per), S.mg_params(**kw)).solve(np.zeros_like(b), b)
        out.append((x, st["residual"], st["coarse_iters_max"]))
    np.testing.assert_array_equal(out[0][0], out[1][0])
    assert out[0][1:] == out[1][1:]
