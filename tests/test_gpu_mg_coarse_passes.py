"""A coarsest level too large for one workgroup's LDS, smoothed by colour passes
of the whole chip (k_coarse_pass), against the FP64 CPU oracle and against the
one-workgroup kernel, bit for bit: odd and even extents, periodic axes (an odd
extent makes a cell and its image neighbour one colour), every wall kind.
"""
import numpy as np
import pytest

import oracle as O
import saras_amd as S

pytestmark = pytest.mark.gpu

CASES = [
    # n, dim, periodic, stretched, bc, mixed
    ((74, 30, 54), 3, (1, 0, 1), False, O.BC_NEUMANN, False),
    ((50, 38, 66), 3, (0, 0, 0), True, O.BC_DIRICHLET, False),
    ((54, 50, 46), 3, (1, 1, 1), False, O.BC_NEUMANN, False),
    ((50, 38, 34), 3, (0, 0, 0), False, O.BC_DIRICHLET_TEST, False),
    ((74, 62, 58), 3, (1, 1, 0), True, O.BC_NEUMANN, True),
    ((190, 1, 186), 2, (1, 0, 0), False, O.BC_NEUMANN, False),
    ((202, 1, 198), 2, (0, 0, 1), True, O.BC_DIRICHLET, False),
]
IDS = ["x".join(map(str, c[0])) + f"-p{''.join(map(str, c[2]))}-bc{c[4]}" + ("-mixed" if c[5] else "") for c in CASES]
BC = {O.BC_NEUMANN: S.BC_NEUMANN, O.BC_DIRICHLET: S.BC_DIRICHLET, O.BC_DIRICHLET_TEST: S.BC_DIRICHLET_TEST}


@pytest.mark.parametrize("case", CASES, ids=IDS)
def test_bitexact(case, monkeypatch):
    n, dim, per, tanh, bc, mixed = case
    kw = dict(dim=dim, periodic=per, gtype=tuple(0 if p or not tanh else 2 for p in per), beta=(0.6, 0.5, 0.7))
    go, gs = O.grid_desc(n, **kw), S.grid_desc(n, **kw)
    pk = dict(vc_count=2, vc_tol=1e-14, mg_tol=1e-2, pre=3, post=2, sor=1.1, solve_flag=0)
    mk = dict(precision=S.PREC_MIXED, inner_cycles=1, max_refine=2) if mixed else {}
    ms = S.Multigrid(gs, S.mg_params(bc=BC[bc], **pk, **mk))
    monkeypatch.setenv("SARAS_COARSE_ONE", "1")
    m1 = S.Multigrid(gs, S.mg_params(bc=BC[bc], **pk, **mk))
    shp = O.field_shape(go, 1)
    rng = np.random.default_rng(43)
    core = (slice(1, -1),) * len(shp)
    b = np.zeros(shp)
    r = rng.standard_normal(tuple(q - 2 for q in shp))
    b[core] = r - r.mean() if bc == O.BC_NEUMANN else r
    x0 = np.zeros(shp)
    x0[core] = 0.1 * rng.standard_normal(r.shape)
    xs, ss, _ = ms.solve(x0.copy(), b)
    x1, s1, _ = m1.solve(x0.copy(), b)
    assert np.array_equal(xs[core], x1[core])
    assert ss["residual"] == s1["residual"]
    if not mixed:
        xo, so = O.Multigrid(go, O.mg_params(bc=bc, **pk)).solve(x0.copy(), b, 1)
        assert np.array_equal(xo[core], xs[core]), np.abs(xo[core] - xs[core]).max()
