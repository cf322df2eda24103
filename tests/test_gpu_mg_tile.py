"""Several passes of a level in one launch (k_tile) against the FP64 CPU oracle
and, in both precisions, against one launch per pass: bit for bit, for every
wall kind, extents that are no multiple of a tile, rows that are no whole
number of vectors, z-contiguous and colour-split levels, sweep counts that
take one and several launches, and an over-relaxed SOR parameter.
"""
import numpy as np
import pytest

import oracle as O
import saras_amd as S

pytestmark = pytest.mark.gpu

CASES = [
    # n, dim, periodic, bc
    ((32, 32, 32), 3, (1, 1, 1), O.BC_NEUMANN),
    ((32, 48, 64), 3, (0, 0, 0), O.BC_DIRICHLET),
    ((36, 28, 50), 3, (1, 1, 0), O.BC_NEUMANN),     # rows of 25 pairs
    ((20, 36, 44), 3, (0, 1, 1), O.BC_NEUMANN),     # 22 pairs: no whole FP32 vectors
    ((40, 24, 56), 3, (1, 0, 0), O.BC_DIRICHLET),
    ((64, 64, 64), 3, (0, 0, 0), O.BC_NEUMANN),
    ((72, 12, 20), 3, (1, 1, 1), O.BC_NEUMANN),     # a y extent close to the halo
    ((128, 1, 128), 2, (0, 0, 0), O.BC_NEUMANN),
    ((196, 1, 100), 2, (1, 0, 0), O.BC_DIRICHLET),  # 50 pairs, tiles cut at the end
    ((96, 1, 260), 2, (1, 0, 1), O.BC_NEUMANN),
]
IDS = [f"{d}d-{'x'.join(map(str, n))}-p{''.join(map(str, p))}-bc{b}" for n, d, p, b in CASES]
SWEEPS = [(2, 2, 1.0), (3, 6, 1.0), (1, 3, 1.2)]


def rhs(g, rng, compatible):
    shp = O.field_shape(g, 1)
    b = np.zeros(shp)
    c = rng.standard_normal(tuple(s - 2 for s in shp))
    b[(slice(1, -1),) * len(shp)] = c - c.mean() if compatible else c
    return b


@pytest.mark.parametrize("pre,post,sor", SWEEPS)
@pytest.mark.parametrize("case", CASES, ids=IDS)
def test_tile_fp64_bitexact(case, pre, post, sor):
    n, dim, per, bc = case
    kw = dict(vc_count=2, vc_tol=1e-14, mg_tol=1e-2, pre=pre, post=post, sor=sor, solve_flag=0)
    gt, beta = (0 if per[0] else 1, 0, 0 if per[2] else 2), (0.5, 1.0, 0.7)
    go = O.grid_desc(n, dim=dim, periodic=per, gtype=gt, beta=beta)
    mo = O.Multigrid(go, O.mg_params(bc=bc, **kw))
    ms = S.Multigrid(S.grid_desc(n, dim=dim, periodic=per, gtype=gt, beta=beta),
                     S.mg_params(bc=S.BC_NEUMANN if bc == O.BC_NEUMANN else S.BC_DIRICHLET, **kw))
    rng = np.random.default_rng(31)
    b, x0 = rhs(go, rng, bc == O.BC_NEUMANN), rhs(go, rng, False) * 0.1
    xo, so = mo.solve(x0.copy(), b, 1)
    xs, ss, _ = ms.solve(x0.copy(), b)
    assert ss["residual"] == so["residual"]
    np.testing.assert_array_equal(xs, xo)


@pytest.mark.parametrize("graphs", [False, True])
@pytest.mark.parametrize("pre,post,sor", SWEEPS)
@pytest.mark.parametrize("case", CASES, ids=IDS)
def test_tile_fp32_matches_passes(case, pre, post, sor, graphs, monkeypatch):
    n, dim, per, bc = case
    kw = dict(vc_count=6, vc_tol=1e-14, mg_tol=1e-6, pre=pre, post=post, sor=sor, precision=S.PREC_MIXED,
              inner_cycles=3, max_refine=2, bc=S.BC_NEUMANN if bc == O.BC_NEUMANN else S.BC_DIRICHLET)
    g = S.grid_desc(n, dim=dim, periodic=per)
    rng = np.random.default_rng(32)
    b = rhs(O.grid_desc(n, dim=dim, periodic=per), rng, bc == O.BC_NEUMANN)
    out = []
    for tile in (True, False):
        if not tile:
            monkeypatch.setenv("SARAS_NO_TILE", "1")
        m = S.Multigrid(g, S.mg_params(**kw))
        m.set_graphs(graphs and tile)
        x, st, _ = m.solve(np.zeros_like(b), b)
        if graphs:   # replays
            x, st, _ = m.solve(np.zeros_like(b), b)
        out.append((x, st["residual"], st["cycles"]))
    np.testing.assert_array_equal(out[0][0], out[1][0])
    assert out[0][1:] == out[1][1:]
