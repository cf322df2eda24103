"""Tiles (k_tile) on thin periodic axes, whose last tile covers more rows than the
level's images: the FP64 solve against the CPU oracle and the FP32 cycles against
one launch per pass, bit for bit.
"""
import numpy as np
import pytest

import oracle as O
import saras_amd as S
from test_gpu_mg_tile import rhs

pytestmark = pytest.mark.gpu

CASES = [
    # n, periodic, (pre, post)
    ((512, 10, 32), (0, 1, 0), (2, 2)),     # y tiles of 8 rows of 10, halo 5
    ((192, 6, 64), (0, 1, 0), (3, 3)),      # y tiles of 4 rows of 6, halo 6
    ((512, 12, 16), (1, 1, 0), (3, 6)),     # y tiles of 8 rows of 12, halo 12
    ((6, 512, 44), (1, 0, 1), (3, 3)),      # x tiles of 4 rows of 6, halo 6
    ((12, 20, 44), (1, 1, 1), (3, 6)),      # rows of 22 pairs
]
IDS = [f"{'x'.join(map(str, n))}-p{''.join(map(str, p))}-v{v[0]}{v[1]}" for n, p, v in CASES]


@pytest.mark.parametrize("n,per,sweeps", CASES, ids=IDS)
def test_fp64_bitexact(n, per, sweeps):
    print(n, per, sweeps, "fp64", flush=True)
    kw = dict(vc_count=2, vc_tol=1e-14, mg_tol=1e-2, pre=sweeps[0], post=sweeps[1], solve_flag=0)
    go, gs = O.grid_desc(n, periodic=per), S.grid_desc(n, periodic=per)
    mo, ms = O.Multigrid(go, O.mg_params(bc=O.BC_NEUMANN, **kw)), S.Multigrid(gs, S.mg_params(bc=S.BC_NEUMANN, **kw))
    rng = np.random.default_rng(51)
    b, x0 = rhs(go, rng, True), rhs(go, rng, False) * 0.1
    xo, so = mo.solve(x0.copy(), b, 1)
    xs, ss, _ = ms.solve(x0.copy(), b)
    assert ss["residual"] == so["residual"]
    np.testing.assert_array_equal(xs, xo)


@pytest.mark.parametrize("n,per,sweeps", CASES, ids=IDS)
def test_fp32_matches_passes(n, per, sweeps, monkeypatch):
    print(n, per, sweeps, "fp32", flush=True)
    kw = dict(vc_count=6, vc_tol=1e-14, mg_tol=1e-6, pre=sweeps[0], post=sweeps[1], precision=S.PREC_MIXED,
              inner_cycles=3, max_refine=2, solve_flag=0, bc=S.BC_NEUMANN)
    b = rhs(O.grid_desc(n, periodic=per), np.random.default_rng(52), True)
    out = []
    for tile in (True, False):
        if not tile:
            monkeypatch.setenv("SARAS_NO_TILE", "1")
        x, st, _ = S.Multigrid(S.grid_desc(n, periodic=per), S.mg_params(**kw)).solve(np.zeros_like(b), b)
        out.append((x, st["residual"]))
    np.testing.assert_array_equal(out[0][0], out[1][0])
    assert out[0][1] == out[1][1]
