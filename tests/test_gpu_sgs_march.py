"""The marching sub-grid stress kernel (k_sgs_stress) against the FP64 CPU oracle
where its blocks are part-filled: rows shorter than a block, longer by a
remainder and of several blocks, row counts that are no multiple of its four,
one chunk of planes and several.  The
stage right-hand side and the diagnostics are held to 1e-9 of the largest value
(double-precision integral) and 1e-6 (single), the bars of the 16^3 comparison.
"""
import numpy as np
import pytest

import oracle as O
from test_gpu_nse import mg_kw, pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sf32,rtol", [(0, 1e-9), (1, 1e-6)], ids=["f64", "f32"])
@pytest.mark.parametrize("n", [(4, 4, 8), (8, 6, 72), (36, 10, 16), (8, 12, 136)], ids=lambda n: "x".join(map(str, n)))
def test_matches_oracle(n, sf32, rtol):
    so, ss = pair(n, periodic=(1, 1, 1), gtype=(0, 0, 0), pad=2, has_T=0, nu=1.0 / 1600, dt=1e-3, cn_tol=1e-10, les=1,
                  mg=mg_kw(vc_count=2, vc_tol=1e-10, pre=2, post=2), gpu_kw={"les_sf32": sf32})
    rng = np.random.default_rng(23)
    sh = so.shape
    z = np.zeros(sh)
    x, y, w = np.meshgrid(*[2 * np.pi * (np.arange(-2, m + 2) + 0.5) / m for m in n], indexing="ij")
    f = dict(vx=np.sin(x) * np.cos(y) * np.cos(w) + 0.1 * rng.uniform(-1, 1, sh),
             vy=-np.cos(x) * np.sin(y) * np.cos(w) + 0.1 * rng.uniform(-1, 1, sh), vz=0.1 * rng.uniform(-1, 1, sh),
             p=z, t=z, pp=z)
    so.set(**f)
    ss.set(**f)
    for _ in range(6):   # the steps before the model enters
        assert so.step() == 0
        assert ss.step()[0] == 0
    f = so.get()
    ss.set(**f)
    c = (slice(2, -2),) * 3
    ro, rs = so.rhs(0), ss.rhs(0)
    for k in ("rx", "ry", "rz", "hx", "hy", "hz"):
        a, b = ro[k][c], rs[k][c]
        assert np.abs(a - b).max() <= rtol * np.abs(a).max(), (k, np.abs(a - b).max())
    do = so.sgs_diag()
    dg, _ = ss.sgs()
    for q, k in enumerate(("sgke", "disp", "nusg")):
        assert abs(dg[k] - do[q]) <= rtol * abs(do[q]), (k, dg[k], do[q])
