"""SOR and SSOR divide by a_ii in both schedules: on diagonal matrices a row's
sum is exactly zero, so the sweeps with the iterate in LDS and those over the
schedule in memory (CD3D_GS_LDS=0) agree bitwise."""
import numpy as np
import pytest

import parmoon_cmg_amd as pm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", [2, 3])
@pytest.mark.parametrize("order,m,levels", [(1, 3, 3), (2, 2, 2)])
def test_diagonal_matrices_bitwise(order, m, levels, kind, monkeypatch):
    out = []
    for lds in ("1", "0"):
        monkeypatch.setenv("CD3D_GS_LDS", lds)
        rng = np.random.default_rng(8)
        P = pm.Problem(order, m, 0, levels)
        P.assemble(pm.coeffs(eps=1.0, f_val=1.0))
        for l in range(levels):
            rp, kc, e = P.csr(l)
            row = np.repeat(np.arange(len(rp) - 1), np.diff(rp))
            e = np.where(kc == row, 1.0 + rng.random(len(e)), 0.0)
            e[rp[P.info(l)["nact"]]:] = 1.0  # identity rows
            P.set_entries(l, e)
        r = rng.standard_normal(P.info(levels - 1)["ndof"])
        out.append(P.vcycle(pm.solver_params(smoother=kind, pre=2, post=1, omega=1.3), r))
        P.close()
    assert np.isfinite(out[0]).all() and np.array_equal(out[0], out[1])
