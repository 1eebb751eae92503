"""SOR and SSOR sweeps with the iterate in LDS (packed schedule) against the
sweeps over the schedule in memory (CD3D_GS_LDS=0): the same rows in the same
order, so only the order of a row's sum (at most 124 terms, 1.4e-14 relative)
and the product with 1/a_ii (2 eps) differ; a V-cycle chains fewer than 20
sweeps: 1e-12.  A solve takes the same number of iterations."""
import numpy as np
import pytest

import parmoon_cmg_amd as pm

pytestmark = pytest.mark.gpu


# levels of one unknown, steps of one row and levels of more than 16 rows, the
# largest level that fits (Q1 20^3 cells) and one that does not (Q1 22^3, the
# levels below it do), Q2's 125-entry rows; 0 to 3 sweeps; nonzero starts (W
# cycles) and Dirichlet data
@pytest.mark.parametrize("order,m,k0,levels,kind,pre,post,cycle", [
    (1, 2, 0, 2, 2, 1, 1, 1), (1, 1, 2, 3, 3, 3, 3, 1), (1, 3, 0, 3, 2, 2, 1, 2), (1, 5, 0, 3, 3, 1, 0, 1),
    (1, 11, 0, 2, 3, 1, 1, 1), (2, 1, 1, 2, 3, 2, 2, 1), (2, 3, 0, 2, 2, 3, 1, 0), (2, 2, 0, 3, 3, 0, 2, 2)])
def test_packed_sweeps_match_schedule_in_memory(order, m, k0, levels, kind, pre, post, cycle, monkeypatch):
    out = []
    for lds in ("1", "0"):
        monkeypatch.setenv("CD3D_GS_LDS", lds)
        P = pm.Problem(order, m, k0, levels, box=(1.0, 0.7, 0.5))
        sp = pm.solver_params(smoother=kind, pre=pre, post=post, omega=1.1, cycle=cycle, rel_tol=1e-10, maxit=60)
        got = []
        for eps in (0.05, 1.0):  # the second assembly: new values in the same schedule
            P.assemble(pm.coeffs(eps=eps, b=(0.3, 0.4, -0.5), supg=1, f_val=1.0))
            r = np.random.default_rng(5).standard_normal(P.info(levels - 1)["ndof"])
            z1 = P.vcycle(sp, r)  # Dirichlet data
            r[P.info(levels - 1)["nact"]:] = 0.0
            x, st = P.solve(sp, check=False)
            got.append((z1, P.vcycle(sp, r), x, st.iterations, st.status))
        out.append(got)
        P.close()
    for a, b in zip(*out):
        assert a[3:] == b[3:]
        for u, v, tol in zip(a[:3], b[:3], (1e-12, 1e-12, 1e-10)):
            assert np.linalg.norm(u - v) <= tol * np.linalg.norm(v)
