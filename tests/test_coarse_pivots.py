"""Pivots off the diagonal in the coarse inverse above 216 unknowns: two to
five and eight rows of the panel per thread, so that the largest entry is
found among several rows of a lane.  One entry off the diagonal dominates
every row.  Elimination with partial pivoting and an explicit inverse of n
unknowns: |A z - r| / |r| of order n eps cond (1-norm), with 10 for the growth."""
import numpy as np
import pytest

import parmoon_cmg_amd as pm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order,m,na", [(1, 9, 512), (1, 10, 729), (2, 6, 1331), (1, 13, 1728), (1, 14, 2197), (1, 15, 2744)])
def test_off_diagonal_pivots(order, m, na):
    P = pm.Problem(order, m, 0, 1, box=(1.0, 0.8, 0.6))
    assert P.info(0)["nact"] == na
    P.assemble(pm.coeffs(eps=1e-3, b=(1.0, -0.4, 0.3), c=0.5, supg=1, f_val=1.0))
    rp, kc, e = P.csr(0)
    row = np.repeat(np.arange(len(rp) - 1), np.diff(rp))
    act = (row < na) & (kc < na)
    for k in range(na):
        s = np.arange(rp[k], rp[k + 1])
        off = s[(kc[s] < na) & (kc[s] != k)]
        e[off[(7 * k) % len(off)]] += 3 * np.abs(e[s]).sum()
    P.set_entries(0, e)
    A = np.zeros((na, na))
    A[row[act], kc[act]] = e[act]
    assert (np.argmax(np.abs(A), axis=1) != np.arange(na)).all()
    cond = np.linalg.norm(A, 1) * np.linalg.norm(np.linalg.inv(A), 1)
    r = np.random.default_rng(5).standard_normal(P.info(0)["ndof"])
    r[na:] = 0.0
    z = P.vcycle(pm.solver_params(coarse_smoother=17), r)[:na]
    res = np.linalg.norm(A @ z - r[:na]) / np.linalg.norm(r[:na])
    print(f"[gpu] pivots na={na}: residual {res:.1e}, condition {cond:.1e}", flush=True)
    assert res < 10 * na * np.finfo(float).eps * cond
    P.close()
