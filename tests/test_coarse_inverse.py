"""The exact coarse solve (explicit inverse by Gauss-Jordan exchange steps) at
the edges of its forms: one thread tile and its remainders (1 to 128
unknowns), panels with a short last one, one to four rows per thread.  A
backward-stable elimination of n unknowns leaves |A z - r| / |r| of order
n eps cond; 1e-12 as in the parity suite."""
import numpy as np
import pytest

import parmoon_cmg_amd as pm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order,m,na", [(1, 2, 1), (1, 3, 8), (1, 5, 64), (2, 3, 125), (1, 7, 216), (1, 10, 729),
                                        (1, 11, 1000), (1, 13, 1728), (1, 14, 2197)])
def test_coarse_inverse_sizes(order, m, na):
    P = pm.Problem(order, m, 0, 1, box=(1.0, 0.8, 0.6))
    i = P.info(0)
    assert i["nact"] == na
    for conv in (0.0, 1.0):  # symmetric, then strongly nonsymmetric (pivots off the diagonal's order)
        P.assemble(pm.coeffs(eps=1e-3 if conv else 1.0, b=(conv, -0.4 * conv, 0.3 * conv), c=0.5 * conv, supg=int(conv),
                             f_val=1.0))
        r = np.random.default_rng(5).standard_normal(i["ndof"])
        r[na:] = 0.0
        z = P.vcycle(pm.solver_params(coarse_smoother=17), r)
        res = np.linalg.norm(P.matvec(0, z) - r) / np.linalg.norm(r)
        print(f"[gpu] coarse inverse na={na} conv={conv}: |A z - r| / |r| = {res:.2e}", flush=True)
        assert res < 1e-12
    # rows whose largest entry lies off the diagonal: a cyclic shift of the rows of A
    rp, kc, e = P.csr(0)
    d = np.zeros((na, na))
    for k in range(na):
        s = slice(rp[k], rp[k + 1])
        act = kc[s] < na
        d[k, kc[s][act]] = e[s][act]
    if na <= 216:
        big = e.copy()
        for k in range(na):  # one off-diagonal entry per row dominates where the row has any
            s = np.arange(rp[k], rp[k + 1])
            off = s[(kc[s] < na) & (kc[s] != k)]
            if len(off):
                big[off[k % len(off)]] += 3 * np.abs(d[k]).sum()
        P.set_entries(0, big)
        A = np.zeros((na, na))
        for k in range(na):
            s = slice(rp[k], rp[k + 1])
            act = kc[s] < na
            A[k, kc[s][act]] = big[s][act]
        z = P.vcycle(pm.solver_params(coarse_smoother=17), r)[:na]
        cond = np.linalg.cond(A)
        res = np.linalg.norm(A @ z - r[:na]) / np.linalg.norm(r[:na])
        print(f"[gpu] pivoting na={na}: residual {res:.2e}, condition {cond:.1e}", flush=True)
        # an explicit inverse's residual grows with the condition number; partial pivoting adds a growth factor
        assert res < 1e-13 * na * cond
    P.close()


@pytest.mark.parametrize("order,m,na", [(1, 9, 512), (2, 6, 1331), (1, 15, 2744)])
def test_coarse_inverse_rows_per_thread(order, m, na):
    """Panels with one row per thread and every thread used, with three, and
    the narrow ones of more than five; bound as above."""
    P = pm.Problem(order, m, 0, 1, box=(1.0, 0.8, 0.6))
    i = P.info(0)
    assert i["nact"] == na
    P.assemble(pm.coeffs(eps=1e-3, b=(1.0, -0.4, 0.3), c=0.5, supg=1, f_val=1.0))
    r = np.random.default_rng(5).standard_normal(i["ndof"])
    r[na:] = 0.0
    z = P.vcycle(pm.solver_params(coarse_smoother=17), r)
    res = np.linalg.norm(P.matvec(0, z) - r) / np.linalg.norm(r)
    print(f"[gpu] coarse inverse na={na}: |A z - r| / |r| = {res:.2e}", flush=True)
    assert res < 1e-12
    P.close()
