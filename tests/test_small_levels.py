"""The one-workgroup program of the V-cycle's bottom levels where levels with
compact stencils and levels with per-node values meet: against the launched
sweeps (CD3D_SMALL_NODES=0), the same node code in the same order, so bitwise.
The host check of the same rule is test_small_levels_host.py."""
import numpy as np
import pytest

import parmoon_cmg_amd as pm

pytestmark = pytest.mark.gpu


def check(P, levels, monkeypatch):
    i = P.info(levels - 1)
    r = np.random.default_rng(3).standard_normal(i["ndof"])
    r[i["nact"]:] = 0.0
    sp = pm.solver_params(omega=0.5, pre=2, post=3, rel_tol=1e-10, maxit=60, precision=pm.MIXED)
    out = []
    for bound in ("3000", "0"):
        monkeypatch.setenv("CD3D_SMALL_NODES", bound)
        x, st = P.solve(sp, check=False)
        out.append((P.vcycle(sp, r), x, st.iterations, st.status))
    assert np.isfinite(out[0][0]).all() and out[0][2:] == out[1][2:]
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])


# rotating field with SUPG: the 3^3-node level holds one unknown and counts as
# uniform, the levels above it vary
@pytest.mark.parametrize("order,levels", [(1, 3), (1, 4), (2, 3)])
def test_one_unknown_below_varying_levels(order, levels, monkeypatch):
    P = pm.Problem(order, 1, 0, levels, box=(1.0, 0.9, 0.8))
    P.assemble(pm.coeffs(eps=0.05, conv_kind=1, rot_c=(0.4, 0.6), supg=1, f_val=1.0))
    check(P, levels, monkeypatch)
    P.close()


# entries set by the caller on one level of a constant-coefficient hierarchy
@pytest.mark.parametrize("order,m,levels,level", [(1, 2, 3, 2), (1, 2, 3, 1), (2, 1, 3, 1)])
def test_entries_set_on_one_level(order, m, levels, level, monkeypatch):
    P = pm.Problem(order, m, 0, levels, box=(1.0, 0.9, 0.8))
    P.assemble(pm.coeffs(eps=0.05, b=(1.0, 0.5, 0.25), supg=1, f_val=1.0))
    e = P.csr(level)[2]
    P.set_entries(level, e * (1.0 + 0.05 * np.random.default_rng(7).uniform(-1, 1, len(e))))
    check(P, levels, monkeypatch)
    P.close()
