"""The finest level's vectors 0 and 1 (cd3d_device_ptr) after a V-cycle of the
FP64 form: z and r in DOF order, with the lattice form and with the CSR one.
Vector 0 is read with cd3d_get_solution, vector 1 through a product."""
import numpy as np
import pytest

import parmoon_cmg_amd as pm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lattice", ["1", "0"])
@pytest.mark.parametrize("order,m,levels,post", [(1, 3, 2, 1), (1, 3, 3, 0), (2, 2, 3, 2)])
def test_vectors_after_a_vcycle(order, m, levels, post, lattice, monkeypatch):
    monkeypatch.setenv("CD3D_FP64_LATTICE", lattice)
    P = pm.Problem(order, m, 0, levels, box=(1.0, 0.8, 0.6))
    P.assemble(pm.coeffs(eps=0.05, b=(1.0, 0.5, 0.25), supg=1, f_val=1.0))
    l = levels - 1
    i = P.info(l)
    r = np.random.default_rng(4).standard_normal(i["ndof"])
    r[i["nact"]:] = 0.0
    z = P.vcycle(pm.solver_params(omega=0.5, pre=2, post=post), r)
    assert np.array_equal(P.solution(), z)
    P.matvec_dev(l, P.device_ptr(l, 1), P.device_ptr(l, 0))
    assert np.array_equal(P.solution(), P.matvec(l, r))
    P.close()
