"""rfinal of a solve that ran on the class stencils is |b - A x| of the
assembled CSR matrix: bitwise the r0 of a solve started from its solution on
the CSR matrices (CD3D_FP64_LATTICE=0), which forms b - A x the same way."""
import pytest

import parmoon_cmg_amd as pm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["FP64", "MIXED"])
@pytest.mark.parametrize("order,m,levels,conv", [(2, 3, 3, 0), (1, 5, 3, 1), (1, 2, 2, 0)])
def test_residual_of_the_assembled_matrix(order, m, levels, conv, prec, monkeypatch):
    P = pm.Problem(order, m, 0, levels, box=(1.0, 0.7, 0.5))
    P.assemble(pm.coeffs(eps=0.05, b=(1.0, 0.5, 0.25), c=0.3, conv_kind=conv, f_val=1.0))
    x, st = P.solve(pm.solver_params(precision=getattr(pm, prec), rel_tol=1e-6))
    monkeypatch.setenv("CD3D_FP64_LATTICE", "0")
    _, again = P.solve(pm.solver_params(maxit=1, rel_tol=0.9), x0=x, check=False)
    print(f"[gpu] rfinal {st.rfinal:.17e}, r0 from there {again.r0:.17e}", flush=True)
    assert st.rfinal == again.r0
    P.close()
