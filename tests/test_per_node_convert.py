"""Per-node FP32 stencils transposed from the CSR values, tile by tile of 64
nodes of a class: classes of less than one tile, of exactly one and with a
remainder.  The mixed V-cycle against the FP64 one on the same matrices: FP32
products of at most 125 terms in a chain of fewer than 14 products with O(1)
factors, 14 * 125 * 2^-24 = 1e-4; a value in the wrong place is off by the size
of the perturbation, 5 %."""
import numpy as np
import pytest

import parmoon_cmg_amd as pm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order,m", [(1, 1), (1, 5), (1, 9), (2, 1), (2, 2), (2, 4), (2, 5)])
def test_mixed_cycle_on_per_node_stencils(order, m, monkeypatch):
    monkeypatch.setenv("CD3D_SMALL_NODES", "0")  # the launched sweeps, not the one-workgroup program
    P = pm.Problem(order, m, 0, 2, box=(1.0, 0.8, 0.6))
    P.assemble(pm.coeffs(eps=0.1, b=(1.0, -0.5, 0.25), c=0.5, f_val=1.0))
    rng = np.random.default_rng(7)
    for l in (0, 1):
        e = P.csr(l)[2]
        P.set_entries(l, e * (1.0 + 0.05 * rng.uniform(-1, 1, len(e))))
    i = P.info(1)
    r = rng.standard_normal(i["ndof"])
    r[i["nact"]:] = 0.0
    z64 = P.vcycle(pm.solver_params(precision=pm.FP64), r)
    z32 = P.vcycle(pm.solver_params(precision=pm.MIXED), r)
    err = np.linalg.norm(z32 - z64) / np.linalg.norm(z64)
    print(f"[gpu] per-node stencils Q{order} {2 * m}^3: mixed against FP64 cycle {err:.1e}", flush=True)
    assert err < 1e-4
    P.close()
