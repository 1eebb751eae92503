"""The cell-by-cell element kernels evaluate coefficients and geometry once
per point of a block's cells.  A block starts at any row of a cell, so blocks
touch different numbers of cells: meshes with less than one block, with a
short last one and with several, in cell order (the two passes) and through
colour lists (the scatter).  Both add the same element matrices in the same
order, so the same bits; one level against the float64 oracle at the bound of
the parity suite is in test_gpu_parity.py."""
import numpy as np
import pytest

import parmoon_cmg_amd as pm

pytestmark = pytest.mark.gpu

FORMS = {
    "rot_supg": dict(eps=1e-2, conv_kind=1, supg=1, t=0.3),
    "rot_manufactured": dict(eps=0.5, conv_kind=1, f_kind=1, c=0.25, t=0.1),
    "const_manufactured_supg": dict(eps=0.05, b=(1.0, -0.5, 0.25), f_kind=1, c=0.5, supg=1),
    "points_supg": dict(supg=1),
}


@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("order,m,mapped", [(1, 1, 0), (1, 3, 0), (1, 4, 1), (2, 1, 0), (2, 2, 1), (2, 3, 0), (2, 3, 1)])
def test_points_of_a_block(order, m, mapped, form, monkeypatch):
    box = (1.0, 0.8, 0.6)
    v = None
    if mapped:
        g = np.arange(m + 1) / m
        z, y, x = np.meshgrid(g, g, g, indexing="ij")
        s = 0.05 * np.sin(np.pi * x) * np.sin(np.pi * y) * np.sin(np.pi * z) + 0.03 * x * y
        v = np.stack([x * box[0] + s, y * box[1] - s, z * box[2] + s], axis=-1).reshape(-1, 3)
    monkeypatch.setenv("CD3D_CELLWISE_ASSEMBLY", "1")
    out = []
    for scatter in ("0", "1"):
        monkeypatch.setenv("CD3D_ASM_SCATTER", scatter)
        P = pm.Problem(order, m, 1, 2, box=box, vertices=v)
        for l in range(2):
            if form == "points_supg":
                x = P.quad_points(l)
                shape = x.shape[:-1]
                q = np.empty(shape + (6,))
                q[..., 0] = 0.01 + 0.1 * x[..., 0]
                q[..., 1] = 1.0 - x[..., 1]
                q[..., 2] = x[..., 0] - 0.5
                q[..., 3] = 0.25
                q[..., 4] = 0.5 * x[..., 2]
                q[..., 5] = 1.0 + x[..., 1]
                P.set_coeffs_qp(l, q)
        P.assemble(pm.coeffs(**FORMS[form]))
        out.append([(P.csr(l)[2], P.rhs(l)) for l in range(2)])
        P.close()
    for (e0, r0), (e1, r1) in zip(*out):
        assert np.isfinite(e0).all() and np.isfinite(r0).all()
        assert np.array_equal(e0, e1) and np.array_equal(r0, r1)
