"""The cell-by-cell element kernels against the float64 oracle, entry by entry,
where test_element_points.py compares their two ways out: blocks that start
inside a cell, a short last block, less than one block, bricks and hexahedra,
coefficients that vary over a cell, and the mass matrix.  The bound is the
parity suite's: 1e-12 of a row's largest entry, 1e-12 of the largest rhs."""
import numpy as np
import pytest

import parmoon_cmg_amd as pm
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

TOL = 1e-12
FORMS = {
    "const_supg": dict(eps=0.05, b=(1.0, -0.5, 0.25), c=0.5, supg=1, f_val=0.7),
    "rot_supg": dict(eps=1e-2, conv_kind=1, supg=1, t=0.3, f_val=1.0),
    "rot_manufactured": dict(eps=0.5, conv_kind=1, f_kind=1, c=0.25, t=0.1),
    "const_manufactured_supg": dict(eps=0.05, b=(1.0, -0.5, 0.25), f_kind=1, c=0.5, supg=1),
    "points_supg": dict(supg=1),
}
BOX = (1.0, 0.8, 0.6)


def row_scaled_err(e, er, rp):
    rowmax = np.maximum.reduceat(np.abs(er), rp[:-1])
    return (np.abs(e - er) / np.repeat(rowmax, np.diff(rp))).max()


def vertices(m):
    g = np.arange(m + 1) / m
    z, y, x = np.meshgrid(g, g, g, indexing="ij")
    s = 0.05 * np.sin(np.pi * x) * np.sin(np.pi * y) * np.sin(np.pi * z) + 0.03 * x * y
    return np.stack([x * BOX[0] + s, y * BOX[1] - s, z * BOX[2] + s], axis=-1).reshape(-1, 3)


def point_values(x):
    q = np.empty(x.shape[:-1] + (6,))
    q[..., 0] = 0.01 + 0.1 * x[..., 0]
    q[..., 1] = 1.0 - x[..., 1]
    q[..., 2] = x[..., 0] - 0.5
    q[..., 3] = 0.25
    q[..., 4] = 0.5 * x[..., 2]
    q[..., 5] = 1.0 + x[..., 1]
    return q


@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("order,m,mapped", [(1, 1, 0), (1, 3, 0), (1, 3, 1), (2, 1, 0), (2, 1, 1), (2, 2, 0), (2, 2, 1)])
def test_entries_and_rhs(order, m, mapped, form, monkeypatch):
    monkeypatch.setenv("CD3D_CELLWISE_ASSEMBLY", "1")
    v = vertices(m) if mapped else None
    P, H = pm.Problem(order, m, 1, 2, box=BOX, vertices=v), po.Hierarchy(order, m, 1, 2, box=BOX, vertices=v)
    if form == "points_supg":
        for l in range(2):
            q = point_values(H.quad_points(l))
            P.set_coeffs_qp(l, q)
            H.set_coeffs_qp(l, q)
    kw = FORMS[form]
    P.assemble(pm.coeffs(**kw))
    for l in range(2):
        rp, _, e = P.csr(l)
        eo, ro = H.assemble_level(l, po.coeffs(**kw), 0)
        err, rerr = row_scaled_err(e, eo, rp), np.abs(P.rhs(l) - ro).max() / np.abs(ro).max()
        print(f"[gpu] element values Q{order} m={m} mapped={mapped} {form} level {l}: {err:.1e} rhs {rerr:.1e}", flush=True)
        assert err < TOL and rerr < TOL
    # the mass matrices of time steps, through the same kernels
    t = kw.get("t", 0.0)
    P.tcd_init(pm.coeffs(**kw), t, np.zeros(P.info(1)["ndof"]))
    for l in range(2):
        rp, _, e = P.csr(l)
        err = row_scaled_err(e, H.assemble_level(l, po.coeffs(**kw), 1)[0], rp)
        print(f"[gpu]   mass level {l}: {err:.1e}", flush=True)
        assert err < TOL
    P.close()
