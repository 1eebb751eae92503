"""Time steps on what the caller changed after cd3d_tcd_init: mass matrices set
entry by entry and per-point coefficients.  Both forms against the FP64 one on
the CSR matrices (CD3D_FP64_LATTICE=0): every solve stops at 1e-10 of its
residual and the matrices M + tau theta A have condition numbers below 100, so
the states agree to 1e-8."""
import numpy as np
import pytest

import parmoon_cmg_amd as pm

pytestmark = pytest.mark.gpu

CO = dict(eps=1e-3, conv_kind=1, rot_c=(0.45, 0.55), pulse_c=(0.3, 0.5, 0.5), f_val=0.7)


def states(order, m, levels, change, monkeypatch):
    """The state after a step, a change of the handle's data and two steps: FP64 on CSR, FP64, mixed."""
    out = []
    for lattice, prec in (("0", pm.FP64), ("1", pm.FP64), ("1", pm.MIXED)):
        monkeypatch.setenv("CD3D_FP64_LATTICE", lattice)
        P = pm.Problem(order, m, 0, levels, box=(1.0, 1.0, 1.0))
        co = pm.coeffs(**CO)
        sp = pm.solver_params(omega=0.5, pre=3, post=3, rel_tol=1e-10, precision=prec)
        P.tcd_init(co, 0.1, P.interp_pulse(levels - 1, co))
        P.tcd_step(co, sp, 2e-3, theta=0.7)
        change(P)
        for _ in range(2):
            u, _ = P.tcd_step(co, sp, 2e-3, theta=0.7)
        out.append(u)
        P.close()
    return out


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


# on every level, on the finest alone and on a level below it
@pytest.mark.parametrize("order,m,levels,which", [(1, 2, 3, (0, 1, 2)), (1, 3, 3, (2,)), (2, 2, 3, (0, 1, 2)), (2, 2, 3, (1,))])
def test_mass_matrix_set_by_the_caller(order, m, levels, which, monkeypatch):
    def change(P):
        for l in which:
            i = P.info(l)
            rp, _, e = P.csr(l)
            e[:rp[i["nact"]]] *= 1.5
            P.set_entries(l, e)

    ref, u64, u32 = states(order, m, levels, change, monkeypatch)
    plain = states(order, m, levels, lambda P: None, monkeypatch)[0]
    print(f"[gpu] mass set on {which}: FP64 {rel(u64, ref):.1e}, mixed {rel(u32, ref):.1e}, effect {rel(plain, ref):.1e}",
          flush=True)
    if levels - 1 in which:
        assert rel(plain, ref) > 1e-4  # the change is seen
    assert rel(u64, ref) < 1e-8 and rel(u32, ref) < 1e-8


# the values of a callback at the quadrature points, set after cd3d_tcd_init on
# every level, on the finest alone, on the coarsest alone
@pytest.mark.parametrize("order,m,levels,which", [(1, 2, 3, (0, 1, 2)), (1, 3, 2, (1,)), (2, 2, 2, (0, 1)), (2, 2, 3, (0,))])
def test_point_coefficients_set_by_the_caller(order, m, levels, which, monkeypatch):
    def change(P):
        for l in which:
            x = P.quad_points(l)
            q = np.zeros(x.shape[:-1] + (6,))
            q[..., 0] = 2e-3
            q[..., 1] = -(x[..., 1] - 0.45)
            q[..., 2] = x[..., 0] - 0.55
            q[..., 3] = 0.3 * x[..., 2]
            q[..., 4] = 0.5 * x[..., 0]
            q[..., 5] = 1.0 + x[..., 1]
            P.set_coeffs_qp(l, q)

    ref, u64, u32 = states(order, m, levels, change, monkeypatch)
    print(f"[gpu] points set on {which}: FP64 {rel(u64, ref):.1e}, mixed {rel(u32, ref):.1e}", flush=True)
    assert rel(u64, ref) < 1e-8 and rel(u32, ref) < 1e-8
