"""Calls that find no device memory for buffers they can do without take the
form that needs none: row-order sweeps over the schedule in memory, FGMRES in
DOF order, MGS vector by vector.  The handle's allocations are bounded from the
host (cd3d_internal_alloc_limit)."""
import ctypes as C

import numpy as np
import pytest

import parmoon_cmg_amd as pm

pytestmark = pytest.mark.gpu

CO = dict(eps=0.05, b=(0.3, 0.4, -0.5), supg=1, f_val=1.0)
RESTART = 12


def bound(P, extra):
    """At most `extra` bytes more than the handle holds now."""
    P.L.cd3d_internal_alloc_limit.argtypes = [C.c_void_p, C.c_size_t]
    P.L.cd3d_internal_alloc_limit(P.h, P.L.cd3d_device_bytes(P.h) + extra)


def krylov_bytes(P, held_restart=None):
    """The Krylov space of RESTART columns on a handle that has that of held_restart."""
    n = P.info(P.levels - 1)["ndof"]
    ld = (n + 31) // 32 * 32
    if held_restart is None:
        return 8 * (2 * (RESTART + 1) * ld + 3 * n)
    return 8 * 2 * (RESTART - held_restart) * ld


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("order,m,kind", [(1, 5, 3), (2, 2, 2)])
def test_row_order_sweeps(order, m, kind, monkeypatch):
    sp = pm.solver_params(smoother=kind, omega=1.0, pre=2, post=2, rel_tol=1e-10, maxit=60, restart=RESTART)
    out = []
    for scarce in (False, True):
        monkeypatch.setenv("CD3D_GS_LDS", "1" if scarce else "0")
        P = pm.Problem(order, m, 0, 2)
        P.assemble(pm.coeffs(**CO))
        if scarce:  # the Krylov space, Gram-Schmidt buffers and 8 bytes per row, not 500
            bound(P, krylov_bytes(P) + 65536 + 64 * P.info(1)["ndof"])
        x, st = P.solve(sp, check=False)
        out.append((x, st.iterations, st.status))
        P.close()
    assert out[0][1:] == out[1][1:] and np.array_equal(out[0][0], out[1][0])


# iteration counts: the lattice form's and the CSR form's agree (test_lattice_fp64.py)
@pytest.mark.parametrize("prec", ["FP64", "MIXED"])
@pytest.mark.parametrize("conv", [0, 1])
def test_solve_without_lattice_vectors(conv, prec):
    sp = pm.solver_params(omega=0.5, pre=3, post=3, rel_tol=1e-10, restart=RESTART, precision=getattr(pm, prec))
    out = []
    for scarce in (False, True):
        P = pm.Problem(1, 5, 0, 3)
        P.assemble(pm.coeffs(**dict(CO, conv_kind=conv, supg=0)))
        if scarce:
            bound(P, krylov_bytes(P))
        x, st = P.solve(sp)
        out.append((x, st.iterations))
        P.close()
    assert out[0][1] == out[1][1] and rel(out[1][0], out[0][0]) < 1e-9


@pytest.mark.parametrize("prec", ["FP64", "MIXED"])
def test_time_steps_without_lattice_vectors(prec, monkeypatch):
    monkeypatch.setenv("CD3D_SMALL_NODES", "0")  # no per-node values of the small levels, which the mixed form needs
    sp = pm.solver_params(omega=0.5, pre=3, post=3, rel_tol=1e-10, restart=RESTART, precision=getattr(pm, prec))
    co = pm.coeffs(eps=1e-3, conv_kind=1, rot_c=(0.45, 0.55), pulse_c=(0.3, 0.5, 0.5), f_val=0.7)
    out = []
    for scarce in (False, True):
        P = pm.Problem(1, 5, 0, 3)
        P.assemble(pm.coeffs(**CO))
        P.tcd_init(co, 0.1, P.interp_pulse(2, co))
        if scarce:
            bound(P, krylov_bytes(P, 1))
        out.append([P.tcd_step(co, sp, 2e-3)[0] for _ in range(2)][-1])
        P.close()
    assert rel(out[1], out[0]) < 1e-9


def test_batch_without_gram_schmidt_buffers():
    sp = pm.solver_params(omega=0.5, pre=3, post=3, rel_tol=1e-10, restart=RESTART)
    out = []
    for scarce in (False, True):
        Ps = [pm.Problem(1, m, 0, 3) for m in (2, 3)]
        for P in Ps:
            P.assemble(pm.coeffs(**CO))
        if scarce:
            bound(Ps[1], krylov_bytes(Ps[1]))
        its = [s.iterations for s in pm.solve_batch(Ps, sp)]
        out.append((its, [P.solution() for P in Ps]))
        for P in Ps:
            P.close()
    assert out[0][0] == out[1][0]
    for a, b in zip(out[0][1], out[1][1]):
        assert rel(b, a) < 1e-9
