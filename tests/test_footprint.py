"""The admission estimate against the memory a handle really takes: solvers
with row schedules (SOR, SSOR, multicolour SSOR), handles that have done a
lattice product, cell-by-cell assembly, time steps.  What a served request
reserves is what a simulated server accounts for it."""
import pytest

import parmoon_cmg_amd as pm

CO = dict(eps=0.05, b=(1.0, 0.5, 0.25), supg=1, f_val=1.0)
ROT = dict(eps=1e-3, conv_kind=1, rot_c=(0.45, 0.55), pulse_c=(0.3, 0.5, 0.5), f_val=0.7)


def reservation(mesh, co, sp, **kw):
    srv = pm.Server(hbm_budget=1 << 40, simulate=True, sim_us_per_dof=0.0)
    r, _ = srv.wait(srv.submit(pm.mesh_desc(*mesh), pm.coeffs(**co), sp, **kw))
    srv.close()
    return r.device_bytes


def test_reservation_counts_the_row_schedules():
    # Q2 m = 5, 2 levels: 19^3 unknowns above the coarsest level, 128 entries
    # of 16 bytes per row
    mesh = (2, 5, 0, 2)
    jac = reservation(mesh, CO, pm.solver_params())
    assert jac == pm.estimate_bytes(pm.mesh_desc(*mesh))
    assert reservation(mesh, CO, pm.solver_params(smoother=3)) - jac >= 19 ** 3 * 128 * 16
    # Q1 32^3: too large for the packed schedule
    mesh = (1, 1, 2, 4)
    extra = reservation(mesh, CO, pm.solver_params(smoother=3)) - reservation(mesh, CO, pm.solver_params())
    assert 31 ** 3 * 8 <= extra <= 31 ** 3 * 8 + 16 ** 3 * 600
    assert reservation(mesh, CO, pm.solver_params(smoother=13)) > reservation(mesh, CO, pm.solver_params())
    assert reservation(mesh, CO, pm.solver_params(maxit=1000)) == reservation(mesh, CO, pm.solver_params(smoother=13))


@pytest.mark.gpu
@pytest.mark.parametrize("smoother", [1, 2, 3, 13])
@pytest.mark.parametrize("mesh", [(2, 5, 0, 2), (1, 5, 0, 3), (1, 1, 2, 4), (2, 3, 0, 4)])
def test_solve_stays_within_the_reservation(mesh, smoother):
    sp = pm.solver_params(smoother=smoother, omega=0.5 if smoother == 1 else 1.0, maxit=20)
    P = pm.Problem(*mesh)
    P.assemble(pm.coeffs(**CO))
    x, _ = P.solve(sp, check=False)
    P.matvec(mesh[3] - 1, x)
    sp.precision = pm.MIXED
    P.solve(sp, check=False)
    used, est = P.L.cd3d_device_bytes(P.h), reservation(mesh, CO, sp)
    print(f"[gpu] {mesh} smoother {smoother}: device bytes {used / 2**20:.1f} MiB, reserved {est / 2**20:.1f}", flush=True)
    assert used <= est
    P.close()


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["FP64", "MIXED"])
@pytest.mark.parametrize("mesh", [(1, 5, 0, 3), (2, 3, 0, 3), (2, 3, 0, 4), (1, 3, 0, 5)])
def test_cellwise_solve_stays_within_the_reservation(mesh, prec):
    co = dict(CO, f_kind=1)
    sp = pm.solver_params(omega=0.5, maxit=20, precision=getattr(pm, prec))
    P = pm.Problem(*mesh)
    for c in (co, dict(ROT, supg=1)):  # both kinds of request the estimate takes for cell by cell
        P.assemble(pm.coeffs(**c))
        P.solve(sp, check=False)
    used, est = P.L.cd3d_device_bytes(P.h), reservation(mesh, co, sp)
    print(f"[gpu] {mesh} {prec}: device bytes {used / 2**20:.1f} MiB, reserved {est / 2**20:.1f}", flush=True)
    # 2 MiB per level of granularity; nothing that is not there (4 bytes per nonzero are 8 %)
    assert used <= est <= 1.06 * used + 2 * mesh[3] * 2**20
    P.close()


@pytest.mark.gpu
@pytest.mark.parametrize("supg", [0, 1])
@pytest.mark.parametrize("mesh", [(1, 5, 0, 3), (2, 3, 0, 4)])
def test_time_steps_stay_within_the_reservation(mesh, supg):
    sp = pm.solver_params(omega=0.5, rel_tol=1e-8)
    P = pm.Problem(*mesh)
    co = pm.coeffs(**dict(ROT, supg=supg))
    for prec in (pm.FP64, pm.MIXED):
        sp.precision = prec
        P.tcd_init(co, 0.0, P.interp_pulse(mesh[3] - 1, co))
        P.tcd_step(co, sp, 1e-3)
    used = P.L.cd3d_device_bytes(P.h)
    est = reservation(mesh, dict(ROT, supg=supg), sp, kind=pm.REQ_TCD, nsteps=1)
    print(f"[gpu] {mesh} time steps supg={supg}: device bytes {used / 2**20:.1f} MiB, reserved {est / 2**20:.1f}", flush=True)
    assert used <= est
    P.close()


@pytest.mark.gpu
def test_mixed_batch_stays_within_the_reservation():
    meshes = [(1, 5, 0, 3), (2, 3, 0, 3)]
    sp = pm.solver_params(omega=0.5, precision=pm.MIXED)
    Ps = [pm.Problem(*m) for m in meshes]
    for P in Ps:
        P.assemble(pm.coeffs(**CO))
    pm.solve_batch(Ps, sp)
    for m, P in zip(meshes, Ps):
        used, est = P.L.cd3d_device_bytes(P.h), reservation(m, CO, sp)
        print(f"[gpu] {m} mixed batch: device bytes {used / 2**20:.1f} MiB, reserved {est / 2**20:.1f}", flush=True)
        assert used <= est
        P.close()
