"""The plain FP64 form on the lattice (class stencils, lattice order) against
the same form on the CSR matrices (CD3D_FP64_LATTICE=0): the same matrices,
smoother and Krylov iteration in FP64, so only the order of the sums differs.
A product sums at most 125 terms (relative rounding <= 125 eps = 2.8e-14) and a
V-cycle chains fewer than 50 of them with O(1) factors: 2e-12 for the cycle;
a solve stops at 1e-10 of its residual after the same number of iterations,
and its solutions agree to that."""
import numpy as np
import pytest

import parmoon_cmg_amd as pm

pytestmark = pytest.mark.gpu

CYCLE_TOL, SOL_TOL = 2e-12, 1e-10


def both(monkeypatch, work):
    out = []
    for on in ("1", "0"):
        monkeypatch.setenv("CD3D_FP64_LATTICE", on)
        out.append(work())
    return out


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


# levels by class, by pairs (more than 40 nodes per side) and by quads (more
# than 2^17 pair groups); odd cells per side; V, W and F cycles; no pre- or
# post-smoothing; an odd number of sweeps; a coarse smoother other than the
# exact solve (the DOF-ordered coarse path)
@pytest.mark.parametrize("order,m,k0,levels,kw", [
    (1, 1, 1, 2, {}), (1, 3, 0, 4, {}), (1, 5, 0, 3, dict(cycle=2)), (1, 1, 2, 5, dict(pre=2, post=1)),
    (2, 1, 1, 2, {}), (2, 3, 0, 3, dict(cycle=0)), (2, 11, 0, 2, dict(pre=0, post=2)), (2, 1, 1, 5, dict(pre=2, post=0)),
    (2, 1, 2, 5, {}), (2, 3, 1, 5, dict(pre=1, post=2)), (2, 2, 0, 3, dict(coarse_smoother=3)),
    (1, 2, 0, 4, dict(coarse_smoother=1, cycle=2))])
def test_fp64_lattice_matches_csr(order, m, k0, levels, kw, monkeypatch):
    P = pm.Problem(order, m, k0, levels, box=(1.0, 0.7, 0.5))
    P.assemble(pm.coeffs(eps=0.05, b=(1.0, 0.5, 0.25), c=0.3, supg=1, f_val=1.0))
    i = P.info(levels - 1)
    r = np.random.default_rng(5).standard_normal(i["ndof"])
    r[i["nact"]:] = 0.0
    rhs = np.random.default_rng(6).standard_normal(i["ndof"])  # Dirichlet values among it
    sp = pm.solver_params(**dict(dict(omega=0.5, pre=3, post=3, rel_tol=1e-10, restart=7), **kw))
    (z1, x1, s1), (z0, x0, s0) = both(monkeypatch, lambda: (P.vcycle(sp, r), *P.solve(sp, rhs=rhs, check=False)))
    print(f"[gpu] fp64 lattice order={order} m={m} levels={levels} {kw}: cycle {rel(z1, z0):.1e}, its {s1.iterations} / "
          f"{s0.iterations}, solution {rel(x1, x0):.1e}", flush=True)
    assert rel(z1, z0) < CYCLE_TOL
    assert (s1.iterations, s1.status) == (s0.iterations, s0.status)
    assert rel(x1, x0) < SOL_TOL and np.array_equal(x1[i["nact"]:], rhs[i["nact"]:])
    # a solve after it that keeps the CSR form (entries set by the caller) finds nothing of the lattice vectors
    P.set_entries(levels - 1, P.csr(levels - 1)[2])
    monkeypatch.setenv("CD3D_FP64_LATTICE", "1")
    x2, s2 = P.solve(sp, rhs=rhs, check=False)
    assert np.array_equal(x2, x0) and s2.iterations == s0.iterations
    P.close()


@pytest.mark.parametrize("order,m,k0,levels,theta", [(1, 2, 1, 2, 0.5), (1, 3, 0, 4, 1.0), (2, 2, 0, 3, 0.5), (2, 3, 1, 3, 0.7)])
def test_fp64_lattice_time_steps_match_csr(order, m, k0, levels, theta, monkeypatch):
    P = pm.Problem(order, m, k0, levels, box=(1.0, 1.0, 1.0))
    co = pm.coeffs(eps=1e-3, conv_kind=1, rot_c=(0.45, 0.55), pulse_c=(0.3, 0.5, 0.5), f_val=0.7)
    sp = pm.solver_params(omega=0.5, pre=3, post=3, rel_tol=1e-10)
    u0 = P.interp_pulse(levels - 1, co)

    def steps():
        P.tcd_init(co, 0.1, u0)
        out = [P.tcd_step(co, sp, 2e-3, theta=theta) for _ in range(3)]
        return out[-1][0], [st.iterations for _, st in out]

    (u1, i1), (u0_, i0) = both(monkeypatch, steps)
    print(f"[gpu] fp64 lattice steps order={order}: its {i1} / {i0}, state {rel(u1, u0_):.1e}", flush=True)
    assert i1 == i0 and rel(u1, u0_) < SOL_TOL
    P.close()


def test_fp64_lattice_rotating_field_solve(monkeypatch):
    P = pm.Problem(1, 3, 0, 4, box=(1.0, 1.0, 1.0))
    P.assemble(pm.coeffs(eps=0.05, conv_kind=1, rot_c=(0.45, 0.55), f_val=1.0))
    sp = pm.solver_params(omega=0.5, pre=3, post=3, rel_tol=1e-10)
    (x1, s1), (x0, s0) = both(monkeypatch, lambda: P.solve(sp))
    assert s1.iterations == s0.iterations and rel(x1, x0) < SOL_TOL
    P.close()


# the one-workgroup program for the bottom levels, both value types: the last
# mesh that takes it and the first that does not, two and three levels in it,
# no pre-smoothing, odd numbers of sweeps (the iterate ends in the other
# buffer), per-node stencils; the same node code in the same order, so bitwise
@pytest.mark.parametrize("order,m,k0,levels,rot,pre,post", [
    (1, 2, 0, 2, 0, 3, 3), (1, 2, 0, 4, 0, 2, 1), (1, 3, 0, 3, 0, 1, 2), (1, 7, 0, 2, 0, 3, 3), (1, 1, 1, 3, 1, 3, 2),
    (2, 1, 0, 3, 0, 0, 3), (2, 2, 0, 2, 0, 2, 3), (2, 3, 0, 2, 0, 3, 3), (2, 1, 1, 3, 1, 3, 3), (1, 3, 0, 3, 1, 2, 3)])
def test_small_program_matches_launches(order, m, k0, levels, rot, pre, post, monkeypatch):
    P = pm.Problem(order, m, k0, levels, box=(1.0, 0.9, 0.8))
    P.assemble(pm.coeffs(eps=0.05, b=(1.0, 0.5, 0.25), conv_kind=rot, rot_c=(0.4, 0.6), supg=1, f_val=1.0))
    i = P.info(levels - 1)
    r = np.random.default_rng(3).standard_normal(i["ndof"])
    r[i["nact"]:] = 0.0
    for prec in (pm.FP64, pm.MIXED):
        sp = pm.solver_params(omega=0.5, pre=pre, post=post, rel_tol=1e-10, maxit=60, precision=prec)
        out = []
        for bound in ("3000", "0"):
            monkeypatch.setenv("CD3D_SMALL_NODES", bound)
            x, st = P.solve(sp, check=False)
            out.append((P.vcycle(sp, r), x, st.iterations, st.status))
        assert out[0][2:] == out[1][2:]
        assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    P.close()


# cd3d_matvec / cd3d_matvec_dev through lattice order (from 5 M nonzeros) against
# CSR: one product of at most 125 terms per row, 1e-13 of the result's norm.
# What is not the assembled stencil matrix stays with CSR: the mass matrices
# after cd3d_tcd_init, and entries set by the caller
@pytest.mark.parametrize("order,m,k0,levels,rot", [(2, 3, 0, 4, 0), (2, 3, 0, 4, 1), (1, 1, 2, 5, 0), (1, 5, 0, 5, 1)])
def test_matvec_through_the_lattice(order, m, k0, levels, rot, monkeypatch):
    P = pm.Problem(order, m, k0, levels, box=(1.0, 0.9, 0.8))
    co = pm.coeffs(eps=0.05, b=(1.0, 0.5, 0.25), conv_kind=rot, rot_c=(0.4, 0.6), f_val=1.0)
    P.assemble(co)
    l = levels - 1
    assert P.info(l)["nnz"] >= 5000000
    x = np.random.default_rng(7).standard_normal(P.info(l)["ndof"])

    def products():
        out = []
        for on in ("1", "0"):
            monkeypatch.setenv("CD3D_MATVEC_LATTICE", on)
            out.append(P.matvec(l, x))
        return out

    y1, y0 = products()
    assert not np.array_equal(y1, y0) and rel(y1, y0) < 1e-13
    e = P.csr(l)[2]
    P.tcd_init(co, 0.0, x)
    y1, y0 = products()
    assert np.array_equal(y1, y0)
    P.assemble(co)
    P.set_entries(l, 2 * e)
    y2, y3 = products()
    assert np.array_equal(y2, y3)
    P.close()


# affine stencils (rotating field) with 1, 2 and 4 nodes of a column per thread:
# each node's sum in the same order, so bitwise; columns that 2 and 4 do not
# divide, levels that take columns by themselves (97^3 nodes and more)
@pytest.mark.parametrize("order,m,k0,levels", [(1, 3, 0, 4), (1, 7, 0, 3), (2, 3, 0, 3), (2, 5, 0, 3), (1, 3, 0, 6)])
def test_affine_columns_match_single_nodes(order, m, k0, levels, monkeypatch):
    P = pm.Problem(order, m, k0, levels, box=(1.0, 0.9, 0.8))
    co = pm.coeffs(eps=1e-2, conv_kind=1, rot_c=(0.45, 0.55), pulse_c=(0.3, 0.5, 0.5), f_val=0.5)
    u0 = P.interp_pulse(levels - 1, co)
    monkeypatch.setenv("CD3D_SMALL_NODES", "0")
    for prec in (pm.FP64, pm.MIXED):
        sp = pm.solver_params(omega=0.5, pre=2, post=1, rel_tol=1e-10, precision=prec)
        out = []
        for zn in ("1", "2", "4", None):
            if zn:
                monkeypatch.setenv("CD3D_AFF_COL", zn)
            else:
                monkeypatch.delenv("CD3D_AFF_COL")
            P.assemble(co)
            x, st = P.solve(sp)
            P.tcd_init(co, 0.1, u0)
            u, s2 = P.tcd_step(co, sp, 2e-3)
            out.append((x, u, st.iterations, s2.iterations))
        for o in out[1:]:
            assert o[2:] == out[0][2:] and np.array_equal(o[0], out[0][0]) and np.array_equal(o[1], out[0][1])
    P.close()


@pytest.mark.parametrize("order,m,k0,levels,prec,conv", [
    (2, 3, 0, 3, "FP64", 0), (2, 3, 0, 3, "MIXED", 0), (1, 5, 0, 3, "FP64", 1),
    (1, 5, 0, 3, "MIXED", 1), (2, 2, 0, 2, "MIXED", 1)])
def test_reported_residual_is_the_csr_residual(order, m, k0, levels, prec, conv):
    """rfinal from the class stencils against b - A x from the assembled CSR
    matrix: both round at most 127 terms per row."""
    P = pm.Problem(order, m, k0, levels, box=(1.0, 0.7, 0.5))
    P.assemble(pm.coeffs(eps=0.05, b=(1.0, 0.5, 0.25), c=0.3, conv_kind=conv, f_val=1.0))
    l = levels - 1
    x, st = P.solve(pm.solver_params(precision=getattr(pm, prec), rel_tol=1e-6))
    b = P.rhs(l)
    rp, kc, e = P.csr(l)
    row = np.repeat(np.arange(len(rp) - 1), np.diff(rp))
    r = b - np.bincount(row, e * x[kc], len(rp) - 1)
    mag = np.abs(b) + np.bincount(row, np.abs(e * x[kc]), len(rp) - 1)
    tol = 2 * 127 * np.finfo(float).eps * np.linalg.norm(mag)
    print(f"[gpu] rfinal {st.rfinal:.6e}, CSR {np.linalg.norm(r):.6e}, bound {tol:.1e}", flush=True)
    assert abs(st.rfinal - np.linalg.norm(r)) < tol
    P.close()
