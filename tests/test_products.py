"""Products on device vectors (cd3d_matvec_dev) on a level large enough for the
lattice route (5 M nonzeros): the first one on a handle allocates nothing, and
a product captured into a graph on the handle's stream gives the eager
product's bits on every replay.  x is the level's scratch vector 3, which
cd3d_interpolate fills; y its vector 0, which cd3d_get_solution reads."""
import ctypes as C

import numpy as np
import pytest

import parmoon_cmg_amd as pm

pytestmark = pytest.mark.gpu

L = 3


@pytest.fixture
def large():
    P = pm.Problem(2, 3, 0, 4, box=(1.0, 0.9, 0.8))  # Q2 24^3, 6.6 M nonzeros
    assert P.info(L)["nnz"] >= 5000000
    P.assemble(pm.coeffs(eps=0.05, b=(1.0, 0.5, 0.25), supg=1, f_val=1.0))
    yield P
    P.close()


def pulse(P, x0):
    """A pulse into vector 3; returns its host copy."""
    return P.interpolate(L, P.FN_PULSE, pm.coeffs(pulse_c=(x0, 0.5, 0.4)))


def test_first_product_allocates_nothing(large):
    P = large
    x = pulse(P, 0.3)
    held = P.L.cd3d_device_bytes(P.h)
    P.matvec_dev(L, P.device_ptr(L, 3), P.device_ptr(L, 0))
    assert P.L.cd3d_device_bytes(P.h) == held
    y = P.solution()
    assert np.array_equal(y, P.matvec(L, x))
    assert P.L.cd3d_device_bytes(P.h) == held


def test_captured_product_replays(large):
    P = large
    hip = C.CDLL("libamdhip64.so.7")

    def ok(rc):
        assert rc == 0, rc

    s = C.c_void_p(P.L.cd3d_stream(P.h))
    graph, ex = C.c_void_p(), C.c_void_p()
    P.synchronize()
    ok(hip.hipStreamBeginCapture(s, 0))
    P.matvec_dev(L, P.device_ptr(L, 3), P.device_ptr(L, 0))
    ok(hip.hipStreamEndCapture(s, C.byref(graph)))
    ok(hip.hipGraphInstantiate(C.byref(ex), graph, None, None, C.c_size_t(0)))
    for x0 in (0.3, 0.5, 0.7):
        x = pulse(P, x0)
        eager = P.matvec(L, x)  # the program's own work between the replays
        ok(hip.hipGraphLaunch(ex, s))
        P.synchronize()
        assert np.array_equal(P.solution(), eager) and np.any(eager)
    ok(hip.hipGraphExecDestroy(ex))
    ok(hip.hipGraphDestroy(graph))


@pytest.mark.parametrize("state", ["assembled", "entries set", "mass"])
def test_staged_product_takes_the_same_route(large, state):
    P = large
    if state == "entries set":
        P.set_entries(L, 2 * P.csr(L)[2])
    if state == "mass":
        P.tcd_init(pm.coeffs(eps=1e-3, conv_kind=1), 0.0, np.zeros(P.info(L)["ndof"]))
    x = np.random.default_rng(9).standard_normal(P.info(L)["ndof"])
    held = P.L.cd3d_device_bytes(P.h)
    y = P.matvec_noalloc(L, x)
    assert P.L.cd3d_device_bytes(P.h) == held
    assert np.array_equal(y, P.matvec(L, x))
