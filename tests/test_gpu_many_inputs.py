"""Stage inputs of three to eight vectors, in every way they can be stored: all
FP64, FP64 and then FP32 (a mixed Runge-Kutta stage), and orders that no stage
has. Against the same operator on one vector that holds the combination, formed
here in long double and rounded once: each of at most eight sums rounds by at
most eps/2 of a partial sum of at most 6 max|v|, on the way through an operator
that is linear, so the results differ by at most ~10 eps times the amplification
that |w| -> |k| already has, below 1e-12 of the largest value."""
import ctypes

import numpy as np
import pytest

from _parity import rel
from hpgem_amd import OP_ACOUSTIC_CENTRAL, RK4, HpgemAPIDevice, Mesh
from hpgem_amd.tableaux import DORMAND_PRINCE

pytestmark = pytest.mark.gpu

COEFFICIENTS = [1.0, -0.3, 0.25, 1.5, -0.125, 0.2, 0.7, -1.1]
# bit v: vector v is stored in FP32
STORAGES = {"fp64": 0x00, "mixed": 0xfe, "first": 0x01, "alternating": 0x55, "third": 0x04, "all": 0xff}


def check(make):
    for name, f32 in STORAGES.items():
        dev = make("fp64" if f32 == 0 else "mixed")
        rng = np.random.default_rng(f32)
        vecs = [rng.standard_normal(dev.n_dof) for _ in range(8)]
        for v in range(8):
            if (f32 >> v) & 1:
                dev.setStorage(v, "mixed")
                vecs[v] = vecs[v].astype(np.float32).astype(np.float64)
            dev.setTimeIntegrationVector(v, vecs[v])
        for m in (3, 4, 5, 8):
            w = sum(np.longdouble(c) * v for c, v in zip(COEFFICIENTS[:m], vecs)).astype(np.float64)
            dev.setTimeIntegrationVector(8, w)
            dev.computeTimeDerivative([8], [1.0], 9)
            want = dev.getTimeIntegrationVector(9)
            dev.computeTimeDerivative(list(range(m)), COEFFICIENTS[:m], 9)
            assert rel(dev.getTimeIntegrationVector(9), want) <= 1e-12, (name, m)
            dev.computeRightHandSide([8], [1.0], 9)
            want = dev.getTimeIntegrationVector(9)
            dev.computeRightHandSide(list(range(m)), COEFFICIENTS[:m], 9)
            assert rel(dev.getTimeIntegrationVector(9), want) <= 1e-12, (name, m)
        dev.close()


@pytest.mark.parametrize("n,p", [([9, 7], 1), ([9, 7], 2), ([9, 7], 3), ([6, 7], 5), ([5, 4, 6], 1), ([5, 4, 3], 2),
                                 ([5, 4, 3], 3), ([3, 4, 3], 4)])
def test_advection(n, p):
    print(f"[case] many inputs, advection n={n} p={p}", flush=True)
    mesh = Mesh.structured(n, periodic=[1] + [0] * (len(n) - 1))
    check(lambda precision: HpgemAPIDevice(mesh, p, velocity=[1.0, -0.7, 0.3][:len(n)], precision=precision,
                                           tableau=RK4, n_extra_vectors=5))


@pytest.mark.parametrize("n,p", [([9, 7], 1), ([9, 7], 2), ([9, 7], 3), ([6, 7], 4), ([6, 7], 5), ([5, 4, 6], 1),
                                 ([5, 4, 3], 2), ([5, 4, 3], 3), ([3, 4, 3], 4), ([3, 2, 2], 5)])
def test_acoustics(n, p):
    print(f"[case] many inputs, acoustics n={n} p={p}", flush=True)
    mesh = Mesh.structured(n, periodic=[int(n[0] > 2)] + [0] * (len(n) - 1))
    cinv = np.random.default_rng(p).uniform(0.5, 2.0, mesh.n_elements)
    check(lambda precision: HpgemAPIDevice(mesh, p, kind=OP_ACOUSTIC_CENTRAL, c_inv=cinv, precision=precision,
                                           tableau=RK4, n_extra_vectors=5))


@pytest.mark.parametrize("orders", [(1,), (2, 3), (4,), (1, 2, 3, 4)])
def test_tetrahedra(orders):
    print(f"[case] many inputs, tetrahedra p={orders}", flush=True)
    mesh = Mesh.structured([3, 4, 3], periodic=[1, 1, 0], simplices=True)
    rng = np.random.default_rng(len(orders))
    p = rng.choice(np.array(orders, dtype=np.int32), mesh.n_elements).astype(np.int32)
    cinv = rng.uniform(0.5, 2.0, mesh.n_elements)
    check(lambda precision: HpgemAPIDevice(mesh, p, kind=OP_ACOUSTIC_CENTRAL, c_inv=cinv, precision=precision,
                                           tableau=RK4, n_extra_vectors=5))


@pytest.mark.parametrize("tets,p", [(True, 0), (False, 2), (False, 4), (False, 5)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_steps_of_many_stages(tets, p, precision):
    """Steps of Dormand-Prince, whose stages have up to seven inputs: replayed as
    pairs with fused updates, replayed one by one, and stage by stage through
    separate calls. The sums are the same wherever they are formed: bit for bit,
    also after another operator's fields changed the vectors' size."""
    print(f"[case] many stages tets={tets} p={p} {precision}", flush=True)
    mesh = Mesh.structured([4, 3, 3], simplices=tets)
    rng = np.random.default_rng(p)
    order = rng.integers(1, 5, mesh.n_elements).astype(np.int32) if tets else p
    cinv = rng.uniform(0.5, 2.0, mesh.n_elements)
    tab, dt, out = DORMAND_PRINCE, 1e-3, []
    for how in ("pairs", "steps", "calls"):
        dev = HpgemAPIDevice(mesh, order, kind=OP_ACOUSTIC_CENTRAL, c_inv=cinv, precision=precision, tableau=tab)
        dev.setFusedTimeStepping(how == "pairs")
        dev.setTimeIntegrationVector(0, np.random.default_rng(7).standard_normal(dev.n_dof))
        if how == "calls":
            if precision == "mixed":
                for v in dev.auxiliaryVectorIds_:
                    dev.setStorage(v, "mixed")
            for _ in range(2):
                for i, row in enumerate(tab.a_matrix()):
                    ids = [0] + [1 + j for j in range(i) if row[j] != 0.0]
                    dev.computeTimeDerivative(ids, [1.0] + [dt * row[j - 1] for j in ids[1:]], 1 + i)
                for j, b in enumerate(tab.b):
                    if b != 0.0:
                        dev.scaleAndAddVector(0, 1 + j, dt * b)
        else:
            dev.computeOneTimeStep(0.0, dt, 2)
        out.append([dev.getTimeIntegrationVector(v) for v in range(tab.stages + 1)])
        dev.close()
    assert np.all(np.isfinite(out[0][0]))
    for other in out[1:]:
        for g, f in zip(out[0], other):
            np.testing.assert_array_equal(f, g)


@pytest.mark.parametrize("tets,p", [(True, 0), (False, 2), (False, 5)])
def test_captured_before_any_other_call(tets, p):
    """A stage of five inputs captured as the first call of its kind, when no
    vector for its sum can be allocated: the kernels sum by themselves, and every
    replay gives what the call gives outside."""
    print(f"[case] many inputs captured tets={tets} p={p}", flush=True)
    hip = ctypes.CDLL("libamdhip64.so")
    mesh = Mesh.structured([4, 3, 3], simplices=tets)
    rng = np.random.default_rng(p)
    order = rng.integers(1, 5, mesh.n_elements).astype(np.int32) if tets else p
    dev = HpgemAPIDevice(mesh, order, kind=OP_ACOUSTIC_CENTRAL, c_inv=rng.uniform(0.5, 2.0, mesh.n_elements), tableau=RK4,
                         n_extra_vectors=2)
    graph, run, stream = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p(dev.stream())
    for v in range(5):
        dev.setTimeIntegrationVector(v, rng.standard_normal(dev.n_dof))
    ids, co = list(range(5)), COEFFICIENTS[:5]
    assert hip.hipStreamBeginCapture(stream, 0) == 0
    dev.computeTimeDerivative(ids, co, 5)
    assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
    assert hip.hipGraphInstantiate(ctypes.byref(run), graph, None, None, 0) == 0
    for _ in range(3):
        dev.setTimeIntegrationVector(1, rng.standard_normal(dev.n_dof))
        dev.computeTimeDerivative(ids, co, 6)
        assert hip.hipGraphLaunch(run, stream) == 0
        np.testing.assert_array_equal(dev.getTimeIntegrationVector(5), dev.getTimeIntegrationVector(6))
    assert hip.hipGraphExecDestroy(run) == 0 and hip.hipGraphDestroy(graph) == 0
    dev.close()
