"""Stage inputs of three to eight vectors, in every way they can be stored: all
FP64, FP64 and then FP32 (a mixed Runge-Kutta stage), and orders that no stage
has. Against the same operator on one vector that holds the combination, formed
here in long double and rounded once: each of at most eight sums rounds by at
most eps/2 of a partial sum of at most 6 max|v|, on the way through an operator
that is linear, so the results differ by at most ~10 eps times the amplification
that |w| -> |k| already has, below 1e-12 of the largest value."""
import numpy as np
import pytest

from _parity import rel
from hpgem_amd import RK4, HpgemAPIDevice, Mesh

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
