"""The Gauss-point RHS kernel where its tiling and its stored geometry can go
wrong: element counts around a workgroup's (8, 9, 1, 2 and 1 elements in 3D for
p = 1..5; 16, 7, 4, 5 and 7 in 2D), order 5 in 3D, walls, FP32 inputs and output,
and a second operator on the same mesh (its geometry replaces the first's).
Against the oracle with the FP64 bar of tests/_parity.py; with an FP32 output
also the rounding to FP32, at most 2^-24 of the largest value."""
import ctypes

import numpy as np
import pytest

import _oracle as orc
from _meshes import perturb, rotate_elements
from _parity import assert_parity, rel
from hpgem_amd import OP_ACOUSTIC_CENTRAL, RK4, HpgemAPIDevice, Mesh, _lib

pytestmark = pytest.mark.gpu

CASES = [([3, 3, 1], 1, "acoustic"), ([5, 2, 1], 2, "acoustic"), ([3, 3, 2], 2, "advection"), ([2, 2, 1], 3, "acoustic"),
         ([3, 1, 1], 4, "acoustic"), ([2, 1, 1], 5, "acoustic"), ([2, 1, 1], 5, "advection"), ([6, 3], 1, "acoustic"),
         ([4, 2], 2, "acoustic"), ([5, 1], 3, "advection"), ([3, 2], 4, "acoustic"), ([4, 2], 5, "acoustic")]


@pytest.mark.parametrize("n,p,kind", CASES)
def test_general_blocks(n, p, kind):
    print(f"[case] Gauss-point blocks n={n} p={p} {kind}", flush=True)
    dim = len(n)
    mesh = Mesh.structured(n, periodic=[0] * dim)
    X, nodes, _ = rotate_elements(perturb(mesh.coords), mesh.node_ids, 3 + p)
    rng = np.random.default_rng(sum(n) + p)
    cinv = 1.0 / rng.uniform(0.5, 2.0, mesh.n_elements) ** 2
    velocities = [[1.0, 0.7, 0.3][:dim], [-0.4, 0.9, -1.1][:dim]]

    def oracle(extended, vel):
        P = orc.Problem(mesh.shape, X, nodes, p, n_fields=1 if kind == "advection" else dim + 1, extended=extended)
        if kind == "advection":
            P.set_advection(vel)
        else:
            P.set_acoustic(cinv)
        return P

    for precision in ("fp64", "mixed"):
        kw = {"velocity": velocities[0]} if kind == "advection" else {"kind": OP_ACOUSTIC_CENTRAL, "c_inv": cinv}
        dev = HpgemAPIDevice(Mesh(mesh.shape, X, nodes), p, precision=precision, tableau=RK4, n_extra_vectors=2,
                             tensor_general=True, **kw)
        for i, vel in enumerate(velocities if kind == "advection" else velocities[:1]):
            if i == 1:
                op = _lib.OpDesc(_lib.OP_ADVECTION_UPWIND, dev.precision, (ctypes.c_double * 3)(*vel), None)
                _lib.check(dev.lib.hgdg_operator_set(dev.h, ctypes.byref(op)))
            u, k = rng.standard_normal((2, dev.n_dof))
            if precision == "mixed":
                dev.setStorage(1, "mixed")
                dev.setStorage(2, "mixed")
                k = k.astype(np.float32).astype(np.float64)
            dev.setTimeIntegrationVector(0, u)
            dev.setTimeIntegrationVector(1, k)
            dev.computeTimeDerivative([0, 1], [1.0, -0.3], 2)
            got = dev.getTimeIntegrationVector(2)
            ld = oracle(True, vel).time_derivative([u, k], [1.0, -0.3])
            if precision == "fp64":
                P = oracle(False, vel)
                assert_parity(got, P.time_derivative([u, k], [1.0, -0.3]), ld, p, P, f"Gauss-point {n} p={p} {kind}")
            else:
                assert rel(got, ld) <= 2.0 ** -24 + 1e-12
        dev.close()
