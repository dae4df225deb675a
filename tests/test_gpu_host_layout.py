"""Where the values of hgdg_state_set and hgdg_state_get go, by something that
does not take the same way: the right-hand side of what was set, read back and
compared with the oracle's, which has hpGEM's layout throughout. A wrong
permutation or offset that set and get share cannot pass, since the operator does
not commute with it. Vectors of a few elements, of several chunks (2^18 unknowns) on one thread and of four threads
(from 2^20), tensor elements (permuted), tetrahedra of mixed order (regrouped)
and matrix operators; elements at both sides of every cut are among the compared.
The same of the library's own copy through pageable memory, which serves where no
pinned memory is left and no entry point of the interface asks for.
The oracle runs the same FP64 algorithm as the reference's; the two differ by
rounding, below 1e-10 of the largest value at these orders (the oracle's own
mass solves are the larger part), while any misplaced value differs by O(1)."""
import ctypes

import numpy as np
import pytest

import _oracle as orc
from _parity import rel
from hpgem_amd import OP_ACOUSTIC_CENTRAL, RK4, HpgemAPIDevice, Mesh, _lib
from hpgem_amd.api import HpgemAPIMatrixDevice

pytestmark = pytest.mark.gpu

TENSOR = [([5, 4], 2, False), ([16, 16], 3, False), ([40, 30], 1, True), ([60, 70], 2, True), ([16, 16, 17], 3, False),
          ([13, 12, 11], 2, True), ([32, 32, 17], 3, False)]


@pytest.mark.parametrize("n,p,acoustic", TENSOR)
def test_tensor_elements(n, p, acoustic):
    print(f"[case] host layout n={n} p={p} acoustic={acoustic}", flush=True)
    mesh = Mesh.structured(n)
    rng = np.random.default_rng(sum(n))
    P = orc.Problem(mesh.shape, mesh.coords, mesh.node_ids, p, n_fields=len(n) + 1 if acoustic else 1, extended="bench")
    if acoustic:
        kw = dict(kind=OP_ACOUSTIC_CENTRAL, c_inv=rng.uniform(0.5, 2.0, mesh.n_elements))
        P.set_acoustic(kw["c_inv"])
    else:
        kw = dict(velocity=[1.0, 0.7, 0.3][:len(n)])
        P.set_advection(kw["velocity"])
    dev = HpgemAPIDevice(mesh, p, tableau=RK4, **kw)
    u = rng.standard_normal(dev.n_dof)
    dev.setTimeIntegrationVector(0, u)
    dev.computeTimeDerivative([0], [1.0], 1)
    want = P.time_derivative_par([u], [1.0])
    assert rel(dev.getTimeIntegrationVector(1), want) <= 1e-10
    # FP32 storage on the way in and on the way out
    dev.setStorage(2, "mixed")
    dev.setStorage(3, "mixed")
    u = u.astype(np.float32).astype(np.float64)
    dev.setTimeIntegrationVector(2, u)
    dev.computeTimeDerivative([2], [1.0], 3)
    assert rel(dev.getTimeIntegrationVector(3), P.time_derivative_par([u], [1.0])) <= 2.0 ** -24 + 1e-10
    dev.close()


@pytest.mark.parametrize("n", [[2, 2, 2], [4, 4, 5], [9, 8, 11], [16, 14, 13]])
def test_tetrahedra(n):
    print(f"[case] host layout tets n={n}", flush=True)
    mesh = Mesh.structured(n, periodic=[0] * 3, simplices=True)
    rng = np.random.default_rng(n[0])
    p = rng.integers(1, 5, mesh.n_elements).astype(np.int32)
    cinv = rng.uniform(0.5, 2.0, mesh.n_elements)
    P = orc.Problem(mesh.shape, mesh.coords, mesh.node_ids, p, n_fields=4, extended="bench")
    P.set_acoustic(cinv)
    dev = HpgemAPIDevice(mesh, p, kind=OP_ACOUSTIC_CENTRAL, c_inv=cinv, tableau=RK4)
    u = rng.standard_normal(dev.n_dof)
    dev.setTimeIntegrationVector(0, u)
    dev.computeTimeDerivative([0], [1.0], 1)
    assert rel(dev.getTimeIntegrationVector(1), P.time_derivative_par([u], [1.0])) <= 1e-10
    dev.close()


@pytest.mark.parametrize("blocks,n", [(30, 7), (700, 7), (40000, 7)])
def test_matrix_operator(blocks, n):
    """Each element another multiple of one matrix that moves every value."""
    print(f"[case] host layout matrices {blocks} of {n}", flush=True)
    rng = np.random.default_rng(n)
    a, scale = rng.standard_normal((n, n)), rng.uniform(0.5, 2.0, blocks)
    dev = HpgemAPIMatrixDevice([np.eye(n)] * blocks, [s * a for s in scale], np.zeros((0, 2)), [], tableau=RK4)
    u = rng.standard_normal((blocks, n))
    dev.setTimeIntegrationVector(0, u.ravel())
    dev.computeTimeDerivative([0], [1.0], 1)
    assert rel(dev.getTimeIntegrationVector(1), (scale[:, None] * (u @ a.T)).ravel()) <= 1e-13
    dev.close()


@pytest.mark.parametrize("kind", ["tensor", "tetrahedra", "matrix"])
def test_pageable(kind):
    print(f"[case] host layout, pageable, {kind}", flush=True)
    copy = _lib.load()._ZN4hgdg18host_copy_pageableEP8hgdg_ctxiPdPKd
    copy.restype, copy.argtypes = None, [ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p]
    rng = np.random.default_rng(7)
    if kind == "tensor":
        dev = HpgemAPIDevice(Mesh.structured([5, 4]), 2, tableau=RK4, velocity=[1.0, 0.7])
    elif kind == "tetrahedra":
        mesh = Mesh.structured([2, 2, 3], periodic=[0] * 3, simplices=True)
        p = rng.integers(1, 5, mesh.n_elements).astype(np.int32)
        dev = HpgemAPIDevice(mesh, p, kind=OP_ACOUSTIC_CENTRAL, c_inv=np.ones(mesh.n_elements), tableau=RK4)
    else:
        dev = HpgemAPIMatrixDevice([np.eye(7)] * 5, [np.eye(7)] * 5, np.zeros((0, 2)), [], tableau=RK4)
    u, got = rng.standard_normal(dev.n_dof), np.empty(dev.n_dof)
    for storage in ("fp64", "mixed"):
        if storage == "mixed":
            if kind == "matrix":
                break
            dev.setStorage(1, "mixed")
            u = u.astype(np.float32).astype(np.float64)
        copy(dev.h, 1, None, u.ctypes.data)
        np.testing.assert_array_equal(dev.getTimeIntegrationVector(1), u)
        dev.setTimeIntegrationVector(1, -u)
        copy(dev.h, 1, got.ctypes.data, None)
        np.testing.assert_array_equal(got, -u)
    dev.close()
