"""The tensor acoustic kernel (one thread per x-pencil with all fields, fluxes
of the y and z face pencils shared through LDS) where its tiling can go wrong:
element counts around a workgroup's, rows that end inside one (x neighbours in
the wavefront, in another one, and outside the workgroup), more face pencils
than threads (p = 1, 2), every workgroup size (64, 128 and 256 threads), walls,
and every way its inputs are stored and counted. Against the oracle with the
FP64 bar of tests/_parity.py; with an FP32 output the result may also differ by
the rounding to FP32, at most 2^-24 of the largest value."""
import numpy as np
import pytest

import _oracle as orc
from _parity import assert_parity, rel
from hpgem_amd import OP_ACOUSTIC_CENTRAL, RK4, HpgemAPIDevice, Mesh

pytestmark = pytest.mark.gpu

CASES = [([21, 3], 2, True), ([11, 6], 2, True), ([16, 4], 3, False), ([13, 5], 4, True), ([5, 4], 5, False),
         ([33, 4], 1, True), ([5, 3, 4], 1, True), ([17, 1, 1], 1, False), ([7, 2, 2], 2, False), ([3, 5, 3], 2, True),
         ([5, 3, 3], 3, True), ([4, 1, 2], 3, False), ([3, 3, 1], 4, False), ([2, 2, 1], 5, False)]


@pytest.mark.parametrize("n,p,periodic", CASES)
def test_acoustic_pencil_kernel(n, p, periodic):
    print(f"[case] acoustic pencils n={n} p={p} periodic={periodic}", flush=True)
    mesh = Mesh.structured(n, periodic=[int(periodic)] * len(n))
    rng = np.random.default_rng(sum(n) + p)
    cinv = 1.0 / rng.uniform(0.5, 2.0, mesh.n_elements) ** 2
    refs = []
    for ext in (False, True):
        P = orc.Problem(mesh.shape, mesh.coords, mesh.node_ids, p, n_fields=len(n) + 1, extended=ext)
        P.set_acoustic(cinv)
        refs.append(P)
    for precision in ("fp64", "mixed"):
        dev = HpgemAPIDevice(mesh, p, precision=precision, kind=OP_ACOUSTIC_CENTRAL, c_inv=cinv, tableau=RK4,
                             n_extra_vectors=2)
        vecs = [rng.standard_normal(dev.n_dof) for _ in range(3)]
        if precision == "mixed":
            for v in (1, 2, 3):
                dev.setStorage(v, "mixed")
            vecs[1:] = [v.astype(np.float32).astype(np.float64) for v in vecs[1:]]
        for i, v in enumerate(vecs):
            dev.setTimeIntegrationVector(i, v)
        for m, co in ((1, [1.0]), (2, [1.0, -0.3]), (3, [0.5, 0.2, 1.5])):
            dev.computeTimeDerivative(list(range(m)), co, 3)
            got = dev.getTimeIntegrationVector(3)
            ld = refs[1].time_derivative(vecs[:m], co)
            if precision == "fp64":
                assert_parity(got, refs[0].time_derivative(vecs[:m], co), ld, p, refs[0], f"acoustic pencils {n} p={p}")
            else:
                assert rel(got, ld) <= 2.0 ** -24 + 1e-12
        dev.close()


@pytest.mark.parametrize("n,p,precision", [([23, 17, 3], 4, "fp64"), ([21, 11, 2], 5, "mixed"), ([60, 31, 2], 2, "fp64"),
                                           ([7, 97, 2], 4, "fp64")])
def test_acoustic_workgroup_order(n, p, precision):
    """Boxes whose planes pass the L2, whose workgroups are taken in columns of
    rows, against the same box with its elements in random order (other rows
    or none): the same operator, so equal within rounding (1e-12, mixed: its
    storage's 2^-24 more)."""
    print(f"[case] acoustic order n={n} p={p} {precision}", flush=True)
    mesh = Mesh.structured(n, periodic=[1, 1, 0])
    rng = np.random.default_rng(p)
    E = mesh.n_elements
    c = 1.0 / rng.uniform(0.5, 2.0, E) ** 2
    perm = rng.permutation(E)
    u = rng.standard_normal((E, 4 * (p + 1) ** 3))
    out = []
    for order in (np.arange(E), perm):
        m = Mesh(mesh.shape, np.array(mesh.coords)[order], np.array(mesh.node_ids)[order])
        dev = HpgemAPIDevice(m, p, precision=precision, kind=OP_ACOUSTIC_CENTRAL, c_inv=c[order], tableau=RK4)
        dev.setTimeIntegrationVector(0, u[order].ravel())
        dev.computeOneTimeStep(0.0, 1e-4, 2)
        dev.computeTimeDerivative([0], [1.0], 1)
        out.append(np.empty_like(u))
        out[-1][order] = dev.getTimeIntegrationVector(1).reshape(E, -1)
        dev.close()
    assert rel(out[1], out[0]) <= 1e-12 + (2.0 ** -24 if precision == "mixed" else 0.0)


@pytest.mark.parametrize("n,p,periodic", CASES)
def test_acoustic_right_hand_side_in_one_launch(n, p, periodic):
    """hgdg_right_hand_side (the mass taken in the kernel itself) at the same
    tiles' edges, FP32 and FP64 inputs, against the oracle."""
    print(f"[case] acoustic right-hand side n={n} p={p} periodic={periodic}", flush=True)
    mesh = Mesh.structured(n, periodic=[int(periodic)] * len(n))
    rng = np.random.default_rng(sum(n) + 2 * p)
    cinv = 1.0 / rng.uniform(0.5, 2.0, mesh.n_elements) ** 2
    refs = []
    for ext in (False, True):
        P = orc.Problem(mesh.shape, mesh.coords, mesh.node_ids, p, n_fields=len(n) + 1, extended=ext)
        P.set_acoustic(cinv)
        refs.append(P)
    dev = HpgemAPIDevice(mesh, p, kind=OP_ACOUSTIC_CENTRAL, c_inv=cinv, tableau=RK4, n_extra_vectors=2)
    dev.setStorage(1, "mixed")
    vecs = [rng.standard_normal(dev.n_dof) for _ in range(3)]
    vecs[1] = vecs[1].astype(np.float32).astype(np.float64)
    for i, v in enumerate(vecs):
        dev.setTimeIntegrationVector(i, v)
    for m, co in ((1, [1.0]), (2, [1.0, -0.3]), (3, [0.5, 0.2, 1.5])):
        dev.computeRightHandSide(list(range(m)), co, 3)
        assert_parity(dev.getTimeIntegrationVector(3), refs[0].right_hand_side(vecs[:m], co),
                      refs[1].right_hand_side(vecs[:m], co), p, refs[0], f"acoustic right-hand side {n} p={p}")
    dev.close()
