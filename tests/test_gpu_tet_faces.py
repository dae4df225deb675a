"""The tetrahedral acoustic kernel where its face matching and its tiling can
go wrong: every local face meeting every other in every orientation (elements
relabelled by random even vertex permutations) between every pair of orders,
element counts around a workgroup's and a column tile's for both block-size
candidates of each order, meshes whose orders leave 4, 8 or 16 lanes per face,
walls, and every way the inputs are stored and counted. Against the oracle with
the FP64 bar of tests/_parity.py; with an FP32 output the result may also
differ by the rounding to FP32, at most 2^-24 of the largest value."""
import itertools

import numpy as np
import pytest

import _oracle as orc
from _parity import assert_parity, rel
from hpgem_amd import OP_ACOUSTIC_CENTRAL, RK4, HpgemAPIDevice, Mesh

pytestmark = pytest.mark.gpu

EVEN = [q for q in itertools.permutations(range(4)) if np.linalg.det(np.eye(4)[list(q)]) > 0]


def relabelled(n, periodic, seed):
    mesh = Mesh.structured(n, periodic=[int(periodic)] * 3, simplices=True)
    rng = np.random.default_rng(seed)
    X, N = np.array(mesh.coords), np.array(mesh.node_ids)
    for e in range(len(N)):
        q = list(EVEN[rng.integers(len(EVEN))])
        X[e], N[e] = X[e][q], N[e][q]
    return Mesh(mesh.shape, X, N)


CASES = [([1, 1, 1], (1,), False, 0), ([2, 1, 1], (4,), False, 1), ([3, 2, 2], (1,), False, 0),
         ([3, 2, 2], (1,), False, 1), ([3, 3, 1], (2,), False, 0), ([3, 3, 2], (2,), False, 1),
         ([2, 2, 2], (3,), False, 0), ([2, 2, 2], (3,), False, 1), ([3, 2, 2], (4,), False, 0),
         ([3, 3, 3], (1, 2), True, 0), ([3, 3, 3], (1, 4), True, 1), ([3, 3, 3], (2, 3), True, 0),
         ([3, 4, 3], (3, 4), True, 1), ([4, 3, 3], (1, 2, 3, 4), True, 0), ([3, 3, 4], (1, 2, 3, 4), False, 1)]


@pytest.mark.parametrize("n,orders,periodic,variant", CASES)
def test_tet_face_kernel(n, orders, periodic, variant):
    print(f"[case] tet faces n={n} p={orders} periodic={periodic} variant={variant}", flush=True)
    seed = sum(n) + 10 * sum(orders) + variant
    mesh = relabelled(n, periodic, seed)
    rng = np.random.default_rng(seed)
    p = rng.choice(np.array(orders, dtype=np.int32), mesh.n_elements).astype(np.int32)
    cinv = 1.0 / rng.uniform(0.5, 2.0, mesh.n_elements) ** 2
    refs = []
    for ext in (False, True):
        P = orc.Problem(mesh.shape, mesh.coords, mesh.node_ids, p, n_fields=4, extended=ext)
        P.set_acoustic(cinv)
        refs.append(P)
    for precision in ("fp64", "mixed"):
        dev = HpgemAPIDevice(mesh, p, precision=precision, kind=OP_ACOUSTIC_CENTRAL, c_inv=cinv, tableau=RK4,
                             n_extra_vectors=2)
        dev.setSimplexThreads([16, 32, 64, 64] if variant else [8, 12, 32, 35])
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
                assert_parity(got, refs[0].time_derivative(vecs[:m], co), ld, int(p.max()), refs[0],
                              f"tet faces {n} p={orders} periodic={periodic} variant={variant}")
            else:
                assert rel(got, ld) <= 2.0 ** -24 + 1e-12
        dev.close()
