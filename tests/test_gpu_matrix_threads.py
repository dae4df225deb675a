"""matrix_rhs at the numbers of elements and sizes where its threads per element
row change (64 to 1024: by the rows, by how few elements there are, and by the
values of a row), and at matrices beyond the last-level cache, which are read
past it. Against numpy, element row by element row: N <= 7 * 300 products of
O(1) values in other orders differ by at most N eps of the sum of magnitudes,
sqrt(N) eps ~ 1e-14 with random signs; 1e-12 of the largest value holds."""
import numpy as np
import pytest

from hpgem_amd import RK4
from hpgem_amd.api import HpgemAPIMatrixDevice

pytestmark = pytest.mark.gpu

# a ring of elements, each with its two neighbours: 3 blocks a row
CASES = [(9000, 1), (4000, 6), (2048, 33), (1025, 20), (1024, 20), (700, 64), (300, 30), (200, 65), (130, 130), (127, 27),
         (40, 3), (20, 257), (3, 300), (16384, 37)]


@pytest.mark.parametrize("elements,n", CASES)
def test_matrix_threads(elements, n):
    print(f"[case] matrix threads {elements} elements of {n}", flush=True)
    rng = np.random.default_rng(elements + n)
    kinds = 5  # element matrices and face blocks repeat: quick to make, and no two neighbours alike
    mass = [np.eye(n) + 0.02 / np.sqrt(n) * (m + m.T) for m in rng.standard_normal((kinds, n, n))]
    stiff = rng.standard_normal((kinds, n, n)) / np.sqrt(n)
    block = rng.standard_normal((kinds, 4, n, n)) / np.sqrt(n)
    e = np.arange(elements)
    faces = np.stack([e, (e + 1) % elements], axis=1)
    dev = HpgemAPIMatrixDevice([mass[i % kinds] for i in e], [stiff[i % kinds] for i in e], faces,
                               [np.concatenate([b.ravel(order="F") for b in block[i % kinds]]) for i in e], tableau=RK4,
                               n_extra_vectors=1)
    u = rng.standard_normal((elements, n))
    dev.setTimeIntegrationVector(0, u.ravel())
    left, right = u, np.roll(u, -1, axis=0)  # of face i: elements i and i + 1
    r = np.einsum("eij,ej->ei", stiff[e % kinds], u)
    b = block[e % kinds]
    r += np.einsum("eij,ej->ei", b[:, 0], left) + np.einsum("eij,ej->ei", b[:, 1], right)
    r += np.roll(np.einsum("eij,ej->ei", b[:, 2], left) + np.einsum("eij,ej->ei", b[:, 3], right), 1, axis=0)
    want = np.empty_like(r)
    for k in range(kinds):
        want[k::kinds] = np.linalg.solve(mass[k], r[k::kinds].T).T
    dev.computeTimeDerivative([0], [1.0], 1)
    assert np.max(np.abs(dev.getTimeIntegrationVector(1) - want.ravel())) <= 1e-12 * np.max(np.abs(want))
    dev.computeRightHandSide([0], [1.0], 2)
    assert np.max(np.abs(dev.getTimeIntegrationVector(2) - r.ravel())) <= 1e-12 * np.max(np.abs(r))
    dev.close()
