"""matrix_rhs where its split of an element row over threads can go wrong: block
sizes around 32, 64, 128 and 256 (the workgroup sizes and their thresholds),
elements of one unknown, sizes that differ inside a mesh, rows of more columns
than the LDS stage holds (2048), rows without neighbours. Against numpy: the
device and numpy sum N <= 6000 products of O(1) values in other orders, and the
masses are identity plus a small symmetric part, so the two differ by at most
N eps ~ 1.4e-12 of the sum of magnitudes; 1e-12 of the largest value holds with
the random signs used here (sqrt(N) eps ~ 2e-14)."""
import numpy as np
import pytest

from hpgem_amd import RK4
from hpgem_amd.api import HpgemAPIMatrixDevice

pytestmark = pytest.mark.gpu

CASES = {
    "around 32": [32, 33, 31, 32], "around 64": [64, 65, 63], "around 128": [127, 128, 129], "around 256": [255, 257],
    "ones": [1, 1, 1], "mixed": [1, 40, 3, 150, 7], "one element": [27], "four rows a thread": [1024, 5],
}


@pytest.mark.parametrize("name", list(CASES) + ["many neighbours"])
def test_matrix_rows(name):
    print(f"[case] matrix rows {name}", flush=True)
    rng = np.random.default_rng(len(name))
    if name == "many neighbours":  # element 0's row has 60 + 30 * 100 columns
        sizes = [60] + [100] * 30
        faces = [(0, i) for i in range(1, 31)]
    else:
        sizes = CASES[name]
        faces = [(i, i + 1) for i in range(len(sizes) - 1)] + [(0, -1)]
    mats = lambda scale: [scale * rng.standard_normal((n, n)) / np.sqrt(n) for n in sizes]
    mass = [np.eye(n) + 0.02 * (r + r.T) for n, r in zip(sizes, mats(1.0))]
    stiff = mats(1.0)
    off = np.concatenate([[0], np.cumsum(sizes)])
    full = np.zeros((off[-1], off[-1]))
    sl = [slice(a, b) for a, b in zip(off[:-1], off[1:])]
    for e, s in enumerate(stiff):
        full[sl[e], sl[e]] += s
    blocks = []
    for L, R in faces:
        parts = []
        for t, u in ([(L, L)] if R < 0 else [(L, L), (L, R), (R, L), (R, R)]):
            b = rng.standard_normal((sizes[t], sizes[u])) / np.sqrt(sizes[u])
            full[sl[t], sl[u]] += b
            parts.append(b.ravel(order="F"))
        blocks.append(np.concatenate(parts))
    dev = HpgemAPIMatrixDevice(mass, stiff, np.array(faces), blocks, tableau=RK4, n_extra_vectors=1)
    u, k = rng.standard_normal((2, dev.n_dof))
    dev.setTimeIntegrationVector(0, u)
    dev.setTimeIntegrationVector(1, k)
    r = full @ (u - 0.25 * k)
    want = np.concatenate([np.linalg.solve(m, r[s]) for m, s in zip(mass, sl)])
    dev.computeTimeDerivative([0, 1], [1.0, -0.25], 2)
    assert np.max(np.abs(dev.getTimeIntegrationVector(2) - want)) <= 1e-12 * np.max(np.abs(want))
    dev.computeRightHandSide([0, 1], [1.0, -0.25], 3)
    assert np.max(np.abs(dev.getTimeIntegrationVector(3) - r)) <= 1e-12 * np.max(np.abs(r))
    dev.close()
