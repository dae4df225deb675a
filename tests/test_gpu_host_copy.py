"""hgdg_state_set / hgdg_state_get through chunks of pinned memory: vectors
smaller than a chunk (2^18 unknowns), of exactly one, one unknown or element
more, several chunks on one thread and on four (from 2^20 unknowns), FP64 and
FP32 storage, tensor elements (permuted), tetrahedra of mixed order (grouped on
the device) and matrix operators. What was set comes back bit for bit (rounded
to FP32 in FP32 storage), and two vectors meet unknown by unknown. Whether each
unknown reaches its place, which a round trip cannot tell, is compared with the
oracle's layout in test_gpu_host_layout.py."""
import numpy as np
import pytest

from hpgem_amd import OP_ACOUSTIC_CENTRAL, RK4, HpgemAPIDevice, Mesh
from hpgem_amd.api import HpgemAPIMatrixDevice

pytestmark = pytest.mark.gpu


def tensor(n, p):
    mesh = Mesh.structured(n, periodic=[int(k > 2) for k in n])
    return HpgemAPIDevice(mesh, p, velocity=[1.0, 0.5, 0.25][:len(n)], tableau=RK4, n_extra_vectors=1)


def tets(n):
    mesh = Mesh.structured(n, periodic=[0] * 3, simplices=True)
    rng = np.random.default_rng(1)
    return HpgemAPIDevice(mesh, rng.integers(1, 5, mesh.n_elements), kind=OP_ACOUSTIC_CENTRAL,
                          c_inv=np.ones(mesh.n_elements), tableau=RK4, n_extra_vectors=1)


def matrix(blocks, n):
    eye = [np.eye(n)] * blocks
    return HpgemAPIMatrixDevice(eye, eye, np.zeros((0, 2)), [], tableau=RK4, n_extra_vectors=1)


CASES = {
    "small quads": lambda: tensor([5, 4], 2), "one chunk": lambda: tensor([16, 16, 16], 3),
    "one element more": lambda: tensor([17, 241, 1], 3), "odd order": lambda: tensor([21, 20, 11], 4),
    "several, one thread": lambda: tensor([30, 30, 12], 3), "four threads": lambda: tensor([32, 32, 17], 3),
    "small tets": lambda: tets([3, 2, 2]), "tets, several": lambda: tets([9, 8, 11]), "tets, threads": lambda: tets([16, 14, 13]),
    "matrix": lambda: matrix(700, 7),
}


@pytest.mark.parametrize("name", list(CASES))
def test_state_round_trip(name):
    print(f"[case] host copy {name}", flush=True)
    dev = CASES[name]()
    rng = np.random.default_rng(3)
    u, w = rng.standard_normal((2, dev.n_dof))
    dev.setTimeIntegrationVector(0, u)
    dev.setTimeIntegrationVector(1, w)
    assert np.array_equal(dev.getTimeIntegrationVector(0), u)
    dev.scaleAndAddVector(0, 1, 2.0)  # unknowns of the two vectors meet one by one
    assert np.array_equal(dev.getTimeIntegrationVector(0), u + 2.0 * w)  # (2 w is exact, so one rounding either way)
    assert np.array_equal(dev.getTimeIntegrationVector(1), w)
    dev.setStorage(2, "mixed")
    dev.setTimeIntegrationVector(2, u)
    assert np.array_equal(dev.getTimeIntegrationVector(2), u.astype(np.float32).astype(np.float64))
    dev.close()
