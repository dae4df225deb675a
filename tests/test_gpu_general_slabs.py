"""The Gauss-point kernels with their geometry formed slab by slab before each use,
as they run on a mesh whose stored geometry does not fit the card. That is asked
for here through the library's own function for it (no entry point of the
interface), with slabs of one element up to more than there are. The kernels and
the geometry's numbers are the same, so the results are, bit for bit."""
import ctypes

import numpy as np
import pytest

from _meshes import perturb, rotate_elements
from hpgem_amd import OP_ACOUSTIC_CENTRAL, RK4, HpgemAPIDevice, Mesh, _lib

pytestmark = pytest.mark.gpu


def results(dev, u):
    dev.setTimeIntegrationVector(0, u)
    dev.computeTimeDerivative([0], [1.0], 5)
    dev.computeRightHandSide([0, 5], [1.0, 0.1], 6)
    out = [dev.getTimeIntegrationVector(5), dev.getTimeIntegrationVector(6)]
    for steps in (1, 4):  # the step graph, and pairs with the update in the kernel
        dev.setTimeIntegrationVector(0, u)
        dev.computeOneTimeStep(0.0, 1e-4, steps)
        out.append(dev.getTimeIntegrationVector(0))
    return out


@pytest.mark.parametrize("n,p,kind", [([5, 4], 2, "advection"), ([4, 3], 4, "acoustic"), ([4, 3, 3], 1, "advection"),
                                      ([3, 4, 3], 2, "acoustic"), ([3, 2, 2], 5, "acoustic")])
def test_slabs_give_the_same_bits(n, p, kind):
    print(f"[case] Gauss-point slabs n={n} p={p} {kind}", flush=True)
    lib = _lib.load()
    in_slabs = lib._ZN4hgdg23tensor_general_in_slabsEP8hgdg_ctxl
    in_slabs.restype, in_slabs.argtypes = None, [ctypes.c_void_p, ctypes.c_int64]
    mesh = Mesh.structured(n, periodic=[1] + [0] * (len(n) - 1) if n[0] > 2 else 0)
    X, N, _ = rotate_elements(perturb(mesh.coords, 0.02), mesh.node_ids, p)
    mesh = Mesh(mesh.shape, X, N)
    rng = np.random.default_rng(p)
    cinv = rng.uniform(0.5, 2.0, mesh.n_elements)
    kw = dict(kind=OP_ACOUSTIC_CENTRAL, c_inv=cinv) if kind == "acoustic" else dict(velocity=[1.0, -0.6, 0.4][:len(n)])
    dev = HpgemAPIDevice(mesh, p, tableau=RK4, n_extra_vectors=2, **kw)
    assert dev.usesTensorGeneral()
    u = rng.standard_normal(dev.n_dof)
    want = results(dev, u)
    for elements in (1, 3, 8, mesh.n_elements - 1, 1000):
        in_slabs(dev.h, elements)
        for a, b in zip(results(dev, u), want):
            np.testing.assert_array_equal(a, b)
    # another operator's geometry is stored whole again
    op = _lib.OpDesc(_lib.OP_ADVECTION_UPWIND if kind == "advection" else _lib.OP_ACOUSTIC_CENTRAL, dev.precision,
                     (ctypes.c_double * 3)(1.0, -0.6, 0.4), _lib.dptr(cinv))
    _lib.check(lib.hgdg_operator_set(dev.h, ctypes.byref(op)))
    for a, b in zip(results(dev, u), want):
        np.testing.assert_array_equal(a, b)
    dev.close()
