"""The step's error estimate and solution size where the lanes per element and
the workgroups change: elements of 4 to 875 values (down to a few lanes each,
up to several rounds of a wavefront), element counts below, around and beyond
one round of the launch, mixed element sizes, FP32 stage vectors. Against the
definition in float64: all terms of both sums are non-negative, so the sums'
own rounding stays below 1e-12."""
import numpy as np
import pytest

import hpgem_amd.tableaux as tableaux
from hpgem_amd import OP_ACOUSTIC_CENTRAL, HpgemAPIDevice, Mesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,p,acoustic,tets,precision", [
    ([3, 3], 1, False, False, "fp64"), ([301, 257], 1, False, False, "mixed"), ([65, 63], 2, False, False, "fp64"),
    ([257, 260], 3, False, False, "fp64"), ([5, 4, 3], 2, False, False, "mixed"), ([12, 11, 10], 2, True, False, "fp64"),
    ([4, 3, 5], 4, True, False, "fp64"), ([6, 6, 6], 0, True, True, "mixed")])
def test_step_error_and_norm(n, p, acoustic, tets, precision):
    print(f"[case] step norm n={n} p={p} acoustic={acoustic} tets={tets} {precision}", flush=True)
    mesh = Mesh.structured(n, simplices=tets)
    rng = np.random.default_rng(sum(n) + p)
    orders = rng.integers(1, 5, mesh.n_elements).astype(np.int32) if tets else p
    tab = tableaux.DORMAND_PRINCE
    kw = dict(kind=OP_ACOUSTIC_CENTRAL, c_inv=np.ones(mesh.n_elements)) if acoustic else dict(
        velocity=[1.0, 0.7, 0.3][:len(n)])
    dev = HpgemAPIDevice(mesh, orders, precision=precision, tableau=tab, **kw)
    fields = len(n) + 1 if acoustic else 1
    size = fields * (orders + 1) * (orders + 2) * (orders + 3) // 6 if tets else np.full(
        mesh.n_elements, fields * (p + 1) ** len(n))
    assert size.sum() == dev.n_dof
    u = rng.standard_normal(dev.n_dof)
    dev.setTimeIntegrationVector(dev.solutionVectorId_, u)
    d = np.zeros(dev.n_dof)
    dt = 0.03
    for j, v in enumerate(dev.auxiliaryVectorIds_):
        k = rng.standard_normal(dev.n_dof)
        if precision == "mixed":
            dev.setStorage(v, "mixed")
            k = k.astype(np.float32).astype(np.float64)
        dev.setTimeIntegrationVector(v, k)
        d += dt * tab.error[j] * k
    err, nrm = dev.computeErrorAndNormOfUpdate(dt)
    off = np.concatenate([[0], np.cumsum(size)[:-1]])
    assert abs(err - np.sqrt(np.sum(d * d))) <= 1e-12 * err
    ref = np.sum(np.sqrt(np.add.reduceat(u * u, off)))
    assert abs(nrm - ref) <= 1e-12 * ref
    dev.close()
