"""The tensor advection kernel (one thread per x-pencil; each y/z face pencil's
flux formed once and shared through LDS) where its tiling can go wrong: element
counts around a workgroup's, rows that end inside one (x neighbours in it and
outside), more face pencils than threads (p = 1, 2 on cubes), every choice of
tiles per workgroup, upwind, averaged and boundary faces, and every count and
storage of its inputs. Against the oracle with the FP64 bar of
tests/_parity.py; with an FP32 output the result may also differ by the
rounding to FP32, at most 2^-24 of the largest value."""
import numpy as np
import pytest

import _oracle as orc
from _parity import assert_parity, rel
import hpgem_amd.tableaux
from hpgem_amd import RK4, HpgemAPIDevice, Mesh

pytestmark = pytest.mark.gpu

CASES = [([43, 3], 1, [1.0, -0.5], True), ([17, 10], 2, [-1.0, 0.0], True), ([17, 5], 2, [1.0, 0.5], False),
         ([16, 4], 3, [1.0, 0.5], True), ([13, 5], 3, [0.0, -0.3], False), ([11, 5], 4, [-0.3, 0.8], True),
         ([5, 13, 1], 1, [1.0, 0.7, 0.3], True), ([5, 3, 4], 1, [1.0, 0.0, -0.3], False),
         ([29, 1, 1], 2, [1.0, 0.7, 0.3], True), ([7, 2, 2], 2, [-1.0, 0.7, 0.0], False),
         ([17, 1, 1], 3, [1.0, -0.7, 0.3], True), ([5, 3, 2], 3, [1.0, 0.7, -0.3], False),
         ([3, 3, 1], 4, [-0.2, 0.7, 0.3], False), ([11, 1, 1], 4, [1.0, 0.7, 0.3], True)]


@pytest.mark.parametrize("n,p,a,periodic", CASES)
def test_advection_pencil_kernel(n, p, a, periodic):
    print(f"[case] advection pencils n={n} p={p} a={a} periodic={periodic}", flush=True)
    mesh = Mesh.structured(n, periodic=[int(periodic and k > 2) for k in n])
    rng = np.random.default_rng(sum(n) + p)
    refs = []
    for ext in (False, True):
        P = orc.Problem(mesh.shape, mesh.coords, mesh.node_ids, p, extended=ext)
        P.set_advection(a)
        refs.append(P)
    for precision in ("fp64", "mixed"):
        dev = HpgemAPIDevice(mesh, p, velocity=a, precision=precision, tableau=RK4, n_extra_vectors=6)
        vecs = [rng.standard_normal(dev.n_dof) for _ in range(8)]
        if precision == "mixed":
            for v in range(1, 9):
                dev.setStorage(v, "mixed")
            vecs[1:] = [v.astype(np.float32).astype(np.float64) for v in vecs[1:]]
        for i, v in enumerate(vecs):
            dev.setTimeIntegrationVector(i, v)
        co = [1.0, -0.3, 0.25, 1.5, -0.125, 0.2, 0.7, -1.1]
        for tiles in (1, 2, 4, 8):
            dev.setAdvectionTiles(tiles)
            for m in (1, 2, 3, 4, 7, 8) if tiles < 4 else (1, 2, 5):
                dev.computeTimeDerivative(list(range(m)), co[:m], 8)
                got = dev.getTimeIntegrationVector(8)
                ld = refs[1].time_derivative(vecs[:m], co[:m])
                if precision == "fp64":
                    assert_parity(got, refs[0].time_derivative(vecs[:m], co[:m]), ld, p, refs[0],
                                  f"advection pencils {n} p={p} m={m}")
                else:
                    assert rel(got, ld) <= 2.0 ** -24 + 1e-12
        dev.close()


@pytest.mark.parametrize("n,p,tab,precision", [
    ([32, 16], 1, "RK4", "fp64"), ([31, 17], 1, "RK4", "mixed"), ([19, 17], 2, "RK3_TVD", "fp64"),
    ([12, 10], 3, "DORMAND_PRINCE", "mixed"), ([12, 11], 3, "RK4", "fp64"), ([10, 10], 4, "RK4", "fp64"),
    ([8, 8, 4], 1, "RK2_TVD", "fp64"), ([4, 4, 3], 2, "RK4", "mixed"), ([4, 4, 4], 2, "RK4", "fp64"),
    ([3, 3, 3], 3, "RK3_TVD", "fp64"), ([3, 3, 3], 1, "RK4", "fp64")])
def test_one_workgroup_steps_bitwise_equal_graph_replay(n, p, tab, precision):
    """Steps in one workgroup with one x-pencil a thread, up to its largest
    number of threads and beyond (the kernel that loops over pencils), against
    the replayed step graph: the same operations, so the same bits."""
    print(f"[case] one workgroup n={n} p={p} {tab} {precision}", flush=True)
    tableau = getattr(hpgem_amd.tableaux, tab)
    mesh = Mesh.structured(n)
    a = [1.0, -0.7, 0.3][:len(n)]
    out = {}
    for fused in (False, True):
        dev = HpgemAPIDevice(mesh, p, velocity=a, precision=precision, tableau=tableau, n_extra_vectors=2)
        dev.setFusedTimeStepping(fused)
        dev.setTimeIntegrationVector(0, np.random.default_rng(p).standard_normal(dev.n_dof))
        dev.computeOneTimeStep(0.0, 0.02 / max(n), 5)
        assert (dev.getFusedTimeStepping()[1] > 0) == fused
        out[fused] = [dev.getTimeIntegrationVector(v) for v in range(tableau.stages + 1)]
        dev.close()
    assert np.all(np.isfinite(out[True][0]))
    for g, f in zip(out[False], out[True]):
        np.testing.assert_array_equal(f, g)
