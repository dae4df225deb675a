"""A non-finite coefficient stays where the operator takes it. Tables padded
with zeros, values loaded for lanes that have none and coefficients of zero are
harmless only while what they multiply is finite, so each kernel is run with
NaN and infinity in one element and the values that came out non-finite are
compared with those that the operator lets the element reach."""
import numpy as np
import pytest

from _meshes import perturb, rotate_elements
from hpgem_amd import OP_ACOUSTIC_CENTRAL, RK4, HpgemAPIDevice, Mesh

pytestmark = pytest.mark.gpu


def neighbours(mesh, corners):
    """Per element the elements that share a face (`corners` node ids) with it."""
    owner = {}
    for e, ids in enumerate(mesh.node_ids):
        for i in ids:
            owner.setdefault(int(i), []).append(e)
    out = []
    for e, ids in enumerate(mesh.node_ids):
        count = np.bincount(np.concatenate([owner[int(i)] for i in ids]), minlength=mesh.n_elements)
        count[e] = 0
        out.append(np.nonzero(count >= corners)[0])
    return out


@pytest.mark.parametrize("orders", [(1,), (2,), (3,), (4,), (1, 2, 3, 4)])
@pytest.mark.parametrize("threads", [[8, 12, 32, 35], [16, 32, 64, 64]])
def test_tetrahedra(orders, threads):
    """v of an element enters k_s of the element and of its neighbours, s enters
    k_v; k_v does not depend on v, nor k_s on s."""
    print(f"[case] non-finite tets p={orders} threads={threads}", flush=True)
    mesh = Mesh.structured([3, 3, 3], simplices=True)
    E = mesh.n_elements
    rng = np.random.default_rng(len(orders))
    p = rng.choice(np.array(orders, dtype=np.int32), E).astype(np.int32)
    nb = (p + 1) * (p + 2) * (p + 3) // 6
    off = np.concatenate([[0], np.cumsum(4 * nb)])
    dev = HpgemAPIDevice(mesh, p, kind=OP_ACOUSTIC_CENTRAL, c_inv=np.ones(E), tableau=RK4)
    dev.setSimplexThreads(threads)
    near = neighbours(mesh, 3)
    u0 = rng.standard_normal(dev.n_dof)
    for e in range(E):
        for field in (0, 1 + e % 3):
            for bad in (np.nan, np.inf):
                u = u0.copy()
                u[off[e] + field * nb[e]:off[e] + (field + 1) * nb[e]] = bad
                dev.setTimeIntegrationVector(0, u)
                dev.computeTimeDerivative([0], [1.0], 1)
                finite = np.isfinite(dev.getTimeIntegrationVector(1))
                reached = np.zeros(dev.n_dof, dtype=bool)
                for a in [e, *near[e]]:
                    lo = off[a] + (nb[a] if field == 0 else 0)
                    reached[lo:off[a + 1] if field == 0 else off[a] + nb[a]] = True
                assert np.all(finite[~reached]), (e, field, bad)
                own = slice(off[e] + nb[e], off[e + 1]) if field == 0 else slice(off[e], off[e] + nb[e])
                assert not np.any(finite[own]), (e, field, bad)
    dev.close()


@pytest.mark.parametrize("n", [[5, 4], [4, 3, 3]])
@pytest.mark.parametrize("p", [1, 2, 4])
@pytest.mark.parametrize("general", [False, True])
@pytest.mark.parametrize("periodic", [False, True])
def test_advection_stays_downwind(n, p, general, periodic):
    """The upwind flux takes one trace: an element reaches itself and the
    neighbours across its outflow faces, no others (the general elements'
    Gauss-point kernel and the tensor kernel; displaced vertices, elements
    turned, and boxes with boundaries and without)."""
    print(f"[case] non-finite advection n={n} p={p} general={general} periodic={periodic}", flush=True)
    dim = len(n)
    a = np.array([1.0, 0.6, 0.4][:dim])  # no face of the meshes is parallel to it
    mesh = Mesh.structured(n, periodic=[int(periodic)] * dim)
    X, N = mesh.coords, mesh.node_ids
    if general:
        X, N, _ = rotate_elements(perturb(X, 0.02), N, 7)
    mesh = Mesh(mesh.shape, X, N)
    dev = HpgemAPIDevice(mesh, p, velocity=list(a), tableau=RK4, tensor_general=general)
    E, nb = mesh.n_elements, dev.n_dof // mesh.n_elements
    box = np.array(n)
    centre = X.mean(axis=1)

    def outflow(e, b):  # the step to a face neighbour, wrapped around the box, is a cell along an axis
        d = (centre[b] - centre[e]) * box
        if periodic:
            d = (d + box / 2) % box - box / 2
        return d[np.argmax(np.abs(d))] > 0

    near = neighbours(mesh, 1 << (dim - 1))
    u0 = np.random.default_rng(p).standard_normal((E, nb))
    for e in range(E):
        for bad in (np.nan, np.inf):
            u = u0.copy()
            u[e, :] = bad
            dev.setTimeIntegrationVector(0, u.ravel())
            dev.computeTimeDerivative([0], [1.0], 1)
            finite = np.isfinite(dev.getTimeIntegrationVector(1).reshape(E, nb))
            reached = np.zeros(E, dtype=bool)
            reached[e] = True
            reached[[b for b in near[e] if outflow(e, b)]] = True
            assert np.all(finite[~reached]), (e, bad)
            assert not np.any(finite[reached].all(axis=1)), (e, bad)
    dev.close()
