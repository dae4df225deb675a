"""hgdg_right_hand_side on cubes of order 5, on both sides of the number of
elements from which the mass is applied in the kernel itself: a periodic box
against a part of it with the same elements and the same values. The result does
not depend on which of them computes it but for rounding (geometry and sums:
1e-12 of the largest value)."""
import numpy as np
import pytest

from _parity import rel
from hpgem_amd import OP_ACOUSTIC_CENTRAL, RK4, HpgemAPIDevice, Mesh

pytestmark = pytest.mark.gpu


def test_right_hand_side_of_a_box_and_of_a_part():
    print("[case] right-hand side, order 5, 4x5x5 and 12x10x10", flush=True)
    small, large, p = [4, 5, 5], [12, 10, 10], 5  # 100 and 1200 elements
    rng = np.random.default_rng(5)
    c = rng.uniform(0.5, 2.0, small[::-1])  # z, y, x: x fastest
    u = rng.standard_normal((*small[::-1], 4 * (p + 1) ** 3))
    times = [b // a for a, b in zip(small, large)][::-1]
    out = []
    for n, cn, un in ((small, c, u), (large, np.tile(c, times), np.tile(u, [*times, 1]))):
        mesh = Mesh.structured(n, upper=[k / m for k, m in zip(n, large)])
        dev = HpgemAPIDevice(mesh, p, kind=OP_ACOUSTIC_CENTRAL, c_inv=cn.ravel(), tableau=RK4)
        dev.setTimeIntegrationVector(0, un.ravel())
        dev.computeRightHandSide([0], [1.0], 1)
        out.append(dev.getTimeIntegrationVector(1).reshape(un.shape))
        dev.close()
    assert rel(out[1], np.tile(out[0], [*times, 1])) <= 1e-12
