"""Served acoustic boxes whose planes pass the L2 (their workgroups are taken in
columns of rows, by a table of their own) resident beside boxes of the same
family without a table, in front of them and behind: one launch serves all, each
workgroup finding its problem and its place in that problem's table. The same
solves run alone give the same bits."""
import numpy as np
import pytest

from hpgem_amd import HpgemAPIDevice, Mesh, OP_ACOUSTIC_CENTRAL
from hpgem_amd.serving import Server

pytestmark = pytest.mark.gpu

# (order, cells): 20 x 20 and 24 x 19 elements of order 4 and 32 x 30 of order 3 pass 4 MB a plane
FAMILIES = [(4, [[5, 4, 3], [20, 20, 3], [3, 3, 4], [24, 19, 4], [6, 5, 4]]), (3, [[32, 30, 3], [7, 5, 3], [30, 33, 4]])]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("order,boxes", FAMILIES)
def test_boxes_with_and_without_a_table(precision, order, boxes):
    print(f"[case] served order tables p={order} {precision}", flush=True)
    steps, dt, amp = 60, 1e-4, [0.7, -0.4]
    k = np.array([[1.0, 2.0, 1.0], [2.0, 1.0, 3.0]])
    srv = Server(precision=precision, hbm_budget_gb=8, max_active=8)
    tickets = [srv.submit(3, "acoustic", order, cells, amp, k, dt, steps, velocity=[0.0] * 3, wave_speed=1.0,
                          keep_state=True) for cells in boxes]
    assert srv.wait(-1, 120)
    served = [srv.result(t, with_state=True)["state"] for t in tickets]
    ticks = srv.stats()["ticks"]
    srv.close()
    assert ticks < len(boxes) * steps  # they were resident together
    for cells, state in zip(boxes, served):
        mesh = Mesh.structured(cells)
        dev = HpgemAPIDevice(mesh, order, precision=precision, kind=OP_ACOUSTIC_CENTRAL, c_inv=np.ones(mesh.n_elements))
        dev.setInitialSolutionModes(amp, k, field=0)
        dev.computeOneTimeStep(0.0, dt, steps)
        np.testing.assert_array_equal(state, dev.getTimeIntegrationVector(0))
        dev.close()
