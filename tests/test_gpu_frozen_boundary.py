"""hd_sediment_run's boundary values: from its second step on a workgroup of
the VTH launch writes them; one step at a time over the whole grid (an upload
of the same mask starts over) runs the boundary kernel.  Level and discharge
edges meet at the corners; edges shorter and longer than a wave's 64 cells and
its 256 of a round."""
import pytest

from hydist_amd.case import BED_EVERY_STEP
from hydist_amd._lib import Solver

from _parity import assert_same_state
from test_gpu_parity import open_basin

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,M", [(30, 26), (64, 67), (20, 261), (330, 18)])
@pytest.mark.parametrize("types", [(0, 2, 2, 1), (1, 1, 1, 1), (2, 2, 2, 2)])
def test_boundary_beside_vth(types, N, M):
    c = open_basin(types, N=N, M=M)
    c.bed_change_start, c.bed_mode = 0.0, BED_EVERY_STEP
    op = c.opts()
    a = Solver(c)
    a.init()
    t = a.run(0.0, 6, op)
    b = a.clone()
    a.sediment_run(t, 5, op)
    for k in range(5):
        b.set("khouot", b.get("khouot"))
        b.sediment_run(t + k * c.dT, 1, op)
    assert_same_state(a, b, f"{types}, 5 steps on a frozen flow")
    a.run(t, 4, op)
    b.run(t, 4, op)
    assert_same_state(a, b, f"{types}, 4 whole steps later")
