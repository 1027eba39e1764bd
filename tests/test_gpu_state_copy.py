"""hd_copy_state and hd_clone carry every byte of a context's state: grids
whose arrays end off a 16-byte and a 32 KB boundary, below and above one 32 KB
piece; the copies then step as the source does, bit for bit."""
import numpy as np
import pytest

from hydist_amd import synth
from hydist_amd._lib import HydistError, Solver

from _parity import assert_same_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,M", [(40, 12), (41, 13), (64, 61), (83, 74), (300, 60)])
def test_copied_state_is_the_source(N, M):
    case = synth.channel_case(N=N, M=M, nsteps=60)
    op = case.opts()
    src, dst = Solver(case), Solver(case)
    src.init()
    dst.init()
    t = src.run(0.0, 9, op)
    dst.run(0.0, 4, op)
    dst.copy_state_from(src)
    other = src.clone()
    for c, what in ((dst, "copy"), (other, "clone")):
        assert_same_state(src, c, what)
    src.copy_state_from(src)
    assert_same_state(src, dst, "a context copied from itself")
    for g in (src, dst, other):
        g.run(t, 11, op)
    for c, what in ((dst, "copy, 11 steps later"), (other, "clone, 11 steps later")):
        assert_same_state(src, c, what)
    assert np.isfinite(src.get("z")).all()


def test_contexts_of_other_sizes_are_refused():
    a, b = Solver(synth.channel_case(N=40, M=12, nsteps=60)), Solver(synth.channel_case(N=41, M=12, nsteps=60))
    a.init()
    b.init()
    with pytest.raises(HydistError):
        a.copy_state_from(b)
