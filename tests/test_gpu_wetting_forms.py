"""GPU: the wetting pass against the CPU checker bit for bit where its forms
change: candidates apart and near each other, cascades that stay within a
candidate's window and that leave it, few and many candidates per line."""
import numpy as np
import pytest

import oracle
from hydist_amd import synth
from hydist_amd._lib import Solver

from _parity import diff_fields

pytestmark = pytest.mark.gpu


def patches(rng, shape, density, longest):
    """dry patches of 1 .. longest cells along both axes"""
    dry = np.zeros(shape, bool)
    for axis in (0, 1):
        for i, j in np.argwhere(rng.random(shape) < density):
            k = rng.integers(1, longest + 1)
            if axis:
                dry[i, j:j + k] = True
            else:
                dry[i:i + k, j] = True
    return dry


@pytest.mark.parametrize("horizontal", [1, 0])
@pytest.mark.parametrize("density,longest", [(0.002, 3), (0.006, 6), (0.02, 4), (0.05, 9), (0.15, 2)])
def test_candidates_and_cascades(density, longest, horizontal):
    c = synth.channel_case(N=150, M=140, nsteps=100, Q=1000.0)
    o, g = oracle.Oracle(c), Solver(c)
    o.init()
    g.init()
    o.run(0.0, 2, c.opts())
    g.run(0.0, 2, c.opts())
    rng = np.random.default_rng(int(density * 1000) + horizontal)
    kh, z = o.get("khouot"), o.get("z")
    wet = kh == 0
    kh[wet & patches(rng, kh.shape, density, longest)] = 1
    # levels above the bed level of the scan (the old z) in most cells, so
    # that cascades run on and stop at different lengths
    tz = np.where(wet, z + 0.02 * (rng.random(z.shape) - 0.25), z)
    for x in (o, g):
        x.set("khouot", kh)
        x.set("t_z", tz)
    o.kernel("update_h_moi")
    o.kernel("reset_states_h" if horizontal else "reset_states_v")
    o.kernel("update_uvz", 0, 0)
    o.kernel("htuongdoi")
    g.kernel("Reset_states", horizontal, 0, 0)
    assert diff_fields(o.get, g.get, ("khouot", "t_z", "H_moi", "FS", "t_u", "t_v", "z", "u", "v", "Htdu",
                                      "Htdv")) == []
    opened = (kh == 1) & (o.get("khouot") == 0)
    assert opened.sum() > 20
