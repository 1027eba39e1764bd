"""GPU: the flow sweeps' rows against the CPU checker bit for bit with grid
spacings and time steps far outside any real case's, where the rows' shared
reciprocals of the case constants do not apply."""
import numpy as np
import pytest

import oracle
from hydist_amd import synth
from hydist_amd._lib import Solver
from hydist_amd.case import make_case_header

from _parity import diff_fields

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dX,dY,dT", [(10.0, 10.0, 2.0), (1e18, 10.0, 2.0), (10.0, 1e18, 2.0), (1e-18, 1e-18, 2.0),
                                      (1e150, 1e150, 1e10), (10.0, 1e153, 2.0), (1e-160, 10.0, 2.0),
                                      (10.0, 10.0, 1e-30), (2.0**-26, 2.0**24, 1.0)])
def test_rows_of_extreme_constants(dX, dY, dT):
    c = synth.channel_case(N=90, M=80)
    c.header = make_case_header(dX, dY, dT, c.segment_limit, H_TINH=0.02, heso=0.94, CORIOLIS_FORCE=1e-4)
    o, g = oracle.Oracle(c), Solver(c)
    o.init()
    g.init()
    rng = np.random.default_rng(1)
    shape = o.get("u").shape
    for n, size in (("u", 0.5), ("v", 0.5), ("z", 0.2), ("VISCOIDX", 1e-3)):
        f = size * rng.standard_normal(shape) * 10.0 ** rng.integers(-40, 1, shape)
        for x in (o, g):
            x.set(n, f)
    for name, entry, hi in (("uz_solve", "UZSolver", c.M), ("vz_solve", "VZSolver", c.N)):
        o.kernel(name, 2, hi)
        g.kernel(entry, 0)
        assert diff_fields(o.get, g.get, ("t_z", "t_u", "t_v")) == [], entry
