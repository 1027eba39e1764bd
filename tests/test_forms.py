"""The rules of csrc/hd_forms.h, compiled for the host: which form of a
computation a lane, a line or a batch takes."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gpu-hydist_amd", "csrc")


def compiled(tmp_path, name, code):
    src, out = tmp_path / f"{name}.cpp", tmp_path / f"{name}_test_lib"
    src.write_text('#include "hd_forms.h"\nextern "C" {\n' + code + "\n}\n")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-fPIC", "-shared", "-I", CSRC, "-o", str(out), str(src)],
                   check=True)
    return ctypes.CDLL(str(out))


@pytest.mark.parametrize("br1,br2", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_rows_of_a_round(tmp_path, br1, br2):
    """Every cell of a run but the last gets its momentum row from exactly one
    lane, and no lane without a lane after it needs one: else the round's fast
    rows would be thrown away for a row that nothing stores."""
    L = compiled(tmp_path, "rows", """
int use(int lane, int k, int first, int last, int br1, int br2)
{
    const HdCellUse u = hd_cell_use(lane, k, first, last, br1, br2);
    return u.row | u.behind << 1 | u.ahead << 2;
}""")
    for n in (1, 2, 3, 62, 63, 64, 65, 126, 127, 128, 190, 253, 300):
        first, last = 5, 4 + n
        rows = np.zeros(n, int)
        for k0 in range(first, last + 1, 63):
            for lane in range(64):
                k = k0 + lane
                u = L.use(lane, k, first, last, br1, br2)
                if not u & 1:
                    continue
                assert lane < 63, "a row with no lane after it"
                rows[k - first] += 1
                assert bool(u & 2) == (n > 2 and not (br1 and k == first))
                assert bool(u & 4) == (n > 2 and not (br2 and k == last - 1))
        assert (rows[:-1] == 1).all() and rows[-1] == 0
