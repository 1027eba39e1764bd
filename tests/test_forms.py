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


def test_wetting_forms(tmp_path):
    """HYDIST_WETTING=window replays every line that the candidate list holds
    and =scan scans every line; by default the lanes visit their candidates at
    once unless one depends on another."""
    L = compiled(tmp_path, "wet", """
int form(int mode, int n, int dependent) { return hd_wet_form(mode, n, 64, dependent); }
int at_once() { return HD_WET_AT_ONCE; }
int replay() { return HD_WET_REPLAY; }
int scan() { return HD_WET_SCAN; }""")
    at_once, replay, scan = L.at_once(), L.replay(), L.scan()
    for n in (1, 8, 9, 64):
        for dependent in (0, 1):
            assert L.form(0, n, dependent) == (replay if dependent else at_once)
            assert L.form(1, n, dependent) == replay
            assert L.form(2, n, dependent) == scan
    assert {L.form(m, 65, 0) for m in (0, 1, 2)} == {scan}


def test_batched_thomas_form(tmp_path):
    """Short systems of a large batch go by lanes whatever the arrays' length
    is: the device takes the longest of 64 systems."""
    L = compiled(tmp_path, "thomas", "int lanes(int nsys, int some, long long rows) "
                                     "{ return hd_thomas_lanes(nsys, some, rows); }")
    lanes = lambda nsys, some, rows: L.lanes(nsys, some, ctypes.c_longlong(rows))
    for nsys, rows, want in ((64, 4, 1), (64, 8, 0), (2000, 8, 1), (2000, 12, 0), (20000, 24, 1), (20000, 64, 0),
                             (1, 2, 1), (1, 503, 0), (2000, 503, 0), (2**31 - 1, 2**20, 1), (5, 2**31, 0), (9, 0, 1)):
        assert lanes(nsys, 1, rows) == want
        assert lanes(nsys, nsys, rows * nsys) == want
