"""Row ownership of the 8-wave attention units (csrc/flash_rows.hpp), on the CPU."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SHIM = """
#include "flash_rows.hpp"
// writers[b][head][row] counts the units that store it; bad counts rows whose
// 32-row strip (the mask bits of the wave that stores them) is not their own
extern "C" int fa_owners(int batch, int kv, int group, int row0, int rows, int share, int S, int *writers) {
    const FaRows r = fa_rows_of(row0, rows, group, share != 0);
    int bad = 0;
    for (int lin = 0; lin < fa_rows_units(r, batch, kv, group); lin++) {
        const FaUnit u = fa_unit(r, batch, kv, group, lin);
        for (int i = 0; i < FA_ROWS; i++) {
            const FaRowHead w = fa_unit_row(u, group, i);
            if (w.row == FA_NO_ROW || w.row >= row0 + rows) continue;
            writers[((long)u.b * kv * group + w.head) * S + w.row]++;
            bad += w.row / 32 != u.qbase / 32 + i / 32;
        }
    }
    return bad;
}
"""


@pytest.fixture(scope="module")
def owners(tmp_path_factory):
    d = tmp_path_factory.mktemp("flash_rows")
    src, so = d / "shim.cpp", d / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(ROOT, "o1.c_amd", "csrc"),
                    "-o", str(so), str(src)], check=True)
    fn = ctypes.CDLL(str(so)).fa_owners

    def run(batch, kv, group, row0, rows, share, S):
        n = np.zeros((batch, kv * group, S), np.int32)
        return n, fn(batch, kv, group, row0, rows, int(share), S, n.ctypes.data_as(ctypes.c_void_p))
    return run


# every remainder of 256 rows, below and past whole tiles, with and without rows in front
@pytest.mark.parametrize("group", [1, 2, 3, 4, 8])
def test_every_row_has_one_writer(owners, group):
    """A (batch, head, row) is stored by exactly one unit, whether left-over rows
    share units (full rows) or not (causal and dense-mask rows); where they do
    not, a wave's rows are the 32 of its own mask strip."""
    for rows in list(range(1, 258)) + [300, 364, 511, 512, 513, 1209, 2371]:
        for row0 in (0, 76) if rows % 64 in (0, 1, 9, 44) else (0,):
            for share in (False, True):
                S = row0 + rows + 3
                n, bad = owners(2, 2, group, row0, rows, share, S)
                assert (n[:, :, row0:row0 + rows] == 1).all(), (group, row0, rows, share)
                assert n.sum() == 2 * 2 * group * rows
                assert share or row0 or bad == 0, (group, rows, bad)
