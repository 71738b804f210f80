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
// keys that the causal unit in place i reads, or -1 if another place names it too
extern "C" int fa_order(int batch, int kv, int group, int rows, int *keys) {
    const FaRows r = fa_rows_of(0, rows, group, false);
    const int n = fa_rows_units(r, batch, kv, group);
    for (int i = 0; i < n; i++) {
        const int lin = fa_longest_first(r, batch, kv, group, i);
        const FaUnit u = fa_unit(r, batch, kv, group, lin);
        keys[i] = lin < 0 || lin >= n ? -1 : u.qbase + (u.left ? u.left : FA_ROWS);
        for (int j = 0; j < i; j++) if (fa_longest_first(r, batch, kv, group, j) == lin) keys[i] = -1;
    }
    return n;
}
"""


@pytest.fixture(scope="module")
def owners(tmp_path_factory):
    d = tmp_path_factory.mktemp("flash_rows")
    src, so = d / "shim.cpp", d / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(ROOT, "o1.c_amd", "csrc"),
                    "-o", str(so), str(src)], check=True)
    shim = ctypes.CDLL(str(so))
    fn = shim.fa_owners

    def run(batch, kv, group, row0, rows, share, S):
        n = np.zeros((batch, kv * group, S), np.int32)
        return n, fn(batch, kv, group, row0, rows, int(share), S, n.ctypes.data_as(ctypes.c_void_p))
    run.order = shim.fa_order
    return run


@pytest.mark.parametrize("batch,kv,group", [(1, 1, 1), (2, 2, 4), (1, 8, 3)])
def test_causal_units_start_longest_first(owners, batch, kv, group):
    """Every causal unit has one place in the order, and none reads more keys than
    the one before it."""
    for rows in (1, 114, 255, 256, 257, 512, 700, 1185):
        keys = np.zeros(batch * kv * group * (rows // 256 + 1), np.int32)
        n = owners.order(batch, kv, group, rows, keys.ctypes.data_as(ctypes.c_void_p))
        assert n == batch * kv * group * -(-rows // 256)
        assert (keys[:n] > 0).all() and (np.diff(keys[:n]) <= 0).all() and keys[0] == rows


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
